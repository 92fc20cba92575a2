// Ragged ensembles of independent 2-D systems in one persistent launch.
//
// Each workgroup owns one system of a CSR (particles [offset, offset + n)) and
// runs the reference's minimisation loop for it,
//
//   for step:  nbrs = nbrs.update(R)            partition.py:1141-1164
//              state = fire_apply(state, nbrs)  minimize.py:170-226
//
// entirely inside the workgroup, separated by workgroup barriers: the skin
// test, the Dense list rebuild on the system's own cell grid (LDS counts, the
// reference's candidate order and both-direction test, partition.py:911-980),
// the velocity-Verlet sub-step with float64 positions (simulate.py:227-243),
// the soft-sphere forces (energy.py:125-173 through smap.py:856-979) with the
// lane grouping of the plain Dense kernel (two accumulators per row, summed in
// float64), and the FIRE reductions and float16 bookkeeping
// (minimize.py:185-221).  No host round trip and no grid-wide
// synchronisation: systems never interact.  Workgroups take systems in the
// order given (largest first balances the tail).
#include "jmd_pair_common.hpp"

namespace jmd {

// Threads per system, one workgroup each: 512 keeps two workgroups a CU and
// wins by 10-35% where every CU has several systems of one size to run (50
// steps of 512 systems of 512 / 1024 / 2048 particles: 2.4 / 3.4 / 5.3 ms
// against 3.3 / 3.9 / 5.8); 1024 shortens each system's own chain and wins
// where the largest one decides (64 systems of 1024 / 2048 / 4000: 1.6 / 2.5 /
// 4.4 ms against 1.9 / 3.4 / 6.4; 512 systems log-uniform in 64..2048 and
// 64..4096: 4.0 and 5.4 against 4.4 and 7.4).  So 1024 when the largest system
// has 768 particles or more (below, its rows leave the second 512 threads too
// little) and at least a CU's share of all of them; also for an average of
// 4096, beyond which 512 threads stage no system in LDS.
constexpr int kEnsThreads = 1024;  // the most a workgroup has
constexpr int kEnsWaves = 4;       // a SIMD (at 8, 64 VGPRs: the run spilled and took 1.5 times as long)
static int g_ens_threads = 0;      // jmd_fire_ensemble_set_threads (0: by size)
constexpr int kEnsCUs = 256;       // of an MI355X
inline int ens_threads(int n_systems, long long n_total, long long n_max) {
  if (n_systems > 0 && n_total / n_systems >= 4096) return 1024;
  return n_max >= 768 && n_max >= n_total / kEnsCUs ? 1024 : 512;
}
// A launch's threads: the override, the caller's (mode >> 8), or the rule for
// a largest system that is not known (taken as the average).
inline int ens_launch_threads(int asked, int n_systems, long long n_total) {
  if (g_ens_threads) return g_ens_threads;
  if (asked) return asked;
  return n_systems > 0 && n_total / n_systems >= 4096 ? 1024 : 512;
}
inline bool ens_threads_ok(int threads) {
  return threads == 0 || threads == 256 || threads == 512 || threads == 1024;
}
constexpr int kEnsMaxCells = 8192;
constexpr int kEnsBatch = 4;       // elements a streaming pass loads together
constexpr int kEnsRowChunk = 4;    // row entries gathered together (one 16-byte load)
constexpr int kEnsParMax = 64;  // species matrices staged in LDS (n_species^2 at most)
constexpr int kEnsPerThread = 8;  // particles per thread of a system staged in LDS
static_assert(kEnsThreads * kEnsPerThread <= (1 << 16), "staged ids are 16-bit");

struct EnsSys {
  int offset, n;
  int cps[2];
  float cell_size[2];
  int fill_cps[2];
  float fill_cell_size[2];
  float side[2];
  int cap, max_occ;
  float cutoff_sq, threshold_sq;  // list cutoff^2, (skin / 2)^2
  int param_offset;               // this system's block of species parameters
  int reserved;
};

// Per-step record of a forward segment for the adjoint (all system-major by
// particle, node k = state after k steps of the segment, k = 0..K):
//   x[k], F[k]: float32 positions and forces at node k ([K+1][ntot][2])
//   q[k]: momentum of step k after the second half kick, before the FIRE
//         mixing ([K][ntot][2])
//   idx[k]: a Dense list slot ([K+1][ntot][width]); slot 0 holds node 0's
//         list, slot k + 1 the list a system rebuilt at step k (a system's
//         other slots are not written)
//   sc[k][s]: step k's scalars of system s: dt, alpha, keep, sqrt(pp),
//         sqrt(ff + 1e-6), and the slot of the list the force at node k + 1
//         was computed with  ([K][nsys][kTapeScalars])
struct EnsTape {
  float* x;
  float* F;
  float* q;
  int* idx;
  float* sc;
  int K;
};
constexpr int kTapeScalars = 6;

struct FireP {
  float dt_start, dt_max;
  int n_min;
  float f_inc, f_dec, alpha_start, f_alpha;
};

enum { ENS_FILL = 0, ENS_OCCUPANCY = 1, ENS_INIT = 2, ENS_RUN = 3 };

__device__ __forceinline__ float f16r(float x) { return (float)(_Float16)x; }

// Workgroup-wide sum of three doubles (all threads call; result in all).
__device__ __forceinline__ void wg_sum3(double& a, double& b, double& c, double* s) {
  a = wave_reduce_sum(a);
  b = wave_reduce_sum(b);
  c = wave_reduce_sum(c);
  const int w = threadIdx.x / kWave, nw = blockDim.x / kWave;
  __syncthreads();
  if (lane_id() == 0) {
    s[3 * w] = a;
    s[3 * w + 1] = b;
    s[3 * w + 2] = c;
  }
  __syncthreads();
  a = b = c = 0.0;
  for (int k = 0; k < nw; ++k) {  // fixed order
    a += s[3 * k];
    b += s[3 * k + 1];
    c += s[3 * k + 2];
  }
  __syncthreads();
}

__device__ __forceinline__ int wg_max(int v, int* s) {
  v = wave_reduce_max(v);
  const int w = threadIdx.x / kWave, nw = blockDim.x / kWave;
  __syncthreads();
  if (lane_id() == 0) s[w] = v;
  __syncthreads();
  int r = 0;
  for (int k = 0; k < nw; ++k) r = max(r, s[k]);
  __syncthreads();
  return r;
}

// ref_mod64 with the library's fmod out of line: within one period past the
// box the remainder is the exact difference (L <= x < 2 L), and -L < x < 0 is
// its own remainder.
__device__ __noinline__ double ens_mod64_far(double x, double L) { return ref_mod64(x, L); }
__device__ __forceinline__ double ens_mod64(double x, double L) {
#pragma clang fp contract(off)
  if (!(x > -L && x < 2.0 * L)) return ens_mod64_far(x, L);
  if (x >= L) return x - L;
  return x < 0.0 ? x + L : x;
}

// Ascending order of 8 values: Batcher's odd-even merge sort network
// (19 compare-exchanges, all indices static so the values stay in registers).
__device__ __forceinline__ void cmp_swap(int& a, int& b) {
  const int lo = min(a, b), hi = max(a, b);
  a = lo;
  b = hi;
}
__device__ __forceinline__ void sort8(int* v) {
  cmp_swap(v[0], v[1]); cmp_swap(v[2], v[3]); cmp_swap(v[4], v[5]); cmp_swap(v[6], v[7]);
  cmp_swap(v[0], v[2]); cmp_swap(v[1], v[3]); cmp_swap(v[4], v[6]); cmp_swap(v[5], v[7]);
  cmp_swap(v[1], v[2]); cmp_swap(v[5], v[6]);
  cmp_swap(v[0], v[4]); cmp_swap(v[1], v[5]); cmp_swap(v[2], v[6]); cmp_swap(v[3], v[7]);
  cmp_swap(v[2], v[4]); cmp_swap(v[3], v[5]);
  cmp_swap(v[1], v[2]); cmp_swap(v[3], v[4]); cmp_swap(v[5], v[6]);
}

// Ascending order of one cell's ids m[0..cnt): up to 8 through the sorting
// network in registers, more by insertion sort in place.
template <typename T>
__device__ __forceinline__ void ens_sort_cell(T* m, int cnt) {
  if (cnt <= 8) {
    int v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = u < cnt ? (int)m[u] : 0x7fffffff;
    sort8(v);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (u < cnt) m[u] = (T)v[u];
    return;
  }
  for (int u = 1; u < cnt; ++u) {
    const T v = m[u];
    int w = u - 1;
    while (w >= 0 && m[w] > v) {
      m[w + 1] = m[w];
      --w;
    }
    m[w + 1] = v;
  }
}

// A system's float32 positions (and species ids) as the pair and list loops
// read them: from LDS when the workgroup staged the system there (l, ls), else
// from global memory.  base is the system's first global id.
template <bool STAGED>
struct EnsView {
  const float* __restrict__ g;
  const float* l;
  const int* __restrict__ gs;
  const uint8_t* ls;  // staged species ids (nullptr: gs)
  int base;
  __device__ __forceinline__ void pos(int i, float* xi) const {
    if constexpr (STAGED) {
      xi[0] = l[2 * (i - base)];
      xi[1] = l[2 * (i - base) + 1];
    } else {
      load_pos<2>(g, i, xi);
    }
  }
  __device__ __forceinline__ int species(int i) const {
    if constexpr (STAGED) {
      if (ls) return (int)ls[i - base];
    }
    return gs ? gs[i] : 0;
  }
};

// Bins the system on grid g: LDS counts, exclusive starts, arrival ranks,
// scatter into sorted[] (system-local), then each cell's ids in ascending
// order (the stable argsort of partition.py:432).  s_cs holds the counts,
// then, scanned in place, the starts (cell c spans s_cs[c] .. s_cs[c + 1]).
// Returns the max filling; all_in: every position lies in [0, L].
template <bool STAGED>
__device__ __forceinline__ int ens_bin(const EnsSys& S, const Grid& g, const Space& sp,
                                       const EnsView<STAGED>& V,
                                       int* __restrict__ cellp, int* __restrict__ rankp,
                                       int* __restrict__ sorted, int* s_cs, int* s_red,
                                       uint16_t* ls, bool* all_in) {
  const int nt = blockDim.x, t = threadIdx.x;
  bool in = true;  // this thread's positions inside [0, L]
  auto inside = [&](const float* x) {
    return x[0] >= 0.0f && x[0] <= sp.L[0] && x[1] >= 0.0f && x[1] <= sp.L[1];
  };
  for (int c = t; c < g.ncell; c += nt) s_cs[c] = 0;
  __syncthreads();
  // staged system (ls: its cell-sorted ids in LDS): counts here, then after
  // the scan a second pass of LDS atomics on the starts places each id (the
  // cells are sorted by id afterwards, so arrival order does not matter);
  // cells are recomputed from the LDS positions, nothing goes to memory
  if constexpr (STAGED) {
    for (int a = t; a < S.n; a += nt) {
      float xi[2];
      V.pos(S.offset + a, xi);
      in = in && inside(xi);
      int ci[2];
      atomicAdd(&s_cs[cell_of<2>(xi, g, ci)], 1);
    }
  } else {
    for (int a = t; a < S.n; a += nt) {
      float xi[2];
      V.pos(S.offset + a, xi);
      in = in && inside(xi);
      int ci[2];
      const int h = cell_of<2>(xi, g, ci);
      cellp[a] = h;
      rankp[a] = atomicAdd(&s_cs[h], 1);
    }
  }
  __syncthreads();
  // exclusive scan of the counts: per-thread chunks, a wavefront scan of the
  // chunk totals, then the wave totals in order
  const int per = (g.ncell + nt - 1) / nt;
  const int beg = min(t * per, g.ncell), end = min(beg + per, g.ncell);
  int local = 0, fill = 0;
  for (int c = beg; c < end; ++c) {
    local += s_cs[c];
    fill = max(fill, s_cs[c]);
  }
  const int lane = lane_id(), wv = t / kWave, nw = nt / kWave;
  int incl = local;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int y = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += y;
  }
  __shared__ int s_wave[kEnsThreads / kWave + 1];
  if (lane == kWave - 1) s_wave[wv] = incl;
  __syncthreads();
  if (t == 0) {
    int acc = 0;
    for (int k = 0; k < nw; ++k) {
      const int v = s_wave[k];
      s_wave[k] = acc;
      acc += v;
    }
    s_wave[nw] = acc;
  }
  __syncthreads();
  int run = s_wave[wv] + incl - local;
  for (int c = beg; c < end; ++c) {
    const int cnt = s_cs[c];  // this thread's own chunk: read, then overwrite
    s_cs[c] = run;
    run += cnt;
  }
  if (t == 0) s_cs[g.ncell] = s_wave[nw];
  __syncthreads();
  if constexpr (STAGED) {
    for (int a = t; a < S.n; a += nt) {
      float xi[2];
      V.pos(S.offset + a, xi);
      int ci[2];
      ls[atomicAdd(&s_cs[cell_of<2>(xi, g, ci)], 1)] = (uint16_t)a;
    }
    __syncthreads();
    // s_cs[c] now holds the end of cell c, the start of cell c + 1: shift
    // back by one, chunks from the top (a chunk reads its own and the next
    // lower chunk's values before any of them is written)
    for (int c0 = ((g.ncell - 1) / nt) * nt; c0 >= 0; c0 -= nt) {
      const int c = c0 + t;
      const int v = c < g.ncell && c > 0 ? s_cs[c - 1] : 0;
      __syncthreads();
      if (c < g.ncell) s_cs[c] = v;
      __syncthreads();
    }
  } else {
    for (int a = t; a < S.n; a += nt) sorted[s_cs[cellp[a]] + rankp[a]] = a;
  }
  __syncthreads();
  // order each cell by id (thread per cell): up to 8 ids through a sorting
  // network in registers, more by insertion sort in place
  if constexpr (STAGED) {
    for (int c = t; c < g.ncell; c += nt) ens_sort_cell(ls + s_cs[c], s_cs[c + 1] - s_cs[c]);
  } else {
    for (int c = t; c < g.ncell; c += nt) ens_sort_cell(sorted + s_cs[c], s_cs[c + 1] - s_cs[c]);
  }
  *all_in = !__syncthreads_or(!in);
  return wg_max(fill, s_red);
}

// First slot's rank in a cell's list: slot order is rank (start + k) mod cap,
// so the first slots hold the members past the next multiple of cap.
template <bool STAGED>
__device__ __forceinline__ int ens_first_rank(int start, int m, int cap, float inv_cap) {
  int over;
  if constexpr (STAGED) {  // start % cap by the reciprocal, corrected
    over = start - (int)((float)start * inv_cap) * cap;
    over = over < 0 ? over + cap : (over >= cap ? over - cap : over);
  } else {
    over = start % cap;
  }
  const int w = cap - over;
  return m > w ? w : 0;
}

// Dense with cells keeps a candidate when both wrap(Ri - Rj) and wrap(Rj - Ri)
// are inside (partition.py:951,971).
__device__ __forceinline__ bool ens_exact(const float* xi, const float* xj, const Space& sp,
                                          float cutoff_sq) {
  return ref_metric_sq<2>(xi, xj, sp) < cutoff_sq && ref_metric_sq<2>(xj, xi, sp) < cutoff_sq;
}

// One Dense row as its entries come: rows whose stride is a multiple of 4
// entries are written 16 bytes at a time (every lane of a store writes a line
// of its own, so a row costs as many line accesses as it has stores: with
// 4-byte ones a 4,096-particle build took 14 us longer), entries past the row are counted.
struct EnsRowOut {
  int* row;
  int width, pad, cnt;
  bool vec;
  int4 quad;
  __device__ __forceinline__ EnsRowOut(int* __restrict__ idx, int i, int w, int p)
      : row(idx + (long long)i * w), width(w), pad(p), cnt(0),
        vec((w & 3) == 0 && ((uintptr_t)idx & 15) == 0), quad(make_int4(p, p, p, p)) {}
  __device__ __forceinline__ void put(int j) {
    if (cnt < width) {
      if (vec) {
        const int slot = cnt & 3;
        quad.x = slot == 0 ? j : quad.x;
        quad.y = slot == 1 ? j : quad.y;
        quad.z = slot == 2 ? j : quad.z;
        quad.w = slot == 3 ? j : quad.w;
        if (slot == 3) {
          *reinterpret_cast<int4*>(row + (cnt & ~3)) = quad;
          quad = make_int4(pad, pad, pad, pad);
        }
      } else {
        row[cnt] = j;
      }
    }
    ++cnt;
  }
  __device__ __forceinline__ void close() {  // the open quad, then pads
    if (vec) {
      int k = cnt < width ? (cnt & ~3) : width;
      if (k < width && (cnt & 3) != 0) {
        *reinterpret_cast<int4*>(row + k) = quad;
        k += 4;
      }
      for (; k < width; k += 4)
        *reinterpret_cast<int4*>(row + k) = make_int4(pad, pad, pad, pad);
    } else {
      for (int k = cnt; k < width; ++k) row[k] = pad;
    }
  }
};

constexpr int kEnsRunMax = 32;  // candidates of three cells in one mask

// Dense rows of a system whose positions all lie in [0, L] and whose cells
// fit their capacity, three of them a 32-bit mask.  The stencil's cells of one
// y are consecutive in the sorted ids (two pieces at the box's edge), so a row
// tests three runs of candidates, four at a time, into three masks, and then
// emits the kept ones cell by cell in the candidate order (x offset slowest,
// slots rotated).  Cell by cell, nine short loops took their fullest lane's
// chunks each and inlined the exact test sixteen times: a 4,096-particle
// build (1024 threads) took 92 us, this one 59.
template <bool STAGED>
__device__ __forceinline__ int ens_rows_runs(const EnsSys& S, const Grid& g, const Space& sp,
                                             float cutoff_sq, float lo_thr, float hi_thr,
                                             const EnsView<STAGED>& V,
                                             const int* __restrict__ sorted, const int* s_cs,
                                             int* __restrict__ idx, int width, int pad,
                                             const uint16_t* ls) {
  const int nt = blockDim.x;
  const float inv_cap = 1.0f / (float)g.cap;
  int occ = 0;
  // rows in cell order: neighbouring lanes read the same candidates
  for (int s = threadIdx.x; s < S.n; s += nt) {
    const int a = STAGED ? (int)ls[s] : sorted[s];
    const int i = S.offset + a;
    float xi[2];
    V.pos(i, xi);
    int ci[2];
    cell_of<2>(xi, g, ci);  // the binning's cell
    const int hx = ci[0], hy = ci[1], lx = g.cps[0] - 1, ly = g.cps[1] - 1;
    const int cx[3] = {hx == 0 ? lx : hx - 1, hx, hx == lx ? 0 : hx + 1};
    const int cy[3] = {g.cps[0] * (hy == 0 ? ly : hy - 1), g.cps[0] * hy,
                       g.cps[0] * (hy == ly ? 0 : hy + 1)};
    unsigned kept[3];
#pragma unroll
    for (int y = 0; y < 3; ++y) {
      const int c0 = cx[0] + cy[y], c1 = cx[1] + cy[y], c2 = cx[2] + cy[y];
      const int b0 = s_cs[c0], b1 = s_cs[c1], b2 = s_cs[c2];
      const int m0 = s_cs[c0 + 1] - b0, m01 = m0 + s_cs[c1 + 1] - b1;
      const int total = m01 + s_cs[c2 + 1] - b2;
      const int split = hx == 0 ? m0 : m01;
      const int second = hx == 0 ? b1 - m0 : b2 - m01;
      unsigned keep = 0, near = 0;
      for (int f0 = 0; f0 < total; f0 += kEnsRowChunk) {
        int jl[kEnsRowChunk];
        float xj[kEnsRowChunk][2];
#pragma unroll
        for (int c = 0; c < kEnsRowChunk; ++c) {
          const int f = min(f0 + c, total - 1);
          const int at = f + (f < split ? b0 : second);
          jl[c] = STAGED ? (int)ls[at] : sorted[at];
        }
#pragma unroll
        for (int c = 0; c < kEnsRowChunk; ++c) V.pos(S.offset + jl[c], xj[c]);
#pragma unroll
        for (int c = 0; c < kEnsRowChunk; ++c) {
          // |x_j - x_i| folded: min(|raw|, L - |raw|), positions in the box
          const float r0 = fabsf(xj[c][0] - xi[0]), r1 = fabsf(xj[c][1] - xi[1]);
          const float e0 = fminf(r0, sp.L[0] - r0), e1 = fminf(r1, sp.L[1] - r1);
          const float d2 = fmaf(e1, e1, e0 * e0);
          const unsigned bit = f0 + c < total && jl[c] != a ? 1u << (f0 + c) : 0u;
          keep |= d2 < lo_thr ? bit : 0u;
          near |= d2 <= hi_thr ? bit : 0u;
        }
      }
      near &= ~keep;
      while (near) {  // within the rounding margin of the cutoff
        const int f = __ffs((int)near) - 1;
        near &= near - 1;
        const int at = f + (f < split ? b0 : second);
        float xj[2];
        V.pos(S.offset + (STAGED ? (int)ls[at] : sorted[at]), xj);
        if (ens_exact(xi, xj, sp, cutoff_sq)) keep |= 1u << f;
      }
      kept[y] = keep;
    }
    const int cnt = __popc(kept[0]) + __popc(kept[1]) + __popc(kept[2]);
    occ = max(occ, cnt);
    if (width > 0) {
      EnsRowOut out(idx, i, width, pad);
#pragma unroll
      for (int x = 0; x < 3; ++x) {
        // the column's kept candidates in slot order, its three cells in turn
        int start[3], first[3], m[3];
        unsigned column = 0;
        int at = 0;
#pragma unroll
        for (int y = 0; y < 3; ++y) {
          const int c = cx[x] + cy[y];
          start[y] = s_cs[c];
          m[y] = s_cs[c + 1] - start[y];
          first[y] = ens_first_rank<STAGED>(start[y], m[y], g.cap, inv_cap);
          const unsigned bits = kept[y] & ((1u << m[y]) - 1u);
          kept[y] >>= m[y];  // the run's next cell
          column |= (bits >> first[y] | (bits & ((1u << first[y]) - 1u)) << (m[y] - first[y])) << at;
          at += m[y];
        }
        while (column) {
          const int f = __ffs((int)column) - 1;
          column &= column - 1;
          const int y1 = f >= m[0], y2 = f >= m[0] + m[1];
          const int my = y2 ? m[2] : (y1 ? m[1] : m[0]);
          int k = f - (y2 ? m[0] + m[1] - first[2] : (y1 ? m[0] - first[1] : -first[0]));
          k = (k >= my ? k - my : k) + (y2 ? start[2] : (y1 ? start[1] : start[0]));
          out.put(S.offset + (STAGED ? (int)ls[k] : sorted[k]));
        }
      }
      out.close();
    }
  }
  return occ;
}

// Dense rows of the system (global ids, padding pad) in the reference's
// candidate order; returns the largest row count.
template <bool STAGED>
__device__ __forceinline__ int ens_rows(const EnsSys& S, const Grid& g, const Space& sp,
                                        float cutoff_sq, const EnsView<STAGED>& V,
                        const int* __restrict__ sorted, const int* s_cs,
                        int* __restrict__ idx, int width, int pad, int* s_red,
                        const uint16_t* ls, bool all_in, int fill) {
  const int nt = blockDim.x, t = threadIdx.x;
  // The candidate test: the minimum-image |x_j - x_i|^2 of positions in the
  // box decides every candidate farther than `margin` from the cutoff; the
  // rest, and positions outside [0, L], take the reference-exact two-way test.
  // The few float32 roundings by which it can differ from the reference's
  // wrapped float32 d^2 are bounded where the cell build sets its margin;
  // this one is four times that bound.
  const float rc = sqrtf(cutoff_sq), Lmax = fmaxf(sp.L[0], sp.L[1]);
  const float margin =
      fmaxf(128.0f * (rc + 1.0f) * (Lmax + rc + 1.0f) * 1.1920929e-7f, 1e-4f * cutoff_sq);
  const float lo_thr = cutoff_sq - margin, hi_thr = cutoff_sq + margin;
  if (all_in && fill <= g.cap && 3 * fill < kEnsRunMax)
    return wg_max(ens_rows_runs(S, g, sp, cutoff_sq, lo_thr, hi_thr, V, sorted, s_cs, idx, width,
                                pad, ls),
                  s_red);
  const float inv_cap = 1.0f / (float)g.cap;
  int occ = 0;
  for (int s = t; s < S.n; s += nt) {
    const int a = STAGED ? (int)ls[s] : sorted[s];
    const int i = S.offset + a;
    float xi[2];
    V.pos(i, xi);
    const bool in_i = xi[0] >= 0.0f && xi[0] <= sp.L[0] && xi[1] >= 0.0f && xi[1] <= sp.L[1];
    int ci[2];
    cell_of<2>(xi, g, ci);  // the binning's cell
    const int hx = ci[0], hy = ci[1];
    // the stencil's columns and rows, wrapped by comparison (offsets of one)
    const int cx[3] = {hx == 0 ? g.cps[0] - 1 : hx - 1, hx, hx + 1 == g.cps[0] ? 0 : hx + 1};
    const int cy[3] = {hy == 0 ? g.cps[1] - 1 : hy - 1, hy, hy + 1 == g.cps[1] ? 0 : hy + 1};
    EnsRowOut out(idx, i, width, pad);
    for (int st = 0; st < 9; ++st) {  // iota order, x offset slowest
      const int c = cx[st / 3] + g.cps[0] * cy[st % 3];
      const int start = s_cs[c];
      const int m = min(s_cs[c + 1] - start, g.cap);
      const int k_first = ens_first_rank<STAGED>(start, m, g.cap, inv_cap);
      for (int q = 0; q < m; ++q) {  // slot order
        int k = q + k_first;
        k = k >= m ? k - m : k;
        const int jl = STAGED ? (int)ls[start + k] : sorted[start + k];
        if (jl == a) continue;  // mask_self
        float xj[2];
        V.pos(S.offset + jl, xj);
        const float r0 = fabsf(xj[0] - xi[0]), r1 = fabsf(xj[1] - xi[1]);
        const float e0 = fminf(r0, sp.L[0] - r0), e1 = fminf(r1, sp.L[1] - r1);
        const float d2 = fmaf(e1, e1, e0 * e0);
        const bool in = in_i && xj[0] >= 0.0f && xj[0] <= sp.L[0] && xj[1] >= 0.0f &&
                        xj[1] <= sp.L[1];
        bool keep = in && d2 < lo_thr;
        if (!keep && (!in || d2 <= hi_thr)) keep = ens_exact(xi, xj, sp, cutoff_sq);
        if (keep) out.put(S.offset + jl);
      }
    }
    out.close();
    occ = max(occ, out.cnt);
  }
  return wg_max(occ, s_red);
}

// A system's species matrices (sigma, epsilon, alpha in species mode, and
// the derivative coefficients dsig) copied to LDS, so that the pair loops
// read them there instead of gathering them per pair.  Returns s_par, or
// nullptr when the matrices are too large (the loops then read memory).
// Called by the whole workgroup.
__device__ __forceinline__ const float* ens_stage_params(const PairArgs& a,
                                                         const float* __restrict__ dsig,
                                                         float* s_par) {
  const int nn = a.ns * a.ns;
  if (a.ns < 1 || nn > kEnsParMax) return nullptr;
  for (int q = threadIdx.x; q < nn; q += blockDim.x) {
    s_par[q] = a.sig_mode == JMD_PARAM_SPECIES ? a.sig_v[q] : 0.0f;
    s_par[kEnsParMax + q] = a.eps_mode == JMD_PARAM_SPECIES ? a.eps_v[q] : 0.0f;
    s_par[2 * kEnsParMax + q] = a.alp_mode == JMD_PARAM_SPECIES ? a.alp_v[q] : 0.0f;
    s_par[3 * kEnsParMax + q] = dsig ? dsig[q] : 0.0f;
  }
  __syncthreads();
  return s_par;
}

// sigma, epsilon, alpha (which = 0, 1, 2) of pair (i, j), species matrices
// from LDS when staged.  PLAIN (ens_plain): epsilon scalar, alpha = 2, sigma
// scalar or staged; the row loops then hold no power function and no gathers
// of parameters (with them inlined four times a chunk the run kernel was
// 94 KB of code and spilled at 128 VGPRs).
template <bool PLAIN>
__device__ __forceinline__ float ens_pick(const PairArgs& a, int which, const float* par, int i,
                                          int j, int si, int sj) {
  if constexpr (PLAIN) {
    if (which == 0) return a.sig_mode == JMD_PARAM_SPECIES ? par[si * a.ns + sj] : a.sig;
    return which == 1 ? a.eps : 2.0f;
  }
  const int mode = which == 0 ? a.sig_mode : (which == 1 ? a.eps_mode : a.alp_mode);
  if (par && mode == JMD_PARAM_SPECIES) return par[which * kEnsParMax + si * a.ns + sj];
  return which == 0 ? pick(a.sig_mode, a.sig, a.sig_v, i, j, si, sj, a.ns)
                    : (which == 1 ? pick(a.eps_mode, a.eps, a.eps_v, i, j, si, sj, a.ns)
                                  : pick(a.alp_mode, a.alp, a.alp_v, i, j, si, sj, a.ns));
}

inline bool ens_plain(const PairArgs& a) {
  return a.eps_mode == JMD_PARAM_SCALAR && a.alp_mode == JMD_PARAM_SCALAR && a.alp == 2.0f &&
         (a.sig_mode == JMD_PARAM_SCALAR ||
          (a.sig_mode == JMD_PARAM_SPECIES && a.ns >= 1 && a.ns * a.ns <= kEnsParMax));
}

// dsig[si, sj], from LDS when staged.
__device__ __forceinline__ float ens_dsig(const PairArgs& a, const float* __restrict__ dsig,
                                          const float* par, int si, int sj) {
  return par ? par[3 * kEnsParMax + si * a.ns + sj] : dsig[si * a.ns + sj];
}

// One Dense row read kEnsRowChunk entries at a time: a 16-byte load where the
// row stride is a multiple of 4 entries, else single loads; pads past its end.
struct EnsRow {
  const int* row;
  int width, pad;
  bool vec;
  __device__ __forceinline__ EnsRow(const int* __restrict__ idx, int i, int w, int p)
      : row(idx + (long long)i * w), width(w), pad(p),
        vec((w & 3) == 0 && ((uintptr_t)idx & 15) == 0) {}
  __device__ __forceinline__ int4 chunk(int k) const {
    int4 q = make_int4(pad, pad, pad, pad);
    if (vec) {
      if (k < width) q = *reinterpret_cast<const int4*>(row + k);
    } else {
      if (k < width) q.x = row[k];
      if (k + 1 < width) q.y = row[k + 1];
      if (k + 2 < width) q.z = row[k + 2];
      if (k + 3 < width) q.w = row[k + 3];
    }
    return q;
  }
};

// Soft-sphere force of row i: two accumulators (entries k even / odd) summed
// in float64, as the Dense kernel's two lanes per row do; optional energy.
template <bool STAGED, bool PLAIN>
__device__ __forceinline__ void ens_force_row(int i, const EnsView<STAGED>& V,
                                              const int* __restrict__ idx, int width, int pad,
                                              const Space& sp, const PairArgs& a,
                                              const float* par, float* F, double* e) {
#pragma clang fp contract(off)
  const EnsRow R(idx, i, width, pad);
  float xi[2], xim[2];
  V.pos(i, xi);
  xim[0] = xi[0] - sp.L[0];
  xim[1] = xi[1] - sp.L[1];
  float f[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
  float en[2] = {0.0f, 0.0f};
  const int si = V.species(i);
  // The row in chunks: the chunk's ids, then all its gathers (position,
  // species), then the terms in entry order; a row ends at its first pad.
  int4 ids = R.chunk(0), next = R.chunk(kEnsRowChunk);
  for (int k0 = 0; k0 < width; k0 += kEnsRowChunk) {
    const int js[kEnsRowChunk] = {ids.x, ids.y, ids.z, ids.w};
    ids = next;
    next = R.chunk(k0 + 2 * kEnsRowChunk);
    int sjs[kEnsRowChunk];
    float xj[kEnsRowChunk][2];
#pragma unroll
    for (int c = 0; c < kEnsRowChunk; ++c) {
      xj[c][0] = xj[c][1] = 0.0f;
      sjs[c] = 0;
      if (js[c] != pad) {
        V.pos(js[c], xj[c]);
        sjs[c] = V.species(js[c]);
      }
    }
    bool end = false;
#pragma unroll
    for (int c = 0; c < kEnsRowChunk; ++c) {
      const int j = js[c];
      if (j == pad) {
        end = true;
        break;
      }
      float d[2];
      d[0] = min_image_disp(xj[c][0], xi[0], xim[0], sp.L[0], sp.half[0]);
      d[1] = min_image_disp(xj[c][1], xi[1], xim[1], sp.L[1], sp.half[1]);
      const float r2 = fmaf(d[1], d[1], d[0] * d[0]);
      const int sj = sjs[c];
      const float sig = ens_pick<PLAIN>(a, 0, par, i, j, si, sj);
      const float eps = ens_pick<PLAIN>(a, 1, par, i, j, si, sj);
      const float alp = ens_pick<PLAIN>(a, 2, par, i, j, si, sj);
      float dEr;
      const float u = pair_eval<JMD_SOFT_SPHERE>(r2, sig, eps, alp, a, &dEr);
      const int l = c & 1;  // k0 is even: the parity of k = k0 + c
      f[l][0] = fmaf(dEr, d[0], f[l][0]);
      f[l][1] = fmaf(dEr, d[1], f[l][1]);
      en[l] += u;
    }
    if (end) break;
  }
  F[0] = (float)((double)f[0][0] + (double)f[1][0]);
  F[1] = (float)((double)f[0][1] + (double)f[1][1]);
  if (e) *e += 0.5 * ((double)en[0] + (double)en[1]);
}

// Copies a system's rows between two Dense lists of one width, 16 bytes at a
// time where the rows allow it.
__device__ __forceinline__ void ens_copy_rows(const EnsSys& S, int* __restrict__ to,
                                              const int* __restrict__ from, int width) {
  const long long base = (long long)S.offset * width, rows = (long long)S.n * width;
  if ((width & 3) == 0 && (((uintptr_t)to | (uintptr_t)from) & 15) == 0) {
    const int4* src = reinterpret_cast<const int4*>(from + base);
    int4* dst = reinterpret_cast<int4*>(to + base);
#pragma unroll 4
    for (long long q = threadIdx.x; q < rows / 4; q += blockDim.x) dst[q] = src[q];
  } else {
#pragma unroll 4
    for (long long q = threadIdx.x; q < rows; q += blockDim.x) to[base + q] = from[base + q];
  }
}

// STAGED: the systems of at most lds_n particles, kept in LDS; else the
// larger ones, read from global memory.  Each instance skips the other's.
template <bool STAGED, bool PLAIN, bool RUN>
__global__ __launch_bounds__(kEnsThreads, kEnsWaves) void k_fire_ensemble(
    const EnsSys* __restrict__ systems, const int* __restrict__ order, int nsys, int ntot,
    int mode, int n_steps, double* __restrict__ x_hi, float* __restrict__ x,
    float* __restrict__ p, float* __restrict__ F, float* __restrict__ x_ref,
    int* __restrict__ idx, int width, int* __restrict__ scratch, PairArgs a0, FireP prm,
    float* __restrict__ fire_state, int* __restrict__ fire_npos, uint8_t* __restrict__ error,
    int* __restrict__ out_stat, double* __restrict__ energy, int* __restrict__ builds,
    EnsTape tape, int lds_n) {
  __shared__ int s_cs[kEnsMaxCells + 1];
  // dynamic LDS: [2 lds_n] float32 positions, [lds_n] uint16 cell-sorted
  // ids, [lds_n] uint8 species ids
  extern __shared__ float4 s_dyn[];
  __shared__ int s_red[kEnsThreads / kWave];
  __shared__ double s_d[3 * (kEnsThreads / kWave)];
  __shared__ float s_scal[4];  // dt, alpha, ratio, keep
  __shared__ int s_flag;
  const int sid = order[blockIdx.x];
  if (sid < 0 || sid >= nsys) return;
  const EnsSys S = systems[sid];
  if (STAGED != (S.n <= lds_n)) return;  // the other instance's system
  const int t = threadIdx.x, nt = blockDim.x;
  const float cutoff_sq = S.cutoff_sq, thr_sq = S.threshold_sq;
  PairArgs a = a0;  // this system's parameter block
  if (a.sig_mode == JMD_PARAM_SPECIES) a.sig_v += S.param_offset;
  if (a.eps_mode == JMD_PARAM_SPECIES) a.eps_v += S.param_offset;
  if (a.alp_mode == JMD_PARAM_SPECIES) a.alp_v += S.param_offset;
  __shared__ float s_par[4 * kEnsParMax];
  const float* par = ens_stage_params(a, nullptr, s_par);
  // A staged system keeps a copy of its positions (and species ids, when
  // they fit a byte) and its cell-sorted ids in LDS for the list and pair
  // loops; the integrator writes both position copies.
  float* lx = STAGED ? reinterpret_cast<float*>(s_dyn) : nullptr;
  uint16_t* lsorted = STAGED ? reinterpret_cast<uint16_t*>(lx + 2 * lds_n) : nullptr;
  uint8_t* lsp = STAGED && a.species && a.ns <= 256
                     ? reinterpret_cast<uint8_t*>(lsorted + lds_n) : nullptr;
  if constexpr (STAGED) {
    for (int k = threadIdx.x; k < 2 * S.n; k += blockDim.x) lx[k] = x[2LL * S.offset + k];
    if (lsp)
      for (int q = threadIdx.x; q < S.n; q += blockDim.x)
        lsp[q] = (uint8_t)a.species[S.offset + q];
    __syncthreads();
  }
  const EnsView<STAGED> V{x, lx, a.species, lsp, S.offset};
  int* cellp = scratch + S.offset;
  int* rankp = scratch + ntot + S.offset;
  int* sorted = scratch + 2LL * ntot + S.offset;
  Space sp;
  sp.dim = 2;
  sp.periodic = 1;
  sp.general = 0;
  for (int d = 0; d < 3; ++d) {
    sp.L[d] = d < 2 ? S.side[d] : 1.0f;
    sp.half[d] = sp.L[d] * 0.5f;
  }
  Grid g;
  g.cps[0] = S.cps[0];
  g.cps[1] = S.cps[1];
  g.cps[2] = 1;
  g.cell_size[0] = S.cell_size[0];
  g.cell_size[1] = S.cell_size[1];
  g.cell_size[2] = 1.0f;
  g.ncell = S.cps[0] * S.cps[1];
  g.cap = S.cap;
  const int pad = ntot;

  if (!RUN && mode == ENS_FILL) {
    Grid g2 = g;
    g2.cps[0] = S.fill_cps[0];
    g2.cps[1] = S.fill_cps[1];
    g2.cell_size[0] = S.fill_cell_size[0];
    g2.cell_size[1] = S.fill_cell_size[1];
    g2.ncell = g2.cps[0] * g2.cps[1];
    bool all_in;
    const int fill = ens_bin(S, g2, sp, V, cellp, rankp, sorted, s_cs, s_red, lsorted, &all_in);
    if (t == 0) out_stat[sid] = fill;
    return;
  }

  uint8_t err = 0;
  int nbuilds = 0;
  int* list = idx;    // the rows a rebuild writes and the forces read
  int list_slot = 0;  // its tape slot (record_node(0) fills 0)
  // list build at the current positions (allocate / update)
  auto rebuild = [&](bool store) {
    bool all_in;
    const int fill = ens_bin(S, g, sp, V, cellp, rankp, sorted, s_cs, s_red, lsorted, &all_in);
    const int occ = ens_rows(S, g, sp, cutoff_sq, V, sorted, s_cs, list,
                             store ? width : 0, pad, s_red, lsorted, all_in, fill);
    if (fill > g.cap) err |= JMD_CELL_LIST_OVERFLOW;
    if (occ > S.max_occ) err |= JMD_NEIGHBOR_LIST_OVERFLOW;
    for (int q = t; q < S.n; q += nt) {
      float xi[2];
      V.pos(S.offset + q, xi);
      store_pos<2>(x_ref, S.offset + q, xi);
    }
    ++nbuilds;
    return occ;
  };

  if (!RUN && mode == ENS_OCCUPANCY) {
    const int occ = rebuild(false);
    if (t == 0) out_stat[sid] = occ;
    return;
  }

  const double L0 = S.side[0], L1 = S.side[1];
  if (!RUN) {  // ENS_INIT
    rebuild(true);
    __syncthreads();
    double e = 0.0, z1 = 0.0, z2 = 0.0;
    for (int q = t; q < S.n; q += nt) {
      const int i = S.offset + q;
      float f[2];
      ens_force_row<STAGED, PLAIN>(i, V, idx, width, pad, sp, a, par, f, &e);
      F[2LL * i] = f[0];
      F[2LL * i + 1] = f[1];
      p[2LL * i] = 0.0f;
      p[2LL * i + 1] = 0.0f;
    }
    wg_sum3(e, z1, z2, s_d);
    if (t == 0) {
      fire_state[2 * sid] = prm.dt_start;
      fire_state[2 * sid + 1] = prm.alpha_start;
      fire_npos[sid] = 0;
      energy[sid] = e;
      error[sid] = (uint8_t)(error[sid] | err);
      builds[sid] += nbuilds;
    }
    return;
  }

  // ENS_RUN
  if (t == 0) {
    s_scal[0] = fire_state[2 * sid];
    s_scal[1] = fire_state[2 * sid + 1];
    s_flag = fire_npos[sid];
  }
  __syncthreads();
  int n_pos = s_flag;
  const long long n2 = 2LL * ntot;
  auto record_node = [&](int k) {  // x, F, list at node k of the segment
    for (int q = t; q < 2 * S.n; q += nt) {
      const long long g = 2LL * S.offset + q;
      tape.x[k * n2 + g] = x[g];
      tape.F[k * n2 + g] = F[g];
    }
    ens_copy_rows(S, tape.idx + (long long)k * ntot * width, idx, width);
  };
  if (tape.x) record_node(0);
  // a taped segment keeps its current list in the tape's slot (a rebuild then
  // writes the next slot and nothing is copied); idx gets the last one at the
  // end
  // The half-step pass also makes the next step's skin test (on the
  // positions it writes, against the reference positions, which only a
  // rebuild changes, before the half-step) and applies the previous step's
  // FIRE mixing to each momentum it reads (the mixing needs the step's
  // reductions, so it waits for the next pass over the momenta); the
  // per-element arithmetic is that of the separate passes.
  // the pending mixing's ratio, keep and alpha (workgroup-uniform: in LDS,
  // out of the registers the force loop needs)
  __shared__ double s_mix[3];
  bool moved_next = false;
  bool mix_pending = false;
  for (int step = 0; step < n_steps; ++step) {
    // neighbour update: rebuild when any particle moved beyond half the skin
    bool moved = moved_next;
    if (step == 0) {
#pragma unroll 4
      for (int q = t; q < S.n; q += nt) {
        float xi[2], ri[2];
        V.pos(S.offset + q, xi);
        load_pos<2>(x_ref, S.offset + q, ri);
        moved = moved || ref_metric_sq<2>(xi, ri, sp) > thr_sq;
      }
    }
    const bool rebuilt = __syncthreads_or(moved);
    if (rebuilt) {
      if (tape.x) {  // the list the force at node step + 1 will use
        list_slot = step + 1;
        list = tape.idx + (long long)list_slot * ntot * width;
      }
      rebuild(true);
    }
    __syncthreads();
    // velocity-Verlet sub-step at the FIRE time step (float16 value), one
    // particle per iteration
    const float dt = s_scal[0];
    const float half = dt / 2.0f;
    const double mix_ratio = s_mix[0], mix_keep = s_mix[1];
    const float mix_alpha = (float)s_mix[2];
    moved_next = false;
    // two particles at a time, all their loads before any store
    for (int q0 = t; q0 < S.n; q0 += 2 * nt) {
      float pq[2][2], fq[2][2], ri[2][2];
      double xq[2][2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int q = min(q0 + u * nt, S.n - 1);
        const long long g0 = 2LL * (S.offset + q);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          pq[u][c] = p[g0 + c];
          fq[u][c] = F[g0 + c];
          xq[u][c] = x_hi[g0 + c];
        }
        load_pos<2>(x_ref, S.offset + q, ri[u]);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int q = q0 + u * nt;
        if (q >= S.n) break;
        const long long g0 = 2LL * (S.offset + q);
        float xn[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const long long gq = g0 + c;
          float p0 = pq[u][c];
          if (mix_pending) {  // the previous step's FIRE mixing
            double pv = p0;
            pv = pv + (double)mix_alpha * ((double)fq[u][c] * mix_ratio - pv);
            p0 = (float)(pv * mix_keep);
          }
          const float pk = p0 + half * fq[u][c];
          double xv = xq[u][c] + (double)dt * (double)pk;
          xv = ens_mod64(xv, c ? L1 : L0);
          p[gq] = pk;
          x_hi[gq] = xv;
          xn[c] = (float)xv;
          x[gq] = xn[c];
          if constexpr (STAGED) lx[2 * q + c] = xn[c];
        }
        moved_next = moved_next || ref_metric_sq<2>(xn, ri[u], sp) > thr_sq;
      }
    }
    __syncthreads();
    // forces of the new positions, the second half kick and the FIRE sums
    double ff = 0.0, pp = 0.0, fp = 0.0;
    for (int q = t; q < S.n; q += nt) {
      const int i = S.offset + q;
      float pk[2], f[2];
      load_pos<2>(p, i, pk);
      ens_force_row<STAGED, PLAIN>(i, V, list, width, pad, sp, a, par, f, nullptr);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        pk[c] = pk[c] + half * f[c];
        const double fv = f[c], pv = pk[c];
        ff += fv * fv;
        pp += pv * pv;
        fp += fv * pv;
      }
      store_pos<2>(F, i, f);
      store_pos<2>(p, i, pk);
      if (tape.x) {
        const long long g0 = 2LL * i;
        float xi[2];
        V.pos(i, xi);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          tape.q[step * n2 + g0 + c] = pk[c];
          tape.x[(step + 1) * n2 + g0 + c] = xi[c];
          tape.F[(step + 1) * n2 + g0 + c] = f[c];
        }
      }
    }
    wg_sum3(ff, pp, fp, s_d);
    // FIRE bookkeeping (minimize.py:190-219) with float16 dt / alpha
    const double ratio = sqrt(pp) / sqrt(ff + 1e-6);
    const float alpha_mix = s_scal[1];
    const double keep = fp >= 0.0 ? 1.0 : 0.0;
    if (tape.x && t == 0) {
      float* sc = tape.sc + ((long long)step * nsys + sid) * kTapeScalars;
      sc[0] = dt;
      sc[1] = alpha_mix;
      sc[2] = (float)keep;
      sc[3] = (float)sqrt(pp);
      sc[4] = (float)sqrt(ff + 1e-6);
      sc[5] = (float)list_slot;
    }
    n_pos = fp >= 0.0 ? n_pos + 1 : 0;
    __syncthreads();
    if (t == 0) {
      float dtn = s_scal[0], al = s_scal[1];
      if (fp > 0.0 && n_pos > prm.n_min) dtn = fminf(f16r(dtn * prm.f_inc), prm.dt_max);
      if (fp < 0.0) dtn = f16r(dtn * prm.f_dec);
      if (fp > 0.0 && n_pos > prm.n_min) al = f16r(al * prm.f_alpha);
      if (fp < 0.0) al = prm.alpha_start;
      s_scal[0] = dtn;
      s_scal[1] = al;
      s_mix[0] = ratio;
      s_mix[1] = keep;
      s_mix[2] = (double)alpha_mix;
    }
    mix_pending = true;  // applied by the next half-step, or below
    __syncthreads();
  }
  if (mix_pending) {  // the last step's FIRE mixing
    const double mix_ratio = s_mix[0], mix_keep = s_mix[1];
    const float mix_alpha = (float)s_mix[2];
#pragma unroll 4
    for (int k = t; k < 2 * S.n; k += nt) {
      const long long q = 2LL * S.offset + k;
      double pv = p[q];
      pv = pv + (double)mix_alpha * ((double)F[q] * mix_ratio - pv);
      p[q] = (float)(pv * mix_keep);
    }
    __syncthreads();
  }
  double e = 0.0, z1 = 0.0, z2 = 0.0;
  for (int q = t; q < S.n; q += nt) {
    float f[2];
    ens_force_row<STAGED, PLAIN>(S.offset + q, V, list, width, pad, sp, a, par, f, &e);
  }
  if (list != idx) ens_copy_rows(S, idx, list, width);
  wg_sum3(e, z1, z2, s_d);
  if (t == 0) {
    fire_state[2 * sid] = s_scal[0];
    fire_state[2 * sid + 1] = s_scal[1];
    fire_npos[sid] = n_pos;
    energy[sid] = e;
    error[sid] = (uint8_t)(error[sid] | err);
    builds[sid] += nbuilds;
  }
}

// ---------------------------------------------------------------------------
// Adjoint of the FIRE trajectory (per system, one workgroup each)
//
// Forward step k (dt, alpha, keep from the tape; float16 bookkeeping is
// piecewise constant and carries no derivative):
//   ph = p_k + h F_k,  x_{k+1} = x_k + dt ph,  F' = F(x_{k+1}),  q = ph + h F',
//   p_{k+1} = keep ((1 - alpha) q + alpha |q| / sqrt(|F'|^2 + 1e-6) F').
// Backward, with X, P the adjoints of x, p and W the pending vector of node
// k + 1 (W = h PH of the step after):
//   G = keep P,  s1 = F'.G,
//   Q  = (1 - alpha) G + alpha s1 q / (|q| sqrt(ff)),
//   Fb = alpha |q|/sqrt(ff) G - alpha s1 |q| F' / sqrt(ff)^3 + h Q,
//   X += J(x_{k+1}) (Fb + W),  theta += (Fb + W)^T dF(x_{k+1})/dtheta,
//   P = Q + dt X,  W = h P.
// One product with the force Jacobian per step.  The loss is
// scale * sum_s E_s(x_T), theta the derivative with respect to each system's
// parameter (the species matrix's derivative coefficients dsigma/dtheta).
//
// Box adjoint (optional): the derivative with respect to the side L of each
// system's square, positions held in real coordinates.  L enters through the
// minimum image, d = x_j - x_i - L n (n the pair's integer image vector, so
// dd/dL = -n), and through the fold of the shift, x_{k+1} = x_k + dt ph -
// L m_k (m_k = rint((x_k - x_{k+1}) / L), a step being far shorter than L/2):
//   Lb  = -scale/2 sum_ij g (d.n)                           at x_T,
//   Lb += -sum_ij V_i.(g n + 2 g' (d.n) d)    at every node (V = Fb + W),
//   Lb += -X_{k+1}.m_k                        for every step.
// ---------------------------------------------------------------------------

enum { BACK_INIT = 0, BACK_STEPS = 1, BACK_FINISH = 2 };

// Integer image of a pair along one axis: the fold min_image_disp applied to
// raw = x_j - x_i (d = raw - n L).
__device__ __forceinline__ float image_of(float raw, float half) {
  return raw >= half ? 1.0f : (raw < -half ? -1.0f : 0.0f);
}

// h_i = (J v)_i over the system's rows at positions x with list idx; returns
// this thread's share of v^T dF/dtheta (rows it owns) and, with box, adds its
// share of v^T dF/dL to lacc.
template <bool STAGED, bool PLAIN>
__device__ __forceinline__ double ens_hvp_rows(const EnsSys& S, const Space& sp,
                                               const PairArgs& a, const float* par,
                                               const float* __restrict__ dsig,
                                               const EnsView<STAGED>& XV,
                                               const int* __restrict__ idx, int width, int pad,
                                               const EnsView<STAGED>& VV,
                                               double* __restrict__ X, bool box,
                                               double& lacc) {
#pragma clang fp contract(off)
  double tacc = 0.0;
  for (int q = threadIdx.x; q < S.n; q += blockDim.x) {
    const int i = S.offset + q;
    float xi[2], xim[2], vi[2];
    XV.pos(i, xi);
    VV.pos(i, vi);
    xim[0] = xi[0] - sp.L[0];
    xim[1] = xi[1] - sp.L[1];
    const int si = XV.species(i);
    float h0 = 0.0f, h1 = 0.0f, tp = 0.0f, lp = 0.0f;
    const EnsRow R(idx, i, width, pad);
    int4 ids = R.chunk(0), next = R.chunk(kEnsRowChunk);
    // the row in chunks: ids, then their gathers, then the terms in order
    for (int k0 = 0; k0 < width; k0 += kEnsRowChunk) {
      const int js[kEnsRowChunk] = {ids.x, ids.y, ids.z, ids.w};
      ids = next;
      next = R.chunk(k0 + 2 * kEnsRowChunk);
      int sjs[kEnsRowChunk];
      float xj[kEnsRowChunk][2], vj[kEnsRowChunk][2];
#pragma unroll
      for (int c = 0; c < kEnsRowChunk; ++c) {
        xj[c][0] = xj[c][1] = vj[c][0] = vj[c][1] = 0.0f;
        sjs[c] = 0;
        if (js[c] != pad) {
          XV.pos(js[c], xj[c]);
          VV.pos(js[c], vj[c]);
          sjs[c] = XV.species(js[c]);
        }
      }
      bool end = false;
#pragma unroll
      for (int c = 0; c < kEnsRowChunk; ++c) {
        const int j = js[c];
        if (j == pad) {
          end = true;
          break;
        }
        float d[2], w[2];
        d[0] = min_image_disp(xj[c][0], xi[0], xim[0], sp.L[0], sp.half[0]);
        d[1] = min_image_disp(xj[c][1], xi[1], xim[1], sp.L[1], sp.half[1]);
        w[0] = vj[c][0] - vi[0];
        w[1] = vj[c][1] - vi[1];
        const float r2 = fmaf(d[1], d[1], d[0] * d[0]);
        const int sj = sjs[c];
        const float sig = ens_pick<PLAIN>(a, 0, par, i, j, si, sj);
        const float eps = ens_pick<PLAIN>(a, 1, par, i, j, si, sj);
        const float alp = ens_pick<PLAIN>(a, 2, par, i, j, si, sj);
        const PairD2 D = pair_eval2<JMD_SOFT_SPHERE>(r2, sig, eps, alp, a);
        const float dw = fmaf(d[1], w[1], d[0] * w[0]);
        const float tt = 2.0f * D.gp * dw;
        h0 = fmaf(D.g, w[0], fmaf(tt, d[0], h0));
        h1 = fmaf(D.g, w[1], fmaf(tt, d[1], h1));
        if (dsig) {
          const float cc = ens_dsig(a, dsig, par, si, sj);
          const float lam = fmaf(vi[1], d[1], vi[0] * d[0]);
          tp = fmaf(cc * D.gs, lam, tp);
        }
        if (box) {
          const float n0 = image_of(xj[c][0] - xi[0], sp.half[0]);
          const float n1 = image_of(xj[c][1] - xi[1], sp.half[1]);
          const float dn = fmaf(d[1], n1, d[0] * n0);
          const float vn = fmaf(vi[1], n1, vi[0] * n0);
          const float vd = fmaf(vi[1], d[1], vi[0] * d[0]);
          lp = fmaf(D.g, vn, fmaf(2.0f * D.gp * dn, vd, lp));
        }
      }
      if (end) break;
    }
    X[2LL * i] += (double)h0;
    X[2LL * i + 1] += (double)h1;
    tacc += (double)tp;
    lacc -= (double)lp;
  }
  return tacc;
}

// STAGED: systems of at most lds_n particles, with the positions of the
// node and the vector of each Jacobian product copied to LDS; else the
// larger ones, read from memory.  Each instance skips the other's systems.
template <bool STAGED, bool PLAIN>
__global__ __launch_bounds__(kEnsThreads, kEnsWaves) void k_fire_ensemble_back(
    const EnsSys* __restrict__ systems, int nsys, int ntot, int mode, int K,
    const float* __restrict__ x, const float* __restrict__ F, const int* __restrict__ idx,
    int width, PairArgs a0, const float* __restrict__ dsig0, EnsTape tape,
    double* __restrict__ X, double* __restrict__ P, float* __restrict__ W,
    float* __restrict__ V, double* __restrict__ theta, double* __restrict__ box_adj,
    float scale, int lds_n) {
#pragma clang fp contract(off)
  // dynamic LDS: [2 lds_n] positions, [2 lds_n] product vector, [lds_n]
  // uint8 species ids
  extern __shared__ float4 s_dynb[];
  __shared__ double s_d[3 * (kEnsThreads / kWave)];
  const int sid = blockIdx.x;
  if (sid >= nsys) return;
  const EnsSys S = systems[sid];
  if (STAGED != (S.n <= lds_n)) return;  // the other instance's system
  const int t = threadIdx.x, nt = blockDim.x;
  PairArgs a = a0;
  if (a.sig_mode == JMD_PARAM_SPECIES) a.sig_v += S.param_offset;
  if (a.eps_mode == JMD_PARAM_SPECIES) a.eps_v += S.param_offset;
  if (a.alp_mode == JMD_PARAM_SPECIES) a.alp_v += S.param_offset;
  const float* dsig = dsig0 ? dsig0 + S.param_offset : nullptr;
  __shared__ float s_par[4 * kEnsParMax];
  const float* par = ens_stage_params(a, dsig, s_par);
  float* lx = STAGED ? reinterpret_cast<float*>(s_dynb) : nullptr;
  float* lv = STAGED ? lx + 2 * lds_n : nullptr;
  uint8_t* lsp = STAGED && a.species && a.ns <= 256
                     ? reinterpret_cast<uint8_t*>(lv + 2 * lds_n) : nullptr;
  if (lsp)
    for (int q = t; q < S.n; q += nt) lsp[q] = (uint8_t)a.species[S.offset + q];
  Space sp;
  sp.dim = 2;
  sp.periodic = 1;
  sp.general = 0;
  for (int d = 0; d < 3; ++d) {
    sp.L[d] = d < 2 ? S.side[d] : 1.0f;
    sp.half[d] = sp.L[d] * 0.5f;
  }
  const int pad = ntot;
  const long long n2 = 2LL * ntot;
  const long long b2 = 2LL * S.offset;
  const bool box = box_adj != nullptr;

  if (mode == BACK_INIT) {  // X = -scale F, P = W = 0, theta = scale dE/dtheta
    double e = 0.0, el = 0.0, z2 = 0.0;
    for (int k = t; k < 2 * S.n; k += nt) {
      X[b2 + k] = -(double)scale * (double)F[b2 + k];
      P[b2 + k] = 0.0;
      W[b2 + k] = 0.0f;
    }
    if (dsig || box) {
      for (int q = t; q < S.n; q += nt) {
        const int i = S.offset + q;
        float xi[2], xim[2];
        load_pos<2>(x, i, xi);
        xim[0] = xi[0] - sp.L[0];
        xim[1] = xi[1] - sp.L[1];
        const int si = a.species ? a.species[i] : 0;
        const int* row = idx + (long long)i * width;
        for (int k = 0; k < width; ++k) {
          const int j = row[k];
          if (j == pad) break;
          float xj[2], d[2];
          load_pos<2>(x, j, xj);
          d[0] = min_image_disp(xj[0], xi[0], xim[0], sp.L[0], sp.half[0]);
          d[1] = min_image_disp(xj[1], xi[1], xim[1], sp.L[1], sp.half[1]);
          const float r2 = fmaf(d[1], d[1], d[0] * d[0]);
          const int sj = a.species ? a.species[j] : 0;
          const float sig = ens_pick<PLAIN>(a, 0, par, i, j, si, sj);
          const float eps = ens_pick<PLAIN>(a, 1, par, i, j, si, sj);
          const float alp = ens_pick<PLAIN>(a, 2, par, i, j, si, sj);
          const PairD2 D = pair_eval2<JMD_SOFT_SPHERE>(r2, sig, eps, alp, a);
          if (dsig) e += 0.5 * (double)(ens_dsig(a, dsig, par, si, sj) * D.us);
          if (box) {
            const float n0 = image_of(xj[0] - xi[0], sp.half[0]);
            const float n1 = image_of(xj[1] - xi[1], sp.half[1]);
            el -= 0.5 * (double)(D.g * fmaf(d[1], n1, d[0] * n0));
          }
        }
      }
    }
    wg_sum3(e, el, z2, s_d);
    if (t == 0) {
      theta[sid] = (double)scale * e;
      if (box) box_adj[sid] = (double)scale * el;
    }
    return;
  }
  if (mode == BACK_FINISH) {  // pending W applied at node 0 of the tape
    double el = 0.0, z2 = 0.0;
    if constexpr (STAGED) {
      for (int m = t; m < 2 * S.n; m += nt) {
        lx[m] = tape.x[b2 + m];
        lv[m] = W[b2 + m];
      }
    }
    __syncthreads();
    const EnsView<STAGED> XV{tape.x, lx, a.species, lsp, S.offset};
    const EnsView<STAGED> VV{W, lv, nullptr, nullptr, S.offset};
    double e = ens_hvp_rows<STAGED, PLAIN>(S, sp, a, par, dsig, XV, tape.idx, width, pad, VV, X, box, el);
    wg_sum3(e, el, z2, s_d);
    if (t == 0) {
      theta[sid] += e;
      if (box) box_adj[sid] += el;
    }
    return;
  }
  double tsum = 0.0, lsum = 0.0;
  // s1 = F'.G of the next step to be taken back: the pass that finishes P
  // for it (3) also makes its sum, so P and F' are read once a step
  double s1n = 0.0;
  if (K > 0) {
    const float keep = tape.sc[((long long)(K - 1) * nsys + sid) * kTapeScalars + 2];
    const float* Fn = tape.F + (long long)K * n2;
#pragma unroll 4
    for (int m = t; m < 2 * S.n; m += nt) s1n += (double)Fn[b2 + m] * (double)keep * P[b2 + m];
  }
  for (int k = K - 1; k >= 0; --k) {
    const float* sc = tape.sc + ((long long)k * nsys + sid) * kTapeScalars;
    const float dt = sc[0], alpha = sc[1], keep = sc[2];
    const double spp = sc[3], sff = sc[4];
    const float h = dt / 2.0f;
    const float* __restrict__ Fn = tape.F + (long long)(k + 1) * n2;
    const float* __restrict__ qk = tape.q + (long long)k * n2;
    // (1) FIRE mixing, backward
    double s1 = s1n, z1 = 0.0, z2 = 0.0;
    wg_sum3(s1, z1, z2, s_d);
    const double ratio = spp / sff;
    const double cq = spp > 0.0 ? (double)alpha * s1 / (spp * sff) : 0.0;
    const double cf = (double)alpha * s1 * spp / (sff * sff * sff);
    const float* __restrict__ xn = tape.x + (long long)(k + 1) * n2;
    // four elements at a time, their loads before any store (one at a time
    // the pass waited for memory once an element)
    for (int m0 = t; m0 < 2 * S.n; m0 += kEnsBatch * nt) {
      double Pm[kEnsBatch];
      float qm[kEnsBatch], Fm[kEnsBatch], Wm[kEnsBatch], xm[kEnsBatch];
#pragma unroll
      for (int u = 0; u < kEnsBatch; ++u) {
        const long long g = b2 + min(m0 + u * nt, 2 * S.n - 1);
        Pm[u] = P[g];
        qm[u] = qk[g];
        Fm[u] = Fn[g];
        Wm[u] = W[g];
        xm[u] = STAGED ? xn[g] : 0.0f;
      }
#pragma unroll
      for (int u = 0; u < kEnsBatch; ++u) {
        const int m = m0 + u * nt;
        if (m >= 2 * S.n) break;
        const double G = (double)keep * Pm[u];
        const double Q = (1.0 - (double)alpha) * G + cq * (double)qm[u];
        const double Fb = (double)alpha * ratio * G - cf * (double)Fm[u] + (double)h * Q;
        P[b2 + m] = Q;  // PH until step (3)
        const float vg = (float)(Fb + (double)Wm[u]);
        if constexpr (STAGED) {
          lv[m] = vg;
          lx[m] = xm[u];
        } else {
          V[b2 + m] = vg;
        }
      }
    }
    __syncthreads();
    // (2) product with the force Jacobian at node k + 1
    const EnsView<STAGED> XV{xn, lx, a.species, lsp, S.offset};
    const EnsView<STAGED> VV{V, lv, nullptr, nullptr, S.offset};
    tsum += ens_hvp_rows<STAGED, PLAIN>(S, sp, a, par, dsig, XV,
                                        tape.idx + (long long)sc[5] * ntot * width, width, pad,
                                        VV, X, box, lsum);
    __syncthreads();
    // (3) x_{k+1} = x_k + dt ph - L m_k, ph = p_k + h F_k
    const float* __restrict__ xk = tape.x + (long long)k * n2;
    const float* __restrict__ Fk = tape.F + (long long)k * n2;
    const double keepn = k > 0 ? (double)sc[2 - (long long)nsys * kTapeScalars] : 0.0;
    s1n = 0.0;
    for (int m0 = t; m0 < 2 * S.n; m0 += kEnsBatch * nt) {
      double Pm[kEnsBatch], Xm[kEnsBatch];
      float Fm[kEnsBatch], xm[kEnsBatch], x1[kEnsBatch];
#pragma unroll
      for (int u = 0; u < kEnsBatch; ++u) {
        const long long g = b2 + min(m0 + u * nt, 2 * S.n - 1);
        Pm[u] = P[g];
        Xm[u] = X[g];
        Fm[u] = Fk[g];
        xm[u] = x1[u] = 0.0f;
        if (box) {
          xm[u] = xk[g];
          x1[u] = xn[g];
        }
      }
#pragma unroll
      for (int u = 0; u < kEnsBatch; ++u) {
        const int m = m0 + u * nt;
        if (m >= 2 * S.n) break;
        if (box) {
          const float fold = rintf((xm[u] - x1[u]) / ((m & 1) ? sp.L[1] : sp.L[0]));
          lsum -= Xm[u] * (double)fold;
        }
        const double PH = Pm[u] + (double)dt * Xm[u];
        P[b2 + m] = PH;
        W[b2 + m] = (float)((double)h * PH);
        s1n += (double)Fm[u] * keepn * PH;
      }
    }
    // end of step k, backward
    __syncthreads();
  }
  double e = tsum, el = lsum, z2 = 0.0;
  wg_sum3(e, el, z2, s_d);
  if (t == 0) {
    theta[sid] += e;
    if (box) box_adj[sid] += el;
  }
}

}  // namespace jmd

using namespace jmd;

extern "C" {

// Allows a staged kernel more than the default dynamic LDS, once per device
// and size (the largest size granted so far is kept per device).
static bool ens_lds_allow(const void* kernel, size_t* granted, size_t bytes) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
  if (bytes <= granted[dev]) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) !=
      hipSuccess)
    return false;
  granted[dev] = bytes;
  return true;
}

int jmd_fire_ensemble_2d(const jmd_system2d* systems, const int32_t* order, int32_t n_systems,
                         int64_t n_total, int32_t mode, int32_t n_steps, double* position_hi,
                         float* position, float* momentum, float* force,
                         float* reference_position, int32_t* idx, int32_t width,
                         int32_t* scratch, const jmd_pair_potential* potential,
                         const float* fire_params, float* fire_state, int32_t* fire_n_pos,
                         uint8_t* error, int32_t* out_stat, double* energy, int32_t* builds,
                         float* tape_x, float* tape_force, float* tape_q, int32_t* tape_idx,
                         float* tape_scalars, void* stream) {
  const int asked = mode >> 8;
  if (mode < 0 || !ens_threads_ok(asked)) return JMD_ERR_INVALID;
  mode &= 0xff;
  if (n_systems < 0 || n_total < 0 || n_total >= 0x7fffffff || width < 0 || n_steps < 0 ||
      mode > ENS_RUN || !fire_params)
    return JMD_ERR_INVALID;
  if (n_systems == 0) return JMD_OK;
  if (!systems || !order || !position || !scratch || !error || !builds) return JMD_ERR_INVALID;
  if ((mode == ENS_FILL || mode == ENS_OCCUPANCY) && !out_stat) return JMD_ERR_INVALID;
  if (mode >= ENS_INIT && (!position_hi || !momentum || !force || !reference_position ||
                           !idx || !fire_state || !fire_n_pos || !energy || width < 1))
    return JMD_ERR_INVALID;
  if (mode == ENS_OCCUPANCY && !reference_position) return JMD_ERR_INVALID;
  PairArgs a;
  if (!make_pair_args(potential, &a) || a.kind != JMD_SOFT_SPHERE) return JMD_ERR_INVALID;
  FireP prm{fire_params[0], fire_params[1], (int)fire_params[2], fire_params[3],
            fire_params[4], fire_params[5], fire_params[6]};
  static_assert(sizeof(jmd_system2d) == sizeof(EnsSys), "system record layout");
  const bool taped = tape_x != nullptr;
  if (taped && (mode != ENS_RUN || !tape_force || !tape_q || !tape_idx || !tape_scalars))
    return JMD_ERR_INVALID;
  EnsTape tape{tape_x, tape_force, tape_q, tape_idx, tape_scalars, n_steps};
  // LDS copy of each system's positions, cell-sorted ids and species ids:
  // systems of up to 8 particles per thread (8 Ki per 1024-thread workgroup,
  // one per CU; 4 Ki per 512, two per CU); larger systems use global memory
  const int threads = ens_launch_threads(asked, n_systems, n_total);
  const int lds_n = threads * kEnsPerThread;
  const size_t lds_bytes = (size_t)lds_n * (2 * sizeof(float) + sizeof(uint16_t) + 1);
  // run mode with the common parameters has row loops without the general
  // ones; the measuring and initial launches keep one form
  const bool run = mode == ENS_RUN, plain = run && ens_plain(a);
  const auto staged = plain ? k_fire_ensemble<true, true, true>
                            : (run ? k_fire_ensemble<true, false, true>
                                   : k_fire_ensemble<true, false, false>);
  const auto memory = plain ? k_fire_ensemble<false, true, true>
                            : (run ? k_fire_ensemble<false, false, true>
                                   : k_fire_ensemble<false, false, false>);
  static size_t granted[3][64] = {};
  if (!ens_lds_allow(reinterpret_cast<const void*>(staged), granted[run + plain], lds_bytes))
    return JMD_ERR_LAUNCH;
  hipLaunchKernelGGL(staged, dim3(n_systems), dim3(threads), lds_bytes,
                     (hipStream_t)stream, reinterpret_cast<const EnsSys*>(systems), order,
                     n_systems, (int)n_total, mode, n_steps, position_hi, position, momentum,
                     force, reference_position, idx, width, scratch, a, prm, fire_state,
                     fire_n_pos, error, out_stat, energy, builds, tape, lds_n);
  JMD_LAUNCH_CHECK();
  hipLaunchKernelGGL(memory, dim3(n_systems), dim3(threads), 0,
                     (hipStream_t)stream, reinterpret_cast<const EnsSys*>(systems), order,
                     n_systems, (int)n_total, mode, n_steps, position_hi, position, momentum,
                     force, reference_position, idx, width, scratch, a, prm, fire_state,
                     fire_n_pos, error, out_stat, energy, builds, tape, lds_n);
  JMD_LAUNCH_CHECK();
  return JMD_OK;
}

int jmd_fire_ensemble_max_cells(void) { return kEnsMaxCells; }

int jmd_fire_ensemble_threads(int32_t n_systems, int64_t n_total, int32_t n_max) {
  return ens_threads(n_systems, n_total, n_max);
}

int jmd_fire_ensemble_set_threads(int32_t threads) {
  if (!ens_threads_ok(threads)) return JMD_ERR_INVALID;
  g_ens_threads = threads;
  return JMD_OK;
}

int jmd_fire_ensemble_adjoint_2d(const jmd_system2d* systems, int32_t n_systems,
                                 int64_t n_total, int32_t mode, int32_t n_steps,
                                 const float* position, const float* force, const int32_t* idx,
                                 int32_t width, const jmd_pair_potential* potential,
                                 const float* dsigma, const float* tape_x,
                                 const float* tape_force, const float* tape_q,
                                 const int32_t* tape_idx, const float* tape_scalars,
                                 double* x_adjoint, double* p_adjoint, float* pending,
                                 float* scratch, double* theta, double* box_adjoint,
                                 float scale, void* stream) {
  const int asked = mode >> 8;
  if (mode < 0 || !ens_threads_ok(asked)) return JMD_ERR_INVALID;
  mode &= 0xff;
  if (n_systems < 0 || n_total < 0 || n_total >= 0x7fffffff || width < 1 || n_steps < 0 ||
      mode > BACK_FINISH)
    return JMD_ERR_INVALID;
  if (n_systems == 0) return JMD_OK;
  if (!systems || !x_adjoint || !p_adjoint || !pending || !scratch || !theta)
    return JMD_ERR_INVALID;
  if (mode == BACK_INIT && (!position || !force || !idx)) return JMD_ERR_INVALID;
  if (mode != BACK_INIT && (!tape_x || !tape_force || !tape_q || !tape_idx || !tape_scalars))
    return JMD_ERR_INVALID;
  PairArgs a;
  if (!make_pair_args(potential, &a) || a.kind != JMD_SOFT_SPHERE) return JMD_ERR_INVALID;
  if (dsigma && a.sig_mode != JMD_PARAM_SPECIES) return JMD_ERR_UNSUPPORTED;
  EnsTape tape{const_cast<float*>(tape_x), const_cast<float*>(tape_force),
               const_cast<float*>(tape_q), const_cast<int*>(tape_idx),
               const_cast<float*>(tape_scalars), n_steps};
  // LDS copy of each system's node positions, product vector and species
  // ids (systems of up to 8 particles per thread; larger ones use memory)
  const int threads = ens_launch_threads(asked, n_systems, n_total);
  const int lds_n = threads * kEnsPerThread;
  const size_t lds_bytes = (size_t)lds_n * (4 * sizeof(float) + 1);
  const bool plain = ens_plain(a);
  const auto staged = plain ? k_fire_ensemble_back<true, true> : k_fire_ensemble_back<true, false>;
  const auto memory = plain ? k_fire_ensemble_back<false, true> : k_fire_ensemble_back<false, false>;
  static size_t granted[2][64] = {};
  if (!ens_lds_allow(reinterpret_cast<const void*>(staged), granted[plain], lds_bytes))
    return JMD_ERR_LAUNCH;
  hipLaunchKernelGGL(staged, dim3(n_systems), dim3(threads), lds_bytes,
                     (hipStream_t)stream, reinterpret_cast<const EnsSys*>(systems), n_systems,
                     (int)n_total, mode, n_steps, position, force, idx, width, a, dsigma, tape,
                     x_adjoint, p_adjoint, pending, scratch, theta, box_adjoint, scale, lds_n);
  JMD_LAUNCH_CHECK();
  hipLaunchKernelGGL(memory, dim3(n_systems), dim3(threads), 0,
                     (hipStream_t)stream, reinterpret_cast<const EnsSys*>(systems), n_systems,
                     (int)n_total, mode, n_steps, position, force, idx, width, a, dsigma, tape,
                     x_adjoint, p_adjoint, pending, scratch, theta, box_adjoint, scale, lds_n);
  JMD_LAUNCH_CHECK();
  return JMD_OK;
}

}  // extern "C"
