// Dense-list pair kernels (templates only): row_sum, k_pair_dense and their
// launch helpers.  The host entry points live in jmd_pair.hip; the
// dispatch_dense instantiations are compiled in jmd_pair_dense_*.hip (one
// translation unit per position layout and potential, built in parallel).
#pragma once

#include "jmd_pair_common.hpp"

namespace jmd {

// Rows of a position table through a buffer descriptor whose stride is the
// row: the load takes the row index itself (no address arithmetic), and an
// index of n or more reads zeros.  The intrinsics have no clang builtin, so
// they are bound by name.
typedef int rsrc_t __attribute__((ext_vector_type(4)));
typedef float f2_t __attribute__((ext_vector_type(2)));
typedef float f3_t __attribute__((ext_vector_type(3)));
__device__ f3_t struct_load3(rsrc_t rsrc, int index, int voffset, int soffset,
                             int aux) __asm("llvm.amdgcn.struct.buffer.load.v3f32");
__device__ f2_t struct_load2(rsrc_t rsrc, int index, int voffset, int soffset,
                             int aux) __asm("llvm.amdgcn.struct.buffer.load.v2f32");

__device__ __forceinline__ rsrc_t row_table(const float* p, unsigned rows, int row_bytes) {
  const unsigned long long b = (unsigned long long)p;
  return rsrc_t{(int)(unsigned)b, (int)((unsigned)(b >> 32) & 0xffffu) | (row_bytes << 16),
                (int)rows, 0x00020000};
}

// Sum over one Dense row slice (entries sub, sub+TPA, ...) into f, e.
//
// What bounds it: the gathers, then VALU issue.  A list at r_c + skin = 3.0
// holds 95 entries a row at rho 0.8442; at N = 262,144 the L1 serves 22.5 M
// requests a launch (88 k of 114 k cycles on each CU) and each SIMD issues
// 80 k cycles of VALU work, 52 lane operations an entry with the ends of the
// rows and the step's epilogue.  (Timing copies: without half of the
// arithmetic 1.5 us of 49 less, with neighbours that are consecutive rows 12 us
// less.  16-byte loads of the entries saved a third of the load instructions
// and made the gathers' L1 requests 15% more; two blocks of entries in flight
// changed nothing.)
// * Folds are decided per block of UNR entries and dimension: while every
//   plain difference of the block is shorter than half the side, it is the
//   minimum image, and a maximum and a ballot replace the selects.  `near`
//   (bit c, wavefront-uniform) is clear where no row of the wavefront lies
//   within the interaction range of a face of dimension c and every position
//   lies in the box: pairs in range then need no fold and the others add
//   zero either way.  (Before, wavefronts near any face, 22% of them at
//   N = 262,144 and all of them when the positions were not known to lie in
//   the box, folded every component of every pair.)
// * In a block whose entries are valid in every lane no entry needs a mask;
//   the masked form runs in the block where some row of the wavefront ends.
// * Constant factors of the potential are applied once per row (lj_reduced).
// * INDEXED gathers (tables below 2 GiB) go through row_table.
// Step kernel at N = 262,144: 48.4 -> 45 us; energy and force of 1,029,897
// particles not known to lie in the box: 202 -> 176 us.
template <int DIM, int STRIDE, int KIND, int TPA, bool GENERAL, bool ENERGY, int SMOOTH,
          int BOX, bool INDEXED, int UNR>
__device__ __forceinline__ void row_sum(const float* __restrict__ pos, unsigned n,
                                        const Space& s, const PairArgs& a,
                                        const int* __restrict__ row, int width, int sub,
                                        unsigned i, const float* xi, unsigned near, float* f,
                                        float* e) {
#pragma clang fp contract(off)
  constexpr bool LJ = KIND == JMD_LENNARD_JONES;
  float sig = a.sig, eps = a.eps, alp = a.alp;
  const float sig2 = a.sig * a.sig;
  int si = 0;
  if (GENERAL && a.species) si = a.species[i];
  const rsrc_t table = row_table(pos, n, STRIDE * 4);
  auto gather = [&](unsigned j, float* xj) {
    if (!INDEXED) {
      load_pos<DIM, STRIDE>(pos, j < n ? j : i, xj);
    } else if (DIM == 3) {
      const f3_t v = struct_load3(table, (int)j, 0, 0, 0);
      xj[0] = v.x;
      xj[1] = v.y;
      xj[2] = v.z;
    } else {
      const f2_t v = struct_load2(table, (int)j, 0, 0, 0);
      xj[0] = v.x;
      xj[1] = v.y;
    }
  };
  auto square = [&](const float* d) {
    return DIM == 3 ? fmaf(d[2], d[2], fmaf(d[1], d[1], d[0] * d[0]))
                    : fmaf(d[1], d[1], d[0] * d[0]);
  };
  // One pair term from its difference; masked: `ok` false adds nothing.
  auto term = [&](unsigned j, const float* d, float r2, bool masked, bool ok) {
    if (GENERAL) {
      int sj = a.species ? a.species[j] : 0;
      sig = pick(a.sig_mode, a.sig, a.sig_v, i, j, si, sj, a.ns);
      eps = pick(a.eps_mode, a.eps, a.eps_v, i, j, si, sj, a.ns);
      if (!LJ) alp = pick(a.alp_mode, a.alp, a.alp_v, i, j, si, sj, a.ns);
    }
    float g, u;
    if (LJ) {
      g = lj_reduced<SMOOTH>(r2, GENERAL ? sig * sig : sig2, a, &u);
      if (GENERAL) {
        g *= eps;
        if (ENERGY) u *= eps;
      }
    } else {
      u = pair_eval<KIND>(r2, sig, eps, alp, a, &g);
    }
    if (masked) g = ok ? g : 0.0f;
#pragma unroll
    for (int c = 0; c < DIM; ++c) f[c] = fmaf(g, d[c], f[c]);
    if (ENERGY) *e += masked && !ok ? 0.0f : u;
  };
  // A block of UNR entries, every one valid in every lane of the wavefront.
  auto full_block = [&](const unsigned* jj, float (*xj)[3]) {
    float d[UNR][3];
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
#pragma unroll
      for (int u = 0; u < UNR; ++u) d[u][c] = xj[u][c] - xi[c];
      if ((near >> c) & 1u) {
        float m = 0.0f;  // (a NaN folds to itself, so the maximum may drop it)
#pragma unroll
        for (int u = 0; u < UNR; ++u) m = fmaxf(m, fabsf(d[u][c]));
        if (__builtin_amdgcn_ballot_w64(m >= s.half[c]) != 0ull) {
          const float xim = xi[c] - s.L[c];
#pragma unroll
          for (int u = 0; u < UNR; ++u)
            d[u][c] = min_image_any(xj[u][c], xi[c], xim, s.L[c], s.half[c], s.inbox);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      if (BOX == 1 || (BOX < 0 && s.general)) box_apply<DIM>(s, d[u]);
      term(jj[u], d[u], square(d[u]), false, true);
    }
  };
  // One entry that is padding in some lane: those add nothing.
  auto masked_entry = [&](unsigned jraw, const float* xj) {
    const bool ok = jraw < n;
    float d[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      d[c] = (near >> c) & 1u
                 ? min_image_any(xj[c], xi[c], xi[c] - s.L[c], s.L[c], s.half[c], s.inbox)
                 : xj[c] - xi[c];
    if (BOX == 1 || (BOX < 0 && s.general)) box_apply<DIM>(s, d);
    term(ok ? jraw : i, d, square(d), true, ok);
  };
  // This lane's entries are sub, sub + TPA, ... < width, in blocks of UNR
  // (the last one may be short).  The next block's entries are loaded before
  // this block's terms are computed (software pipeline: one dependent round
  // trip per block, the position gather).  The row ends at the first block
  // that is padding in every lane.
  const unsigned nfull = (unsigned)width / (UNR * TPA);
  const unsigned nblk = ((unsigned)width + UNR * TPA - 1) / (UNR * TPA);
  const int* p = row + sub;
  // (a short block reads its row's last entry where it has none; what it
  // read is replaced by n when the block is used)
  auto entries = [&](unsigned b, unsigned* v) {
    if (b < nfull) {
      const int* q = p + (long long)b * (UNR * TPA);
#pragma unroll
      for (int u = 0; u < UNR; ++u) v[u] = (unsigned)q[u * TPA];
    } else {
#pragma unroll
      for (int u = 0; u < UNR; ++u)
        v[u] = (unsigned)row[min((int)(b * (UNR * TPA)) + u * TPA + sub, width - 1)];
    }
  };
  if (nfull == 0) {
    // Rows of less than a block: no loads but those of the entries there are.
    // (Taken as a short block, soft spheres in 2-D, rows of 5 on 2 lanes, loaded
    // twice what they needed: a force of 1,000,000 rows 17.5 us, now 12.9; in
    // 3-D, rows of 11 on 8 lanes, 512,000 of them 24.4 and 21.5.)
    unsigned jj[UNR];
    float xj[UNR][3];
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      jj[u] = n;
      if (u * TPA < width) jj[u] = (unsigned)row[min(u * TPA + sub, width - 1)];
    }
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      if (u * TPA + sub >= width) jj[u] = n;
      xj[u][0] = xj[u][1] = xj[u][2] = 0.0f;
      if (u * TPA < width) gather(jj[u], xj[u]);
    }
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      if (__builtin_amdgcn_ballot_w64(jj[u] < n) != 0ull) masked_entry(jj[u], xj[u]);
    }
    return;
  }
  unsigned nxt[UNR];
  entries(0, nxt);
  for (unsigned b = 0; b < nblk; ++b) {
    unsigned jj[UNR], jmin = n, jmax = 0u;
#pragma unroll
    for (int u = 0; u < UNR; ++u) jj[u] = nxt[u];
    if (b >= nfull) {
#pragma unroll
      for (int u = 0; u < UNR; ++u)
        if ((int)(b * (UNR * TPA)) + u * TPA + sub >= width) jj[u] = n;
    }
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      jmin = min(jmin, jj[u]);
      jmax = max(jmax, jj[u]);
    }
    if (__builtin_amdgcn_ballot_w64(jmin < n) == 0ull) return;  // the rows have ended
    float xj[UNR][3];
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
      xj[u][0] = xj[u][1] = xj[u][2] = 0.0f;
      gather(jj[u], xj[u]);
    }
    // (always issued: a wait that had to allow for both cases would also wait
    // for these loads)
    entries(min(b + 1, nblk - 1), nxt);
    if (__builtin_amdgcn_ballot_w64(jmax >= n) == 0ull) {
      full_block(jj, xj);
    } else {
#pragma unroll
      for (int u = 0; u < UNR; ++u) {
        if (__builtin_amdgcn_ballot_w64(jj[u] < n) != 0ull) masked_entry(jj[u], xj[u]);
      }
    }
  }
}

// STEP (with KICK): after the closing half kick, the start of the next
// velocity-Verlet step for each row's particle, from the force and momentum
// in registers: the skin criterion of the positions just used against the
// list's reference positions raises kd.gate_next (the next step's update
// decision), and with kd.active the opening half kick and the drift write
// the next positions to kd.x_out (float64 master positions in place).
template <int DIM, int STRIDE, int KIND, int TPA, bool GENERAL, bool ENERGY, bool KICK,
          bool STEP = false>
__global__ __launch_bounds__(256) void k_pair_dense(
    const float* __restrict__ pos, int n, Space s, PairArgs a, const int* __restrict__ idx,
    int width, float* __restrict__ force, float* __restrict__ e_atom,
    double* __restrict__ e_part, float* __restrict__ mom, float half_dt,
    const float* __restrict__ dt_dev, KickDrift kd) {
  float kdt = kd.dt;
  if (KICK && dt_dev) {
    if (STEP) kdt = dt_dev[0];
    half_dt = dt_dev[0] / 2.0f;
  }
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const unsigned gt = (unsigned)tile * 256u + threadIdx.x;
  const int i = (int)(gt / TPA);
  const int sub = (int)(gt % TPA);
  const bool active = i < n;
  float f[3] = {0.0f, 0.0f, 0.0f};
  float e = 0.0f;
  float xi[3] = {0, 0, 0};
  // STEP with TPA >= DIM: lane `sub` of a row's group takes component `sub`
  // of the next step's start; its inputs are loaded here, ahead of the row
  // loop, so their latency hides behind it.
  constexpr bool SPREAD = STEP && TPA >= DIM;
  const bool mine = SPREAD && active && sub < DIM;
  double st_xh = 0.0;
  float st_ref = 0.0f, st_p = 0.0f, st_m = 0.0f;
  if (mine) {
    st_p = mom[(long long)i * DIM + sub];
    if (kd.active) {
      st_xh = kd.xhi_in[(long long)i * DIM + sub];
      if (kd.mass) st_m = kd.mass[i];
    }
    if (kd.gate_next) st_ref = kd.ref[(long long)i * DIM + sub];
  }
  // (the closing kick without STEP: the row's first lane, loaded ahead too)
  float pm[3] = {0.0f, 0.0f, 0.0f};
  if (KICK && !SPREAD && active && sub == 0) {
#pragma unroll
    for (int c = 0; c < DIM; ++c) pm[c] = mom[(long long)i * DIM + c];
  }
  if (active) {
    load_pos<DIM, STRIDE>(pos, i, xi);
    const int* row = idx + (long long)i * width;
    unsigned near = 0u;
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
      // (fractional coordinates: a reach of r_c is r_c |row c of T^-1|)
      const float w = s.general ? a.rc * s.fw[c] : a.rc;
      const bool edge = !(s.inbox && xi[c] >= w && xi[c] <= s.L[c] - w);
      if (s.periodic && __builtin_amdgcn_ballot_w64(edge) != 0ull) near |= 1u << c;
    }
    // box matrix, switch and table size are uniform: taken once here
#define JMD_ROW(SM, BX, F32, U)                                                     \
  row_sum<DIM, STRIDE, KIND, TPA, GENERAL, ENERGY, SM, BX, F32, U>(pos, n, s, a, row, \
                                                                   width, sub, i, xi, near, \
                                                                   f, &e)
#define JMD_ROW_SM(BX, F32, U)                                                   \
  do {                                                                           \
    if (KIND == JMD_LENNARD_JONES && a.smooth) JMD_ROW(1, BX, F32, U);           \
    else JMD_ROW(0, BX, F32, U);                                                 \
  } while (0)
    // Tables beyond 2 GiB (134 million 16-byte rows) are gathered by address.
    // Four entries in flight as below, two where the registers of four
    // addresses would cost every launch of the instance a wavefront per SIMD.
    // 134,479,872 rows of 26 entries (scalar and species Lennard-Jones, soft
    // sphere): 8.9, 16.4 and 9.5 ms; 10.6, 18.3 and 11.6 with one in flight and
    // the switch tested per pair.
    constexpr int kWideUnr = !GENERAL && (KIND == JMD_LENNARD_JONES || DIM == 3) ? 4 : 2;
    if ((long long)n * (STRIDE * 4) > 0x7fffffffLL) {
      JMD_ROW_SM(-1, false, kWideUnr);
    } else if (s.general) {
      JMD_ROW_SM(1, true, 4);
    } else {
      JMD_ROW_SM(0, true, 4);
    }
#undef JMD_ROW_SM
#undef JMD_ROW
  }
  // the Lennard-Jones sums lack -24 epsilon (force) and 4 epsilon (energy)
  // (lj_reduced), epsilon included per pair where it is not one number
  constexpr bool LJ = KIND == JMD_LENNARD_JONES;
  const double eps1 = GENERAL ? 1.0 : (double)a.eps;
  double fd[3];
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    fd[c] = group_sum<TPA>((double)f[c]);
    if (LJ) fd[c] *= -24.0 * eps1;
  }
  double ed = 0.0;
  if (ENERGY) {
    ed = group_sum<TPA>((double)e);
    if (LJ) ed *= 4.0 * eps1;
  }
  bool moved = false;
  if (SPREAD) {
    // the opening half kick, drift and skin test round every product and
    // sum as kick_drift_atom and ref_metric_sq do (no contraction)
#pragma clang fp contract(off)
    // lane `sub` < DIM: component sub of the row's particle
    const int c = sub;
    float fc = (float)fd[0], xc = xi[0];
#pragma unroll
    for (int q = 1; q < DIM; ++q) {
      fc = c == q ? (float)fd[q] : fc;
      xc = c == q ? xi[q] : xc;
    }
    const int base = lane_id() - sub;  // first lane of the row's group
    float pk = 0.0f;
    if (mine) {
      if (force) force[(long long)i * DIM + c] = fc;
      pk = fmaf(half_dt, fc, st_p);  // the closing half kick, fused as in the other forms
    }
    if (kd.gate_next) {
      // the skin criterion of ref_metric_sq: component terms, T for a
      // general box, squares summed in component order
      float v = 0.0f;
      if (mine) {
        v = xc - st_ref;
        if (kd.s.periodic) v = ref_wrap1(v, kd.s.L[c], kd.s.half[c]);
      }
      float vv[3];
#pragma unroll
      for (int q = 0; q < DIM; ++q) vv[q] = __shfl(v, base + q, kWave);
      if (kd.s.general) {
        box_apply_ref<DIM>(kd.s, vv);
      }
      if (sub == 0 && active) {
        float acc = 0.0f;
#pragma unroll
        for (int q = 0; q < DIM; ++q) {
          const float sq = vv[q] * vv[q];
          acc = q == 0 ? sq : acc + sq;
        }
        moved = acc > kd.thr_sq;
      }
    }
    float pn = pk;
    if (kd.active) {
      // the opening half kick and the float64 drift of kick_drift_regs
      pn = pk + half_dt * fc;
      const double w = (double)kdt * (double)pn;
      double dx = kd.mass_pow2 ? w * kd.inv_mass
                               : w / (kd.mass ? (double)st_m : (double)kd.mass_scalar);
      if (kd.s.general) {
        double dv[3];
#pragma unroll
        for (int q = 0; q < DIM; ++q) dv[q] = __shfl(dx, base + q, kWave);
        double acc = 0.0;
#pragma unroll
        for (int b = 0; b < DIM; ++b) {
          float t = kd.Ti[0][b];
#pragma unroll
          for (int q = 1; q < DIM; ++q) t = c == q ? kd.Ti[q][b] : t;
          acc += (double)t * dv[b];
        }
        dx = acc;
      }
      if (mine) {
        double x = st_xh + dx;
        if (kd.s.periodic) {
          float Lc = kd.s.L[0];
#pragma unroll
          for (int q = 1; q < DIM; ++q) Lc = c == q ? kd.s.L[q] : Lc;
          x = ref_mod64(x, (double)Lc);
        }
        kd.xhi_out[(long long)i * DIM + c] = x;
        kd.x_out[(long long)i * STRIDE + c] = (float)x;
      }
    }
    if (mine) mom[(long long)i * DIM + c] = pn;
  }
  if (active && sub == 0 && !SPREAD) {
    float fcv[3] = {0.0f, 0.0f, 0.0f}, pk[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
      float fc = (float)fd[c];
      if (force) force[(long long)i * DIM + c] = fc;
      if (KICK && !STEP) mom[(long long)i * DIM + c] = fmaf(half_dt, fc, pm[c]);
      if (STEP) {
        fcv[c] = fc;
        pk[c] = fmaf(half_dt, fc, pm[c]);
      }
    }
    if (STEP) {
      if (kd.gate_next) {
        float r[3];
        load_pos<DIM>(kd.ref, i, r);
        moved = ref_metric_sq<DIM>(xi, r, kd.s) > kd.thr_sq;
      }
      if (kd.active) {
        float xn[3];
        kick_drift_regs<DIM>(kd, i, kdt, half_dt, pk, fcv, xn);
        store_pos<DIM, STRIDE>(kd.x_out, i, xn);
      }
#pragma unroll
      for (int c = 0; c < DIM; ++c) mom[(long long)i * DIM + c] = pk[c];
    }
  }
  if (ENERGY && active && sub == 0 && e_atom) e_atom[i] = (float)(0.5 * ed);
  if (STEP && kd.gate_next) raise_gate(kd.gate_next, moved);
  if (ENERGY) {
    // block partial of 0.5 * sum_i e_i in float64
    __shared__ double s_e[256 / kWave];
    double v = (active && sub == 0) ? 0.5 * ed : 0.0;
    v = wave_reduce_sum(v);
    if (lane_id() == 0) s_e[threadIdx.x / kWave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int w = 0; w < (int)(blockDim.x / kWave); ++w) t += s_e[w];
      e_part[tile] = t;
    }
  }
}

struct DenseLaunch {
  dim3 grid;
  hipStream_t st;
  const float* pos;
  int n;
  Space s;
  PairArgs a;
  const int* idx;
  int width;
  float* force;
  float* e_atom;
  double* e_part;
  float* mom;
  float half_dt;
  const float* dt_dev;
  KickDrift kd;  // the next step's start (STEP launches only)
};

template <int DIM, int STRIDE, int KIND, int TPA, bool GENERAL>
void launch_dense(const DenseLaunch& L, bool energy, bool kick, bool step) {
#define JMD_PD(E, K, S)                                                                      \
  hipLaunchKernelGGL((k_pair_dense<DIM, STRIDE, KIND, TPA, GENERAL, E, K, S>), L.grid,       \
                     dim3(256), 0, L.st, L.pos, L.n, L.s, L.a, L.idx, L.width, L.force,      \
                     L.e_atom, L.e_part, L.mom, L.half_dt, L.dt_dev, L.kd)
  if (energy) JMD_PD(true, false, false);
  else if (step) JMD_PD(false, true, true);
  else if (kick) JMD_PD(false, true, false);
  else JMD_PD(false, false, false);
#undef JMD_PD
}

template <int DIM, int STRIDE, int KIND>
void dispatch_dense(int tpa, bool general, const DenseLaunch& L, bool energy, bool kick,
                    bool step) {
#define JMD_TPA(T)                                                               \
  (general ? launch_dense<DIM, STRIDE, KIND, T, true>(L, energy, kick, step)     \
           : launch_dense<DIM, STRIDE, KIND, T, false>(L, energy, kick, step))
  switch (tpa) {
    case 2: JMD_TPA(2); break;
    case 8: JMD_TPA(8); break;
    case 16: JMD_TPA(16); break;
    case 32: JMD_TPA(32); break;
    default: JMD_TPA(4); break;
  }
#undef JMD_TPA
}

// Explicit instantiations live in jmd_pair_dense_*.hip.
#define JMD_DENSE_INSTANCES(X)                      \
  X(3, 4, JMD_LENNARD_JONES) X(3, 4, JMD_SOFT_SPHERE) \
  X(3, 3, JMD_LENNARD_JONES) X(3, 3, JMD_SOFT_SPHERE) \
  X(2, 2, JMD_LENNARD_JONES) X(2, 2, JMD_SOFT_SPHERE)
#define JMD_DENSE_EXTERN(D, S, K)                                                     \
  extern template void dispatch_dense<D, S, K>(int, bool, const DenseLaunch&, bool, bool, \
                                               bool);
#define JMD_DENSE_INSTANTIATE(D, S, K)                                         \
  template void dispatch_dense<D, S, K>(int, bool, const DenseLaunch&, bool, bool, bool);

}  // namespace jmd
