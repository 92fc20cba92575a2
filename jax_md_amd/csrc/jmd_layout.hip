// Particle reordering for the native block loop on gfx950.
//
// The pair kernel's cost is set by how many distinct cache lines a
// wavefront's neighbour gather touches.  Inside a block of steps the loop
// keeps particles in cell order (the order of the cell list: cells in hash
// order, ids ascending inside a cell), so that the particles of a wavefront
// share a cell and their neighbours lie in a few contiguous runs.  The
// reference's user order is restored at the end of the block, and the
// neighbour list is translated back to user ids.
#include "jmd_common.hpp"

namespace jmd {

// out[r] = in[perm[r]] for rows of `row_bytes` bytes (multiple of 4).
__global__ __launch_bounds__(256) void k_gather_rows(const uint32_t* __restrict__ in,
                                                     uint32_t* __restrict__ out,
                                                     const int* __restrict__ perm, int n,
                                                     int row_words, int in_stride_words,
                                                     int out_stride_words) {
  long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  long long total = (long long)n * row_words;
  long long step = (long long)gridDim.x * blockDim.x;
  for (; t < total; t += step) {
    int r = (int)(t / row_words);
    int w = (int)(t - (long long)r * row_words);
    out[(long long)r * out_stride_words + w] = in[(long long)perm[r] * in_stride_words + w];
  }
}

// out[perm[r]] = in[r] (the inverse of k_gather_rows).
__global__ __launch_bounds__(256) void k_scatter_rows(const uint32_t* __restrict__ in,
                                                      uint32_t* __restrict__ out,
                                                      const int* __restrict__ perm, int n,
                                                      int row_words, int in_stride_words,
                                                      int out_stride_words) {
  long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  long long total = (long long)n * row_words;
  long long step = (long long)gridDim.x * blockDim.x;
  for (; t < total; t += step) {
    int r = (int)(t / row_words);
    int w = (int)(t - (long long)r * row_words);
    out[(long long)perm[r] * out_stride_words + w] = in[(long long)r * in_stride_words + w];
  }
}

// Dense list in permuted ids -> user ids: out[perm[r], k] = perm[in[r, k]]
// (padding n stays n).
__global__ __launch_bounds__(256) void k_remap_dense(const int* __restrict__ in,
                                                     int* __restrict__ out,
                                                     const int* __restrict__ perm, int n,
                                                     int width) {
  // one wavefront per row: the row's destination is read once, lanes walk the
  // entries (no per-entry division to find the row)
  const int lane = lane_id();
  const long long nw = (long long)gridDim.x * (blockDim.x / kWave);
  for (long long r = (long long)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; r < n;
       r += nw) {
    const int* src = in + r * width;
    int* dst = out + (long long)perm[r] * width;
    for (int k = lane; k < width; k += kWave) {
      const int j = src[k];
      dst[k] = j < n ? perm[j] : n;
    }
  }
}

// The same over the flat [n * width] array in 16-byte chunks: each lane
// loads four consecutive entries with one vector load, finds their row once
// (32-bit division; n * width < 2^31), gathers the four ids' new numbers
// independently and writes the entries into the destination row(s).  The
// rows' entries stay contiguous, so consecutive lanes write consecutive
// addresses except where a chunk crosses a row end.  in must be 16-byte
// aligned; total % 4 trailing entries are done by the first lanes.
__global__ __launch_bounds__(256) void k_remap_dense_flat(const int* __restrict__ in,
                                                          int* __restrict__ out,
                                                          const int* __restrict__ perm, int n,
                                                          int width) {
  const unsigned total = (unsigned)n * (unsigned)width;
  const unsigned nq = total / 4u;
  const unsigned step = gridDim.x * blockDim.x;
  for (unsigned q = blockIdx.x * blockDim.x + threadIdx.x; q < nq; q += step) {
    const int4 v = reinterpret_cast<const int4*>(in)[q];
    const unsigned e = q * 4u;
    unsigned row = e / (unsigned)width;
    unsigned col = e - row * (unsigned)width;
    const int jv[4] = {v.x, v.y, v.z, v.w};
    int pj[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) pj[u] = jv[u] < n ? perm[jv[u]] : n;
    long long dst = (long long)perm[row] * width;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      out[dst + col] = pj[u];
      if (++col == (unsigned)width && u < 3) {
        col = 0;
        ++row;
        dst = (long long)perm[row] * width;
      }
    }
  }
  if (blockIdx.x == 0 && threadIdx.x < total % 4u) {
    const unsigned e = nq * 4u + threadIdx.x;
    const unsigned row = e / (unsigned)width, col = e - row * (unsigned)width;
    const int j = in[e];
    out[(long long)perm[row] * width + col] = j < n ? perm[j] : n;
  }
}

// Sparse list [2, width] through perm (entries keep their slots).
// OrderedSparse keeps receiver < sender (partition.py:998): a pair whose
// order the renumbering reversed is stored swapped.
__global__ __launch_bounds__(256) void k_remap_ids(const int* __restrict__ in,
                                                   int* __restrict__ out,
                                                   const int* __restrict__ perm, int n,
                                                   long long width, int ordered) {
  long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  long long step = (long long)gridDim.x * blockDim.x;
  for (; t < width; t += step) {
    const int a = in[t], b = in[width + t];
    int ra = a < n ? perm[a] : n;
    int sb = b < n ? perm[b] : n;
    if (ordered && ra < n && sb < n && ra > sb) {
      const int x = ra;
      ra = sb;
      sb = x;
    }
    out[t] = ra;
    out[width + t] = sb;
  }
}

// Dense rows -> a Sparse-format list: each row i's entries j in row order as
// (receiver j, sender i), rows in order (OrderedSparse: entries below the
// row's id only), then padding.  Bound by memory: the rows are read twice
// (once to count, once to write; 36 MB at N = 64,000 stay in the last-level
// cache between) and the list is written once.  One wavefront per row and 8
// per workgroup; kRowsPerBlock rows share one partial count, so that the scan
// between the passes is a single workgroup over n / 64 values.  With torch's
// masked indexing and cumsum the conversion took 0.75 ms a block at
// N = 64,000 (it sorted out the kept entries of the flattened rows in several
// library passes and waited on the host for their number).
constexpr int kRowsPerBlock = 64;

__device__ __forceinline__ unsigned long long kept_entries(const int* __restrict__ row, int n,
                                                           int width, int k, int i, int ordered,
                                                           int* j) {
  *j = k < width ? row[k] : n;
  return __builtin_amdgcn_ballot_w64((unsigned)*j < (unsigned)n && (!ordered || *j < i));
}

constexpr int kSparseBlock = 512;

__global__ __launch_bounds__(kSparseBlock) void k_sparse_count(const int* __restrict__ rows,
                                                               int n, int width, int ordered,
                                                               int* __restrict__ row_count,
                                                               int* __restrict__ block_total) {
  __shared__ int s_sum[kSparseBlock / kWave];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  int sum = 0;  // wavefront-uniform
  for (int r = wave; r < kRowsPerBlock; r += kSparseBlock / kWave) {
    const int i = blockIdx.x * kRowsPerBlock + r;
    if (i >= n) break;
    const int* row = rows + (long long)i * width;
    int count = 0;
    for (int k = lane; k - lane < width; k += kWave) {
      int j;
      count += __popcll(kept_entries(row, n, width, k, i, ordered, &j));
    }
    if (lane == 0) row_count[i] = count;
    sum += count;
  }
  if (lane == 0) s_sum[wave] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int w = 0; w < kSparseBlock / kWave; ++w) t += s_sum[w];
    block_total[blockIdx.x] = t;
  }
}

// One workgroup: block totals -> exclusive 64-bit offsets, the list's length,
// and the overflow bit.
__global__ __launch_bounds__(1024) void k_sparse_offsets(const int* __restrict__ block_total,
                                                         int nblocks, long long capacity,
                                                         long long* __restrict__ offset,
                                                         uint8_t* __restrict__ error) {
  __shared__ long long s_w[1024 / kWave];
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  long long carry = 0;
  for (int b0 = 0; b0 < nblocks; b0 += 1024) {
    const long long v = b0 + t < nblocks ? block_total[b0 + t] : 0;
    long long incl = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const long long y = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += y;
    }
    if (lane == kWave - 1) s_w[wave] = incl;
    __syncthreads();
    long long before = 0, all = 0;
    for (int w = 0; w < 1024 / kWave; ++w) {
      before += w < wave ? s_w[w] : 0;
      all += s_w[w];
    }
    if (b0 + t < nblocks) offset[b0 + t] = carry + before + incl - v;
    carry += all;
    __syncthreads();  // s_w is rewritten by the next chunk
  }
  if (t == 0) {
    offset[nblocks] = carry;
    if (carry > capacity) error[0] = (uint8_t)(error[0] | JMD_NEIGHBOR_LIST_OVERFLOW);
  }
}

__global__ __launch_bounds__(kSparseBlock) void k_sparse_write(
    const int* __restrict__ rows, int n, int width, int ordered,
    const int* __restrict__ row_count, const long long* __restrict__ offset, int nblocks,
    long long capacity, int* __restrict__ idx) {
  __shared__ int s_first[kRowsPerBlock];  // a row's first slot inside the block
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  // padding beyond the list's length, spread over the grid
  for (long long k = offset[nblocks] + (long long)blockIdx.x * kSparseBlock + threadIdx.x;
       k < capacity; k += (long long)gridDim.x * kSparseBlock) {
    idx[k] = n;
    idx[capacity + k] = n;
  }
  if (wave == 0) {
    const int i = blockIdx.x * kRowsPerBlock + lane;
    const int v = i < n ? row_count[i] : 0;
    int incl = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int y = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += y;
    }
    s_first[lane] = incl - v;
  }
  __syncthreads();
  const long long base = offset[blockIdx.x];
  for (int r = wave; r < kRowsPerBlock; r += kSparseBlock / kWave) {
    const int i = blockIdx.x * kRowsPerBlock + r;
    if (i >= n) break;
    const int* row = rows + (long long)i * width;
    long long at = base + s_first[r];
    for (int k = lane; k - lane < width; k += kWave) {
      int j;
      const unsigned long long bal = kept_entries(row, n, width, k, i, ordered, &j);
      const long long slot = at + wave_prefix_count(bal);
      if (__builtin_amdgcn_inverse_ballot_w64(bal) && slot < capacity) {
        idx[slot] = j;             // receiver
        idx[capacity + slot] = i;  // sender
      }
      at += __popcll(bal);
    }
  }
}

static int grid_for(long long total) {
  long long b = (total + 255) / 256;
  if (b < 1) b = 1;
  if (b > 8192) b = 8192;
  return (int)b;
}

}  // namespace jmd

using namespace jmd;

extern "C" {

int jmd_permute_rows(const void* in, void* out, const int32_t* perm, int64_t n,
                     int32_t row_bytes, int32_t in_stride_bytes, int32_t out_stride_bytes,
                     int32_t inverse, void* stream) {
  if (n < 0 || n > 0x7fffffff || row_bytes <= 0 || (row_bytes & 3) || (in_stride_bytes & 3) ||
      (out_stride_bytes & 3) || in_stride_bytes < row_bytes || out_stride_bytes < row_bytes ||
      (n > 0 && (!in || !out || !perm)) || in == out)
    return JMD_ERR_INVALID;
  if (n == 0) return JMD_OK;
  hipStream_t st = (hipStream_t)stream;
  int rw = row_bytes / 4;
  long long total = n * (long long)rw;
  if (inverse)
    hipLaunchKernelGGL(k_scatter_rows, dim3(grid_for(total)), dim3(256), 0, st,
                       (const uint32_t*)in, (uint32_t*)out, perm, (int)n, rw,
                       in_stride_bytes / 4, out_stride_bytes / 4);
  else
    hipLaunchKernelGGL(k_gather_rows, dim3(grid_for(total)), dim3(256), 0, st,
                       (const uint32_t*)in, (uint32_t*)out, perm, (int)n, rw,
                       in_stride_bytes / 4, out_stride_bytes / 4);
  JMD_LAUNCH_CHECK();
  return JMD_OK;
}

int jmd_remap_neighbor_ids(const int32_t* idx_in, int32_t* idx_out, const int32_t* perm,
                           int64_t n, int32_t format, int64_t width, void* stream) {
  if (n < 0 || n > 0x7fffffff || width < 0 || (n > 0 && !perm) || idx_in == idx_out ||
      (width > 0 && (!idx_in || !idx_out)))
    return JMD_ERR_INVALID;
  if (format != JMD_DENSE && format != JMD_SPARSE && format != JMD_ORDERED_SPARSE)
    return JMD_ERR_INVALID;
  if (width == 0 || n == 0) return JMD_OK;
  hipStream_t st = (hipStream_t)stream;
  if (format == JMD_DENSE) {
    if (width > 0x7fffffff) return JMD_ERR_INVALID;
    if (n * width < 0x7fffffffLL && ((uintptr_t)idx_in & 15) == 0) {
      long long qb = (n * width / 4 + 255) / 256;
      if (qb < 1) qb = 1;
      if (qb > 16384) qb = 16384;
      hipLaunchKernelGGL(k_remap_dense_flat, dim3((unsigned)qb), dim3(256), 0, st, idx_in,
                         idx_out, perm, (int)n, (int)width);
    } else {
      long long rb = (n + 3) / 4;  // four rows (wavefronts) per workgroup
      hipLaunchKernelGGL(k_remap_dense,
                         dim3((unsigned)(rb < 65536 ? (rb < 1 ? 1 : rb) : 65536)), dim3(256), 0,
                         st, idx_in, idx_out, perm, (int)n, (int)width);
    }
  } else {
    hipLaunchKernelGGL(k_remap_ids, dim3(grid_for(width)), dim3(256), 0, st, idx_in, idx_out,
                       perm, (int)n, width, format == JMD_ORDERED_SPARSE ? 1 : 0);
  }
  JMD_LAUNCH_CHECK();
  return JMD_OK;
}

size_t jmd_dense_rows_to_sparse_workspace_bytes(int64_t n) {
  const long long nb = n > 0 ? (n + kRowsPerBlock - 1) / kRowsPerBlock : 0;
  return (size_t)(nb + 1) * (sizeof(long long) + sizeof(int)) +
         (size_t)(n > 0 ? n : 0) * sizeof(int) + 64;
}

int jmd_dense_rows_to_sparse(const int32_t* rows, int64_t n, int64_t width, int32_t format,
                             int32_t* idx, int64_t capacity, uint8_t* error, void* workspace,
                             void* stream) {
  if (n < 0 || n > 0x7fffffff || width < 0 || width > 0x7fffffff || capacity < 0 ||
      (format != JMD_SPARSE && format != JMD_ORDERED_SPARSE) || !error || !workspace ||
      (n > 0 && width > 0 && !rows) || (capacity > 0 && !idx) || ((uintptr_t)workspace & 7) != 0)
    return JMD_ERR_INVALID;
  hipStream_t st = (hipStream_t)stream;
  const int nb = ceil_div(n, kRowsPerBlock);
  long long* offset = (long long*)workspace;
  int* total = (int*)(offset + nb + 1);
  int* row_count = total + nb + 1;
  const int nn = (int)n, w = (int)width, ordered = format == JMD_ORDERED_SPARSE ? 1 : 0;
  if (nb > 0) {
    hipLaunchKernelGGL(k_sparse_count, dim3(nb), dim3(kSparseBlock), 0, st, rows, nn, w, ordered,
                       row_count, total);
    JMD_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_sparse_offsets, dim3(1), dim3(1024), 0, st, total, nb, (long long)capacity,
                     offset, error);
  JMD_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_sparse_write, dim3(nb > 0 ? nb : 1), dim3(kSparseBlock), 0, st, rows, nn, w,
                     ordered, row_count, offset, nb, (long long)capacity, idx);
  JMD_LAUNCH_CHECK();
  return JMD_OK;
}

}  // extern "C"
