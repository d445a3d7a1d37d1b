// build.hip -- index-build kernels: probe counts (A3), k-means update (A14),
// PQ encoding (A16), PQ codebook training (A15), k-means++ seeding.
#include "common.hpp"
#include "kernels.hpp"

#include <cmath>

namespace fgpu {
namespace {

// ---- A3: probe counts + exclusive scan (gpu_global.cu:31-77, 704-723) -----
__global__ void probe_counts_kernel(const uint32_t* __restrict__ probes, int nq, int nprobe, int nlist,
                                    const int32_t* __restrict__ offsets, int32_t* __restrict__ counts) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nq) return;
  int c = 0;
  for (int p = 0; p < nprobe; ++p) {
    const uint32_t l = probes[(size_t)q * nprobe + p];
    if (l < (uint32_t)nlist) c += offsets[l + 1] - offsets[l];  // pruned ids are >= nlist
  }
  counts[q] = c;
}

// Single-workgroup exclusive scan; out[n] = total.
__global__ __launch_bounds__(1024) void exclusive_scan_kernel(const int32_t* __restrict__ in, int n,
                                                               int32_t* __restrict__ out) {
  __shared__ int32_t part[16];
  __shared__ int32_t carry;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < n; base += 1024) {
    const int i = base + threadIdx.x;
    const int32_t v = i < n ? in[i] : 0;
    int32_t inc = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      int32_t t = __shfl_up(inc, o, kWave);
      if (lane >= o) inc += t;
    }
    if (lane == 63) part[wave] = inc;
    __syncthreads();
    int32_t wbase = 0;
    for (int w = 0; w < wave; ++w) wbase += part[w];
    const int32_t c0 = carry;
    if (i < n) out[i] = c0 + wbase + inc - v;
    __syncthreads();
    if (threadIdx.x == 1023) carry = c0 + wbase + inc;
    __syncthreads();
  }
  if (threadIdx.x == 0) out[n] = carry;
}

// ---- helpers ------------------------------------------------------------------
__global__ void maxabs_partial_kernel(const float* __restrict__ x, int64_t count, float* __restrict__ part) {
  float m = 0.0f;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
    m = fmaxf(m, fabsf(x[i]));
  __shared__ float s[4];
  m = wave_max_f(m);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
}

__global__ void fill_u64_kernel(unsigned long long* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0ull;
}
__global__ void fill_i32_kernel(int32_t* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

__global__ void add_i32_kernel(int32_t* __restrict__ p, const int32_t* __restrict__ q, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] += q[i];
}

__global__ void gather_rows_kernel(const float* __restrict__ x, int dim, const int32_t* __restrict__ rows,
                                   int nrows, float* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)nrows * dim) return;
  const int r = (int)(t / dim), d = (int)(t % dim);
  out[t] = x[(int64_t)rows[r] * dim + d];
}

// ---- A14: deterministic Lloyd update ------------------------------------------
// Sums of round(x * 2^shift) in int64 (two's complement through unsigned
// atomics): integer addition is associative, so the result does not depend on
// the order the atomics land, unlike the reference's float atomicAdd
// (kmeans_gpu.cuh:94-97).
// Two forms.  kmeans_accumulate_kernel: one 64-bit atomic a coordinate.  Where
// grouping_pays, the rows are first grouped by centre (a histogram, its
// scan, a scatter of the row numbers; the order within a centre is free), then
// each wave sums 128 consecutive grouped rows in registers and adds a centre's
// sums once: 1M rows of 128 dims and 4096 centres 0.90 -> 0.14 ms (128 M
// atomics before, 1.6 M now; reading the rows once takes 0.1 ms).
constexpr int kOrdThreads = 1024, kOrdPer = 8;  // rows a workgroup of the grouping kernels: 8192
constexpr int kOrdSeg = 128;                    // grouped rows a wave sums

// The workgroup's rows per centre in LDS; the rank of this thread's row i
// (strided by the workgroup size) among them.
__device__ __forceinline__ void order_local(const int32_t* assign, int64_t row0, int64_t n, int k, int32_t* bins,
                                            int (&c)[kOrdPer], int (&rank)[kOrdPer]) {
  for (int b = threadIdx.x; b < k; b += kOrdThreads) bins[b] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kOrdPer; ++i) {
    const int64_t r = row0 + (int64_t)i * kOrdThreads + threadIdx.x;
    c[i] = r < n ? assign[r] : -1;
    rank[i] = (uint32_t)c[i] < (uint32_t)k ? atomicAdd(&bins[c[i]], 1) : -1;
  }
  __syncthreads();
}

__global__ __launch_bounds__(kOrdThreads) void order_count_kernel(const int32_t* __restrict__ assign, int64_t n, int k,
                                                                  int32_t* __restrict__ counts) {
  extern __shared__ int32_t bins[];
  int c[kOrdPer], rank[kOrdPer];
  order_local(assign, (int64_t)blockIdx.x * kOrdThreads * kOrdPer, n, k, bins, c, rank);
  for (int b = threadIdx.x; b < k; b += kOrdThreads)
    if (bins[b] > 0) atomicAdd(&counts[b], bins[b]);
}

// cursor: the exclusive scan of counts, advanced past each centre's rows.
__global__ __launch_bounds__(kOrdThreads) void order_scatter_kernel(const int32_t* __restrict__ assign, int64_t n,
                                                                    int k, int32_t* __restrict__ cursor,
                                                                    int32_t* __restrict__ order) {
  extern __shared__ int32_t bins[];
  const int64_t row0 = (int64_t)blockIdx.x * kOrdThreads * kOrdPer;
  int c[kOrdPer], rank[kOrdPer];
  order_local(assign, row0, n, k, bins, c, rank);
  for (int b = threadIdx.x; b < k; b += kOrdThreads) {
    const int m = bins[b];
    if (m > 0) bins[b] = atomicAdd(&cursor[b], m);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kOrdPer; ++i)
    if (rank[i] >= 0) order[bins[c[i]] + rank[i]] = (int32_t)(row0 + (int64_t)i * kOrdThreads + threadIdx.x);
}

// round(x * 2^shift) as __float2ll_rn gives it.  Below 2^50 (small: 2^50 / 2^shift)
// by one double fma: x * 2^shift is exact there, adding 1.5 * 2^52 rounds it to an
// integer, to even at ties, and leaves it in the low bits; 4 instructions
// for the 20 of the 64-bit conversion, which the others (and NaN) take.  That
// conversion bound the sums: 500k x 128 133 -> 46 us (5.6 TB/s), 1M x 128 174 ->
// 103 us.  (16 rows in flight or 64 a wave: no change.)
__device__ __forceinline__ long long to_fixed(float x, double scale, float small, int shift) {
  if (__builtin_expect(fabsf(x) < small, 1))
    return (long long)((unsigned long long)__double_as_longlong(__builtin_fma((double)x, scale, 0x1.8p52)) -
                       0x4338000000000000ull);
  return __float2ll_rn(ldexpf(x, shift));
}

// One wave a segment of kOrdSeg grouped rows, lanes over dimensions (NV of
// them a lane).  total: the grouped rows (rows whose centre is in range).
template <int NV>
__global__ __launch_bounds__(256) void order_sum_kernel(const float* __restrict__ x, const int32_t* __restrict__ total,
                                                        const int32_t* __restrict__ assign,
                                                        const int32_t* __restrict__ order, int dim, int shift,
                                                        unsigned long long* __restrict__ sums) {
  constexpr int B = 8;  // rows whose loads are in flight together
  const double scale = ldexp(1.0, shift);
  const float small = ldexpf(1.0f, 50 - shift);
  const int lane = threadIdx.x & 63;
  const int p0 = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))) * kOrdSeg;
  const int p1 = min(p0 + kOrdSeg, *total);
  long long acc[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) acc[j] = 0;
  int cur = -1;
  auto flush = [&]() {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if (cur >= 0 && lane + 64 * j < dim)
        atomicAdd(&sums[(int64_t)cur * dim + lane + 64 * j], (unsigned long long)acc[j]);
      acc[j] = 0;
    }
  };
  for (int b0 = p0; b0 < p1; b0 += kWave) {
    // this batch's rows and centres, one a lane
    const int r_l = b0 + lane < p1 ? order[b0 + lane] : 0;
    const int c_l = b0 + lane < p1 ? assign[r_l] : -1;
    const int m = min(kWave, p1 - b0);
    for (int i0 = 0; i0 < m; i0 += B) {
      float v[B][NV];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const float* xr = x + (int64_t)__builtin_amdgcn_readlane(r_l, min(i0 + i, m - 1)) * dim;
#pragma unroll
        for (int j = 0; j < NV; ++j) v[i][j] = lane + 64 * j < dim ? xr[lane + 64 * j] : 0.0f;
      }
#pragma unroll
      for (int i = 0; i < B; ++i) {
        if (i0 + i >= m) break;
        const int c = __builtin_amdgcn_readlane(c_l, i0 + i);
        if (c != cur) {
          flush();
          cur = c;
        }
#pragma unroll
        for (int j = 0; j < NV; ++j) acc[j] += to_fixed(v[i][j], scale, small, shift);
      }
    }
  }
  flush();
}

__global__ __launch_bounds__(256) void kmeans_accumulate_kernel(
    const float* __restrict__ x, int64_t n, const int32_t* __restrict__ assign, int k, int dim, int shift,
    unsigned long long* __restrict__ sums, int32_t* __restrict__ counts) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * dim) return;
  const int64_t i = t / dim;
  const int d = (int)(t % dim);
  const int c = assign[i];
  if ((uint32_t)c >= (uint32_t)k) return;  // a row without a centre (no finite distance)
  const long long q = __float2ll_rn(ldexpf(x[t], shift));
  atomicAdd(&sums[(int64_t)c * dim + d], (unsigned long long)q);
  if (d == 0) atomicAdd(&counts[c], 1);
}

__global__ void kmeans_finalize_kernel(const unsigned long long* __restrict__ sums,
                                       const int32_t* __restrict__ counts, int k, int dim, int shift,
                                       int empty_rule, float* __restrict__ cent) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)k * dim) return;
  const int c = (int)(t / dim);
  const int cnt = counts[c];
  if (cnt == 0) {
    if (empty_rule == 0) cent[t] = 0.0f;
    return;
  }
  const float inv = __fdiv_rn(1.0f, (float)cnt);
  const float s = (float)ldexp((double)(long long)sums[t], -shift);
  cent[t] = __fmul_rn(s, inv);
}

// ---- nearest codeword of a subspace (A15's E step and A16) -------------------------
// ||r - p||^2 in dimension order.  FMA: the device form, dist = fmaf(diff, diff,
// dist); otherwise the product and the sum each rounded.  (The chain's first
// term adds to zero: the rounded square in both forms.)
template <int S, bool FMA>
__device__ __forceinline__ float pq_dist(const float (&r)[S], const float* p) {
  float d = __fmul_rn(r[0] - p[0], r[0] - p[0]);
#pragma unroll
  for (int j = 1; j < S; ++j) {
    const float df = r[j] - p[j];
    d = FMA ? __builtin_fmaf(df, df, d) : __fadd_rn(d, __fmul_rn(df, df));
  }
  return d;
}

// The first codeword of the smallest distance below FLT_MAX (0 if there is
// none), for R vectors.  Codewords go in blocks: a block's minimum (half an
// instruction a codeword, v_min3) decides whether it takes the lead, and the
// leading block is looked through once more at the end, instead of a compare
// and two selects a codeword.  Each codeword read serves R vectors.  VALU bounds
// both callers, then LDS: 500k x 32 codes of 4 dims encoded in 1231 -> 938 us, an
// E step of 50k rows 114 -> 102 us.  R is 2, or 1 for calls that leave threads
// idle (the launches' rules).  cw: codeword k at cw + k * stride.
constexpr int kPQBlock = 16;
template <int S, bool FMA, int R>
__device__ __forceinline__ void pq_nearest(const float (&r)[R][S], const float* cw, int stride, int (&out)[R]) {
  float best[R];
  int lead[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    best[q] = FLT_MAX;
    lead[q] = -1;
  }
#pragma unroll 1
  for (int k0 = 0; k0 < kPQK; k0 += kPQBlock) {
    float mn[R];
#pragma unroll
    for (int k = 0; k < kPQBlock; k += 2) {
      float p0[S], p1[S];
#pragma unroll
      for (int j = 0; j < S; ++j) {
        p0[j] = cw[(k0 + k) * stride + j];
        p1[j] = cw[(k0 + k + 1) * stride + j];
      }
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const float m2 = fminf(pq_dist<S, FMA>(r[q], p0), pq_dist<S, FMA>(r[q], p1));
        mn[q] = k == 0 ? m2 : fminf(mn[q], m2);
      }
    }
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (mn[q] < best[q]) {
        best[q] = mn[q];
        lead[q] = k0;
      }
  }
#pragma unroll
  for (int q = 0; q < R; ++q) {
    out[q] = 0;
    if (lead[q] < 0) continue;
    for (int k = kPQBlock - 1; k >= 0; --k)
      if (pq_dist<S, FMA>(r[q], cw + (lead[q] + k) * stride) == best[q]) out[q] = lead[q] + k;
  }
}

// ---- A16: residual PQ encoding (kmeans_gpu.cuh:403-445) ---------------------------
// Codebook staged in LDS as [k][m][S] so lanes of one wave (consecutive
// subspaces, same codeword) read consecutive 16-byte chunks.  FMA: the device
// form, dist = fmaf(diff, diff, dist) as nvcc contracts encode_residuals_kernel
// (kmeans_gpu.cuh:428-433); otherwise the host form of encode_residuals_to_pq
// (pq_utils.h:160-166, built without FMA): the product and the sum each rounded.
// A thread takes the same subspace of R rows; one workgroup a CU, as the codebook
// fills its LDS, each staging it once.
// pos (may be null): row i's codes go to row pos[i], nowhere if it is below 0.
template <int S, bool FMA, int R>
__global__ __launch_bounds__(1024) void pq_encode_kernel(const float* __restrict__ x, int64_t n, int dim, int m,
                                                         const int32_t* __restrict__ assign,
                                                         const float* __restrict__ cent, uint32_t ncent,
                                                         const float* __restrict__ codebook,
                                                         const int32_t* __restrict__ pos,
                                                         uint8_t* __restrict__ codes) {
  extern __shared__ __align__(16) float cbs[];  // [256][m][S]
  for (int t = threadIdx.x; t < kPQK * m * S; t += blockDim.x) {
    const int j = t % S, sub = (t / S) % m, kk = t / (S * m);
    cbs[t] = codebook[((size_t)sub * kPQK + kk) * S + j];
  }
  __syncthreads();
  const int64_t total = (n + R - 1) / R * m;
  for (int64_t pr = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; pr < total; pr += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i0 = pr / m * R;
    const int sub = (int)(pr % m);
    float r[R][S];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int64_t i = min(i0 + q, n - 1);
      const float* xi = x + i * dim + sub * S;
      const uint32_t c = (uint32_t)assign[i];
      const float* ci = cent + (int64_t)(c < ncent ? c : 0u) * dim + sub * S;
#pragma unroll
      for (int j = 0; j < S; ++j) r[q][j] = xi[j] - ci[j];
    }
    int bk[R];
    pq_nearest<S, FMA, R>(r, cbs + sub * S, m * S, bk);
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (i0 + q < n) {
        const int64_t to = pos ? (int64_t)pos[i0 + q] : i0 + q;
        if (to >= 0) codes[to * m + sub] = (uint8_t)bk[q];
      }
  }
}

// ---- A17: inverted lists (build_global.cu:225-240) ---------------------------------
// Rows in list order, ids ascending inside a list: a stable counting sort by
// list.  The rows are cut into chunks, one wave each; tab[chunk][list] first
// counts, then holds where the chunk's rows of that list begin inside it, and
// the scatter advances it batch by batch of 64 rows.  The table lives in global
// memory, so any number of lists works; a wave's adds to it are in batch order.
// Latency bounds it (a wave's 32 batches each wait for an atomic): the scatter
// takes 110 us at 500k rows and 1024 lists.  The host sorted before: a build of
// those rows 48.7 -> 44.6 ms.
__global__ __launch_bounds__(256) void list_count_kernel(const int32_t* __restrict__ assign, int64_t n, int nlist,
                                                         int64_t chunk, int32_t* __restrict__ tab) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int32_t l = assign[i];
  if ((uint32_t)l < (uint32_t)nlist) atomicAdd(&tab[(i / chunk) * nlist + l], 1);
}

// tab's columns to exclusive prefix sums over the chunks, and the lists' sizes.
__global__ __launch_bounds__(64) void list_prefix_kernel(int32_t* __restrict__ tab, int nchunks, int nlist,
                                                         int32_t* __restrict__ sizes) {
  constexpr int B = 16;  // chunks whose loads are in flight together
  const int l = blockIdx.x * 64 + threadIdx.x;
  if (l >= nlist) return;
  int32_t run = 0;
  for (int c0 = 0; c0 < nchunks; c0 += B) {
    int32_t v[B];
#pragma unroll
    for (int b = 0; b < B; ++b) v[b] = c0 + b < nchunks ? tab[(int64_t)(c0 + b) * nlist + l] : 0;
#pragma unroll
    for (int b = 0; b < B; ++b) {
      if (c0 + b < nchunks) tab[(int64_t)(c0 + b) * nlist + l] = run;
      run += v[b];
    }
  }
  sizes[l] = run;
}

// One wave a chunk: row -> place in list order.
__global__ __launch_bounds__(64) void list_scatter_kernel(const int32_t* __restrict__ assign, int64_t n, int nlist,
                                                          int64_t chunk, const int32_t* __restrict__ offsets,
                                                          int32_t* __restrict__ tab, int32_t* __restrict__ ids,
                                                          int32_t* __restrict__ pos) {
  const int lane = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.x * chunk, r1 = min(r0 + chunk, n);
  int32_t* t = tab + (int64_t)blockIdx.x * nlist;
  for (int64_t b = r0; b < r1; b += kWave) {
    const int64_t i = b + lane;
    const int32_t l = i < r1 ? assign[i] : -1;
    const bool ok = (uint32_t)l < (uint32_t)nlist;
    // the lanes of the same list: their first one, how many come before this
    // one, and how many there are
    int first = kWave, before = 0, all = 0;
#pragma unroll
    for (int o = 0; o < kWave; ++o) {
      const bool same = __builtin_amdgcn_readlane(l, o) == l;
      first = same && first == kWave ? o : first;
      before += same && o < lane;
      all += same;
    }
    const int32_t old = ok && lane == first ? atomicAdd(&t[l], all) : 0;
    const int32_t at = __shfl(old, first, kWave);
    if (ok) {
      const int32_t p = offsets[l] + at + before;
      ids[p] = (int32_t)i;
      pos[i] = p;
    } else if (i < r1) {
      pos[i] = -1;
    }
  }
}

// ---- A15: PQ codebook training (pq_utils.h:17-138) ------------------------------
__global__ void pq_residuals_kernel(const float* __restrict__ x, int dim, const int32_t* __restrict__ rows,
                                    int nrows, const int32_t* __restrict__ assign,
                                    const float* __restrict__ cent, uint32_t ncent, float* __restrict__ res) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)nrows * dim) return;
  const int r = (int)(t / dim), d = (int)(t % dim);
  const int64_t o = rows[r];
  const uint32_t c = (uint32_t)assign[o];
  res[t] = x[o * dim + d] - cent[(int64_t)(c < ncent ? c : 0u) * dim + d];
}

// codebook[m][c][j] = res[init_rows[m][c]][m*S + j]
__global__ void pq_init_kernel(const float* __restrict__ res, int dim, int m, int S,
                               const int32_t* __restrict__ init_rows, float* __restrict__ codebook) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= m * kPQK * S) return;
  const int j = t % S, c = (t / S) % kPQK, sub = t / (S * kPQK);
  codebook[t] = res[(int64_t)init_rows[sub * kPQK + c] * dim + sub * S + j];
}

// E-step of run_kmeans_pq_fast (pq_utils.h:39-52), host floating point: the
// square and the running sum are rounded separately (no fused multiply-add).
template <int S, int R>
__global__ __launch_bounds__(256) void pq_estep_kernel(const float* __restrict__ res, int ns, int dim, int m,
                                                       const float* __restrict__ codebook,
                                                       uint8_t* __restrict__ assign_pq, int stride) {
  __shared__ __align__(16) float cbs[kPQK * S];
  const int sub = blockIdx.y;
  for (int t = threadIdx.x; t < kPQK * S; t += blockDim.x) cbs[t] = codebook[(size_t)sub * kPQK * S + t];
  __syncthreads();
  const int i0 = blockIdx.x * 256 * R + threadIdx.x;
  if (i0 >= ns) return;
  float xv[R][S];
#pragma unroll
  for (int q = 0; q < R; ++q)
#pragma unroll
    for (int j = 0; j < S; ++j) xv[q][j] = res[(int64_t)min(i0 + 256 * q, ns - 1) * dim + sub * S + j];
  int bc[R];
  pq_nearest<S, false, R>(xv, cbs, S, bc);
#pragma unroll
  for (int q = 0; q < R; ++q)
    if (i0 + 256 * q < ns) assign_pq[(size_t)sub * stride + i0 + 256 * q] = (uint8_t)bc[q];
}

// M-step (pq_utils.h:54-71): members of cluster c summed in double in
// ascending row order, (float)(sum / count); an empty cluster keeps its
// centre.  One wave per (cluster, subspace): it reads the subspace's
// assignments a byte each, 1024 a step, lists the members in LDS in order, and
// once 64 or more are
// listed reads their values 64 rows at a time, all loads in flight together, before lane j < S adds dimension j's in order.  Scanning the
// assignments bounds it (every cluster's wave reads them all, from L2).
constexpr int kMStep = 1024, kMList = kMStep + 64;
template <int S>
__global__ __launch_bounds__(64) void pq_mstep_kernel(const float* __restrict__ res, int ns, int dim,
                                                      const uint8_t* __restrict__ assign_pq, int stride,
                                                      float* __restrict__ codebook) {
  __shared__ int list[kMList];
  __shared__ float val[kWave * S];
  const int c = blockIdx.x, sub = blockIdx.y, lane = threadIdx.x;
  const uint4* as = reinterpret_cast<const uint4*>(assign_pq + (size_t)sub * stride);
  const uint32_t c4 = (uint32_t)c * 0x01010101u;
  const float* rs = res + sub * S;
  double acc = 0.0;
  int cnt = 0, m = 0;  // members so far, and of them those listed but not yet added
  // adds the first r <= 64 listed rows from `at` on
  auto add = [&](int at, int r) {
    float v[S];
#pragma unroll
    for (int k = 0; k < S; ++k) {
      const int e = min(lane + k * kWave, r * S - 1);
      v[k] = rs[(int64_t)list[at + e / S] * dim + e % S];
    }
#pragma unroll
    for (int k = 0; k < S; ++k) val[lane + k * kWave] = v[k];
    wave_lds_order();
    if (lane < S)
#pragma unroll 8
      for (int i = 0; i < r; ++i) acc += (double)val[i * S + lane];
    wave_lds_order();
  };
  // the lane's 16 rows of a step: bit i set where row i is a member
  auto members = [&](int base, uint4 w) {
    const uint32_t v[4] = {w.x, w.y, w.z, w.w};
    uint32_t hit = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t x = v[k] ^ c4;  // a zero byte: a member
      const uint32_t z = ~(((x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | x) & 0x80808080u;
      hit |= (((z >> 7) * 0x01020408u) >> 24) << (4 * k);
    }
    const int left = ns - (base + 16 * lane);
    return left >= 16 ? hit : left > 0 ? hit & ((1u << left) - 1u) : 0u;
  };
  const int last = stride / 16 - 1;
  uint4 next = as[min(lane, last)];
  for (int base = 0; base < ns; base += kMStep) {
    uint32_t hit = members(base, next);
    next = as[min((base + kMStep) / 16 + lane, last)];  // past the end: the last 16, unused
    const int h = __popc(hit);
    int incl = h;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int u = __shfl_up(incl, o, kWave);
      if (lane >= o) incl += u;
    }
    const int all = __builtin_amdgcn_readlane(incl, kWave - 1);
    int at = m + incl - h;
    while (hit) {
      list[at++] = base + 16 * lane + __ffs((int)hit) - 1;
      hit &= hit - 1;
    }
    wave_lds_order();
    m += all;
    cnt += all;
    if (m >= kWave) {  // at least 1024 free places after it
      int i = 0;
      for (; i + kWave <= m; i += kWave) add(i, kWave);
      const int rest = m - i;
      const int keep = lane < rest ? list[i + lane] : 0;
      wave_lds_order();
      if (lane < rest) list[lane] = keep;
      wave_lds_order();
      m = rest;
    }
  }
  if (m > 0) add(0, m);
  if (lane < S && cnt > 0) codebook[((size_t)sub * kPQK + c) * S + lane] = (float)(acc / (double)cnt);
}

// ---- k-means++ seeding (definition: oracle.cpp orc_kmeans_init_pp) ---------------
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

constexpr int kPPBlock = 1024;

// The exact skip of the d2 update.  asg[i] is the centre whose distance d2[i]
// holds, cc[a] = ||c_new - c_a||^2 for every earlier centre a.  By the
// triangle inequality ||x - c_new|| >= ||c_new - c_a|| - ||x - c_a||, so with
// cc >= 4 (1 + 1%) d2 the new distance exceeds d2 by about 2% even after the
// roundings of the three fused chains (each within 1e-4 relative of its exact
// value, D <= 256): the row cannot move, and its d2, weight and asg stay as
// they are without reading the row.  d2 = 0 rows never move either.  The
// 1e-4 bound is relative and needs values far above the fp32 subnormal range
// (where a rounding step is absolute), so rows with 0 < d2 < 2^-100 always
// compute; from d2 >= 2^-100 on, cc >= 4 d2 is as far above it.
constexpr float kPPSkip = 4.04f;
constexpr float kPPSkipMin = 0x1p-100f;

// Whether row i must compute its distance to the new centre (always, when
// asg is null: the first passes).
__device__ __forceinline__ bool pp_needs(const int32_t* asg, const float* cc, int64_t i, float old) {
  if (asg == nullptr) return true;
  if (old == 0.0f) return false;
  return !(old >= kPPSkipMin && cc[asg[i]] >= kPPSkip * old);
}

// d2[i] = min(d2[i], ||x_i - c||^2) (init: d2 = dist); w[i] = round(d2 * 2^S);
// part[b] = sum of w over block b.  With asg: rows the triangle bound clears
// are skipped, and a row that moves records centre j.
__global__ __launch_bounds__(kPPBlock) void pp_update_kernel(const float* __restrict__ x, int64_t n, int dim,
                                                             const float* __restrict__ c, int init,
                                                             float* __restrict__ d2, const int* __restrict__ shift,
                                                             uint64_t* __restrict__ w, uint64_t* __restrict__ part,
                                                             int32_t* __restrict__ asg, const float* __restrict__ cc,
                                                             int j, const int32_t* __restrict__ picked,
                                                             uint8_t* __restrict__ chosen) {
  if (picked && blockIdx.x == 0 && threadIdx.x == 0) chosen[*picked] = 1;  // the pick itself must not see it
  const int64_t i = (int64_t)blockIdx.x * kPPBlock + threadIdx.x;
  uint64_t wi = 0;
  if (i < n) {
    const float old = init ? 0.0f : d2[i];
    float v = old;
    bool moved = false;
    if (init || pp_needs(init ? nullptr : asg, cc, i, old)) {
      const float* xi = x + i * dim;
      float acc = 0.0f;
      for (int d = 0; d < dim; ++d) {
        const float df = xi[d] - c[d];
        acc = __builtin_fmaf(df, df, acc);
      }
      moved = init || acc < old;
      v = moved ? acc : old;
    }
    if (moved) {
      d2[i] = v;
      if (asg) asg[i] = j;
    }
    if (shift) {
      wi = (uint64_t)__double2ll_rn(ldexp((double)v, *shift));
      if (moved || !asg) w[i] = wi;
    }
  }
  if (shift) {
    __shared__ uint64_t s[kPPBlock / kWave];
    uint64_t t = wi;
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) t += __shfl_xor(t, m, kWave);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
      uint64_t tot = 0;
      for (int j = 0; j < kPPBlock / kWave; ++j) tot += s[j];
      part[blockIdx.x] = tot;
    }
  }
}

// The same update for rows of whole 128-byte lines.  A workgroup takes the
// kPPBlock rows of one part sum, four a thread; the rows that must compute are
// packed per wave and read 64 at a time, eight lanes a row (wave_rows_l2: the
// same chain, on c - x).  The rows read bound it: of 500k rows of 128 dims in
// 1000 clusters a pass computes a third on average, 14.9 us, 10.4 us in the
// median.  (One lane a row, 1024 threads and 128 registers of row: 15.0 us; 512
// threads with half the hand-over buffer a wave: 15.6 us.)  Two lines a load batch:
// seeding 1M x 128, 1024 centres, 39.3 -> 37.4 ms, 500k 22.9 -> 22.8; four lines
// 39.3 and 23.4.  (Ruling rows out on a half-size fp16 copy first: 25 and 39 ms, the
// second look's latency costs what the bytes save.)
constexpr int kPPThreads = 256;
template <int D>
__global__ __launch_bounds__(kPPThreads) void pp_update_rows_kernel(
    const float* __restrict__ x, int64_t n, const float* __restrict__ c, int init, float* __restrict__ d2,
    const int* __restrict__ shift, uint64_t* __restrict__ w, uint64_t* __restrict__ part, int32_t* __restrict__ asg,
    const float* __restrict__ cc, int jc, const int32_t* __restrict__ picked, uint8_t* __restrict__ chosen) {
  constexpr int kPer = kPPBlock / kPPThreads, kWaves = kPPThreads / kWave;
  __shared__ __align__(16) float tr_s[kWaves][row_tr_floats()];
  __shared__ float cs[D];
  __shared__ int list_s[kWaves][kPer * kWave];
  __shared__ float dist_s[kWaves][kPer * kWave];
  __shared__ uint64_t s[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (picked && blockIdx.x == 0 && tid == 0) chosen[*picked] = 1;  // the pick itself must not see it
  for (int d = tid; d < D; d += kPPThreads) cs[d] = c[d];
  __syncthreads();
  const int64_t b0 = (int64_t)blockIdx.x * kPPBlock;
  int* list = list_s[wave];
  float* dist = dist_s[wave];
  float old[kPer];
  int at[kPer];  // the row's place in the wave's list, -1: none
  int m = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int64_t i = b0 + k * kPPThreads + tid;
    old[k] = i < n && !init ? d2[i] : 0.0f;
    const bool f = i < n && (init || pp_needs(asg, cc, i, old[k]));
    const uint64_t bm = __ballot(f);
    at[k] = f ? m + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u))
              : -1;
    if (f) list[at[k]] = (int)i;
    m += __popcll(bm);
  }
  wave_lds_order();
  for (int p = 0; p < m; p += kWave)
    dist[p + lane] = wave_rows_l2<D, kWave, 2>(x, list[min(p + lane, m - 1)], cs, tr_s[wave]);
  wave_lds_order();
  uint64_t sum = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int64_t i = b0 + k * kPPThreads + tid;
    if (i >= n) continue;
    const float acc = at[k] >= 0 ? dist[at[k]] : 0.0f;
    const bool moved = at[k] >= 0 && (init || acc < old[k]);
    const float v = moved ? acc : old[k];
    if (moved) {
      d2[i] = v;
      if (asg) asg[i] = jc;
    }
    if (shift) {
      const uint64_t wi = (uint64_t)__double2ll_rn(ldexp((double)v, *shift));
      if (moved || !asg) w[i] = wi;
      sum += wi;
    }
  }
  if (shift) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, kWave);
    if (lane == 0) s[wave] = sum;
    __syncthreads();
    if (tid == 0) {
      uint64_t tot = 0;
      for (int k = 0; k < kWaves; ++k) tot += s[k];
      part[blockIdx.x] = tot;
    }
  }
}

// One pass of the d2 update: the row kernel for the common dims (rows 16-byte
// aligned), the generic one otherwise.
// asg == nullptr: every row computes (the first passes); otherwise the skip
// above applies (cc filled for centre j).  picked: the row of centre j, which
// the pass marks in chosen (nullptr: already marked).
fgpu_status pp_update(const float* x, int64_t n, int dim, const float* c, int init, float* d2, const int* shift,
                      uint64_t* w, uint64_t* part, int nb, int32_t* asg, const float* cc, int j,
                      const int32_t* picked, uint8_t* chosen, hipStream_t s) {
  const bool vec = ((uintptr_t)x & 15) == 0;
#define FGPU_PP(D)                                                                                                   \
  if (vec && dim == D) {                                                                                             \
    hipLaunchKernelGGL(pp_update_rows_kernel<D>, dim3(nb), dim3(kPPThreads), 0, s, x, n, c, init, d2, shift, w, part, \
                       asg, cc, j, picked, chosen);                                                                  \
    FGPU_HIP(hipGetLastError());                                                                                     \
    return FGPU_OK;                                                                                                  \
  }
  FGPU_PP(128)
  FGPU_PP(96)
  FGPU_PP(64)
  FGPU_PP(32)
#undef FGPU_PP
  hipLaunchKernelGGL(pp_update_kernel, dim3(nb), dim3(kPPBlock), 0, s, x, n, dim, c, init, d2, shift, w, part, asg, cc, j,
                     picked, chosen);
  FGPU_HIP(hipGetLastError());
  return FGPU_OK;
}

// shift from the first round's max d2 (so n * max w < 2^62).
__global__ __launch_bounds__(1024) void pp_shift_kernel(const float* __restrict__ d2, int64_t n, int* __restrict__ shift) {
  __shared__ float part[16];
  float m = 0.0f;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) m = fmaxf(m, d2[i]);
  m = wave_max_f(m);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    float mx = 0.0f;
    for (int j = 0; j < 16; ++j) mx = fmaxf(mx, part[j]);
    int e = 0;
    if (mx > 0.0f) frexp((double)mx, &e);
    int lg = 0;
    while ((1LL << lg) < n) ++lg;
    int s = 62 - lg - e;
    *shift = s > 60 ? 60 : (s < 0 ? 0 : s);
  }
}

// Inclusive scan of one u64 a thread over a workgroup of kPPBlock threads.
__device__ __forceinline__ uint64_t pp_scan(uint64_t v, uint64_t* wsum) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint64_t t = __shfl_up(v, o, kWave);
    if (lane >= o) v += t;
  }
  __syncthreads();  // wsum's last readers
  if (lane == kWave - 1) wsum[wave] = v;
  __syncthreads();
  uint64_t before = 0;
#pragma unroll
  for (int i = 0; i < kPPBlock / kWave; ++i) before += i < wave ? wsum[i] : 0;
  return v + before;
}

// Pick the next centre: smallest i with inclusive prefix(w) > u, u = r_j % total
// (every weight zero: the lowest row not yet chosen), and its squared distance
// to every earlier centre, cc[a] = ||c_j - c_a||^2, which only the update's skip
// bound reads (any summation order).  Every workgroup finds the same pick and
// takes 16 earlier centres, a wave each, lanes over dimensions; the first one
// writes the row and the centre.  One launch: the pick (two scans by wave
// shuffles) and the distances took 8.3 + 3.2 us as two kernels and a
// launch more, 6.7 us now (500k rows, 1024 centres).
__global__ __launch_bounds__(kPPBlock) void pp_pick_kernel(const uint64_t* __restrict__ w,
                                                           const uint64_t* __restrict__ part, int nblocks, int64_t n,
                                                           uint64_t seed, int j, const uint8_t* __restrict__ chosen,
                                                           int32_t* __restrict__ rows, const float* __restrict__ x,
                                                           int dim, float* __restrict__ cent, float* __restrict__ cc) {
  __shared__ uint64_t wsum[kPPBlock / kWave];
  __shared__ uint64_t s_before, s_tot;
  __shared__ int s_blk;
  __shared__ int64_t s_pick;
  const int tid = threadIdx.x;
  if (tid == 0) {
    s_blk = -1;
    s_pick = -1;
    s_before = 0;
  }
  uint64_t tot = 0, first = 0;  // first: this thread's part sum of the first chunk, scanned
  for (int base = 0; base < nblocks; base += kPPBlock) {
    const uint64_t incl = pp_scan(base + tid < nblocks ? part[base + tid] : 0, wsum);
    if (base == 0) first = incl;
    if (tid == kPPBlock - 1) s_tot = incl;
    __syncthreads();
    tot += s_tot;
    __syncthreads();
  }
  if (tot != 0) {
    const uint64_t u = mix64(seed ^ mix64(7) ^ mix64(0x100000000ull + (uint64_t)j)) % tot;
    uint64_t acc = 0;  // the chunks before this one
    for (int base = 0; base < nblocks; base += kPPBlock) {
      const uint64_t v = base + tid < nblocks ? part[base + tid] : 0;
      const uint64_t in = base == 0 ? first : pp_scan(v, wsum);
      const uint64_t incl = acc + in, excl = incl - v;
      if (base + tid < nblocks && excl <= u && u < incl) {
        s_blk = base + tid;
        s_before = excl;
      }
      if (base + kPPBlock < nblocks) {
        if (tid == kPPBlock - 1) s_tot = in;
        __syncthreads();
        acc += s_tot;
        __syncthreads();
      }
    }
    __syncthreads();
    const int64_t i = (int64_t)max(s_blk, 0) * kPPBlock + tid;  // (a block holds u by construction)
    const uint64_t wi = i < n ? w[i] : 0;
    const uint64_t incl = s_before + pp_scan(wi, wsum), excl = incl - wi;
    if (i < n && excl <= u && u < incl) s_pick = i;
    __syncthreads();
    if (tid == 0 && s_pick < 0) s_pick = (int64_t)max(s_blk, 0) * kPPBlock;
  } else if (tid == 0) {
    int64_t pick = 0;
    for (int64_t i = 0; i < n; ++i)
      if (!chosen[i]) {
        pick = i;
        break;
      }
    s_pick = pick;
  }
  __syncthreads();
  const float* xr = x + s_pick * dim;
  if (blockIdx.x == 0) {
    if (tid == 0) rows[j] = (int32_t)s_pick;
    for (int d = tid; d < dim; d += kPPBlock) cent[(int64_t)j * dim + d] = xr[d];
  }
  const int a = blockIdx.x * (kPPBlock / kWave) + (tid >> 6), lane = tid & 63;
  if (a >= j) return;
  const float* ca = cent + (size_t)a * dim;
  float acc = 0.0f;
  for (int d = lane; d < dim; d += kWave) {
    const float df = xr[d] - ca[d];
    acc = __builtin_fmaf(df, df, acc);
  }
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) acc += shfl_xor_f(acc, m);
  if (lane == 0) cc[a] = acc;
}

__global__ void pp_take_kernel(const float* __restrict__ x, int dim, const int32_t* __restrict__ rows, int j,
                               float* __restrict__ cent, uint8_t* __restrict__ chosen) {
  const int r = rows[j];
  for (int d = threadIdx.x; d < dim; d += blockDim.x) cent[(int64_t)j * dim + d] = x[(int64_t)r * dim + d];
  if (threadIdx.x == 0) chosen[r] = 1;
}

__global__ void pp_first_kernel(int64_t n, uint64_t seed, int32_t* __restrict__ rows, uint8_t* __restrict__ chosen) {
  const int64_t r0 = (int64_t)(mix64(seed ^ mix64(7)) % (uint64_t)n);
  rows[0] = (int32_t)r0;
  (void)chosen;
}

template <class K, class... A>
fgpu_status launch1d(K kern, int64_t n, int block, hipStream_t s, A... args) {
  if (n <= 0) return FGPU_OK;
  hipLaunchKernelGGL(kern, dim3((unsigned)((n + block - 1) / block)), dim3(block), 0, s, args...);
  FGPU_HIP(hipGetLastError());
  return FGPU_OK;
}

// ---------------------------------------------------------------------------
// Per-list radius of the decoded residuals: rmax[l] >= ||decode(x)|| for every
// vector x of list l, where decode(x)_m = codebook[m][code_m].  Squared
// codeword norms and their sums are formed in double (each product of two
// floats is exact in double; the few roundings of the sums are far below the
// final margin), and the float result is rounded up.  One block per list.
__global__ __launch_bounds__(256) void list_radius_kernel(const float* __restrict__ cb, int m, int sub,
                                                          const uint8_t* __restrict__ codes,
                                                          const int32_t* __restrict__ offsets,
                                                          float* __restrict__ rmax) {
  extern __shared__ double cbn2[];  // [m][256]
  for (int i = threadIdx.x; i < m * kPQK; i += blockDim.x) {
    double t = 0.0;
    for (int d = 0; d < sub; ++d) {
      const double v = cb[(size_t)i * sub + d];
      t += v * v;
    }
    cbn2[i] = t;
  }
  __syncthreads();
  const int l = blockIdx.x;
  const int start = offsets[l], end = offsets[l + 1];
  double mx = 0.0;
  for (int v = start + threadIdx.x; v < end; v += blockDim.x) {
    const uint8_t* c = codes + (size_t)v * m;
    double t = 0.0;
    for (int j = 0; j < m; ++j) t += cbn2[j * kPQK + c[j]];
    mx = fmax(mx, t);
  }
  __shared__ double red[256];
  red[threadIdx.x] = mx;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + o]);
    __syncthreads();
  }
  if (threadIdx.x == 0) rmax[l] = __double2float_ru(sqrt(red[0]) * (1.0 + 0x1p-30));
}

}  // namespace

fgpu_status launch_probe_counts(const uint32_t* probes, int nq, int nprobe, int nlist, const int32_t* offsets,
                                int32_t* counts, int32_t* offs, hipStream_t s) {
  FGPU_TRY(launch1d(probe_counts_kernel, nq, 256, s, probes, nq, nprobe, nlist, offsets, counts));
  hipLaunchKernelGGL(exclusive_scan_kernel, dim3(1), dim3(1024), 0, s, counts, nq, offs);
  FGPU_HIP(hipGetLastError());
  return FGPU_OK;
}

fgpu_status launch_maxabs(const float* x, int64_t count, float* out, hipStream_t s) {
  // out must hold 1024 floats of scratch; the result lands in out[1023].
  hipLaunchKernelGGL(maxabs_partial_kernel, dim3(1023), dim3(256), 0, s, x, count, out);
  FGPU_HIP(hipGetLastError());
  return launch_max_reduce(out, 1023, out + 1023, s);
}

// From kOrderedMinRows rows on, the form that takes less time by these fits (us).
// Atomics: 7.5 a million of them, at least 24, and 0.22 for each row a centre
// has on average (they queue on its sums).  Grouped: the launches, a row's loads
// (64 dims each), and the scan and the histograms of the centres.  Measured,
// atomics / grouped: 32768 rows of 128 dims, 256 centres 70 / 39, 1024 40 / 41,
// 4096 35 / 52, 16384 42 / 86; 65536 rows, 4096 60 / 53, 8192 61 / 64; 131072 rows,
// 16384 115 / 83; 65536 rows of 32 dims, 256 95 / 35, 2048 29 / 39; 262144 rows,
// 8192 68 / 56, 16384 66 / 71; 32768 rows of 200 dims, 256 80 / 53, 2048 49 / 59.
static bool grouping_pays(int64_t n, int k, int dim) {
  const double atomics = std::max(24.0, 7.5 * (double)n * dim / (1 << 20)) + 0.22 * (double)n / k;
  return n >= kOrderedMinRows && k <= kOrderedMaxCentres && dim <= 256 &&
         atomics > 28.0 + 8.0 * ((dim + 63) / 64) + 3.75 * k / 1024;
}

// Grouping scratch: the centres' offsets and chunk counts, and the row order.
static size_t order_fixed_bytes(int k) { return carve_bytes<int32_t>((size_t)k + 1) + carve_bytes<int32_t>(k) + 256; }
size_t kmeans_order_bytes(int k, int64_t rows) { return order_fixed_bytes(k) + carve_bytes<int32_t>(rows); }

fgpu_status launch_kmeans_accumulate(const float* x, int64_t n, const int32_t* assign, int k, int dim, int shift,
                                     unsigned long long* sums, int32_t* counts, void* ows, size_t ows_bytes,
                                     hipStream_t s) {
  FGPU_TRY(launch1d(fill_u64_kernel, (int64_t)k * dim, 256, s, sums, (int64_t)k * dim));
  FGPU_TRY(launch1d(fill_i32_kernel, (int64_t)k, 256, s, counts, (int64_t)k));
  const size_t fixed = order_fixed_bytes(k);
  const int64_t fit = ows && ows_bytes > fixed ? (int64_t)((ows_bytes - fixed) / sizeof(int32_t)) : 0;
  if (!grouping_pays(n, k, dim) || fit < std::min<int64_t>(n, kOrderedMinRows))
    return launch1d(kmeans_accumulate_kernel, n * dim, 256, s, x, n, assign, k, dim, shift, sums, counts);
  Carve cv(ows, ows_bytes);
  int32_t* cursor = cv.take<int32_t>((size_t)k + 1);
  int32_t* cnt = cv.take<int32_t>((size_t)k);  // this chunk's counts
  const int64_t rows = std::min<int64_t>({n, fit, (int64_t)1 << 30});  // a chunk's row numbers are 32-bit
  int32_t* order = cv.take<int32_t>((size_t)rows);
  FGPU_CHECK(cv.ok(), FGPU_ERR_WORKSPACE, "kmeans_update: workspace too small");
  const size_t lds = (size_t)k * sizeof(int32_t);
  for (const void* f : {(const void*)order_count_kernel, (const void*)order_scatter_kernel})
    FGPU_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  const int nv = (dim + 63) / 64;
  for (int64_t b = 0; b < n; b += rows) {
    const int64_t nb = std::min<int64_t>(rows, n - b);
    const unsigned g = (unsigned)((nb + kOrdThreads * kOrdPer - 1) / (kOrdThreads * kOrdPer));
    int32_t* cc = n <= rows ? counts : cnt;
    if (cc == cnt) FGPU_TRY(launch1d(fill_i32_kernel, (int64_t)k, 256, s, cnt, (int64_t)k));
    hipLaunchKernelGGL(order_count_kernel, dim3(g), dim3(kOrdThreads), lds, s, assign + b, nb, k, cc);
    hipLaunchKernelGGL(exclusive_scan_kernel, dim3(1), dim3(1024), 0, s, cc, k, cursor);
    hipLaunchKernelGGL(order_scatter_kernel, dim3(g), dim3(kOrdThreads), lds, s, assign + b, nb, k, cursor, order);
    const dim3 sg((unsigned)((nb + 4 * kOrdSeg - 1) / (4 * kOrdSeg)));
    const float* xb = x + b * dim;
    const int32_t* tot = cursor + k;  // the scan's total; the scatter leaves it alone
#define FGPU_OS(V) \
  if (nv == V)     \
    hipLaunchKernelGGL(order_sum_kernel<V>, sg, dim3(256), 0, s, xb, tot, assign + b, order, dim, shift, sums)
    FGPU_OS(1);
    FGPU_OS(2);
    FGPU_OS(3);
    FGPU_OS(4);
#undef FGPU_OS
    if (cc == cnt) FGPU_TRY(launch1d(add_i32_kernel, (int64_t)k, 256, s, counts, cnt, (int64_t)k));
  }
  FGPU_HIP(hipGetLastError());
  return FGPU_OK;
}

fgpu_status launch_kmeans_finalize(const unsigned long long* sums, const int32_t* counts, int k, int dim, int shift,
                                   int empty_rule, float* cent, hipStream_t s) {
  return launch1d(kmeans_finalize_kernel, (int64_t)k * dim, 256, s, sums, counts, k, dim, shift, empty_rule, cent);
}

fgpu_status launch_gather_rows(const float* x, int dim, const int32_t* rows, int nrows, float* out, hipStream_t s) {
  return launch1d(gather_rows_kernel, (int64_t)nrows * dim, 256, s, x, dim, rows, nrows, out);
}

// Rows of a chunk: 2048, more once the table would pass 256 MB.
static int64_t list_chunk(int64_t n, int nlist) {
  const int64_t most = std::max<int64_t>(1, (int64_t)(256 << 20) / (4 * (int64_t)nlist));
  const int64_t c = std::max<int64_t>(2048, (n + most - 1) / most);
  return (c + kWave - 1) / kWave * kWave;
}
static int list_chunks(int64_t n, int nlist) {
  const int64_t c = list_chunk(n, nlist);
  return (int)((n + c - 1) / c);
}

size_t list_order_ws_bytes(int64_t n, int nlist) {
  return carve_bytes<int32_t>((size_t)list_chunks(n, nlist) * nlist) + carve_bytes<int32_t>((size_t)nlist);
}

fgpu_status launch_list_order(const int32_t* assign, int64_t n, int nlist, int32_t* offsets, int32_t* ids,
                              int32_t* pos, void* ws, size_t ws_bytes, hipStream_t s) {
  const int64_t chunk = list_chunk(n, nlist);
  const int nc = list_chunks(n, nlist);
  Carve cv(ws, ws_bytes);
  int32_t* tab = cv.take<int32_t>((size_t)nc * nlist);
  int32_t* sizes = cv.take<int32_t>((size_t)nlist);
  FGPU_CHECK(cv.ok(), FGPU_ERR_WORKSPACE, "list_order: workspace too small");
  FGPU_TRY(launch1d(fill_i32_kernel, (int64_t)nc * nlist, 256, s, tab, (int64_t)nc * nlist));
  FGPU_TRY(launch1d(list_count_kernel, n, 256, s, assign, n, nlist, chunk, tab));
  FGPU_TRY(launch1d(list_prefix_kernel, nlist, 64, s, tab, nc, nlist, sizes));
  hipLaunchKernelGGL(exclusive_scan_kernel, dim3(1), dim3(1024), 0, s, sizes, nlist, offsets);
  hipLaunchKernelGGL(list_scatter_kernel, dim3((unsigned)nc), dim3(kWave), 0, s, assign, n, nlist, chunk, offsets, tab,
                     ids, pos);
  FGPU_HIP(hipGetLastError());
  return FGPU_OK;
}

fgpu_status launch_pq_encode(const float* x, int64_t n, int dim, int m, const int32_t* assign, const float* cent,
                             const float* codebook, uint8_t* codes, hipStream_t s, int fma_mode, int ncent,
                             const int32_t* pos) {
  const int S = dim / m;
  const size_t lds = (size_t)kPQK * dim * sizeof(float);
  FGPU_CHECK(lds <= 160 * 1024, FGPU_ERR_UNSUPPORTED, "pq_encode: codebook exceeds LDS");
  if (n <= 0) return FGPU_OK;
  // Two rows a thread, unless one row each leaves none of the 256 x 1024 threads a
  // second turn: then a thread's own work is the time.  Measured (us, two / one row
  // a thread, 128 dims): 1000 rows, 32 codes 39 / 30, 16 codes 59 / 46; 16000 rows,
  // 16 codes 61 / 50, 32 codes 44 / 61; 40000 rows, 16 codes 108 / 136.
  const int rows = n * m <= 256 * 1024 ? 1 : 2;
  const int64_t units = (n + rows - 1) / rows * m;
  const unsigned grid = (unsigned)std::min<int64_t>((units + 1023) / 1024, 256);
#define FGPU_ENC(SS, F, RR)                                                                                   \
  if (S == SS && (fma_mode != 0) == F && rows == RR) {                                                        \
    FGPU_HIP(hipFuncSetAttribute((const void*)pq_encode_kernel<SS, F, RR>,                                    \
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                      \
    hipLaunchKernelGGL((pq_encode_kernel<SS, F, RR>), dim3(grid), dim3(1024), lds, s, x, n, dim, m, assign, cent, \
                       (uint32_t)ncent, codebook, pos, codes);                                                                 \
    FGPU_HIP(hipGetLastError());                                                                              \
    return FGPU_OK;                                                                                           \
  }
#define FGPU_ENC_S(SS) FGPU_ENC(SS, true, 1) FGPU_ENC(SS, true, 2) FGPU_ENC(SS, false, 1) FGPU_ENC(SS, false, 2)
  FGPU_ENC_S(1) FGPU_ENC_S(2) FGPU_ENC_S(3) FGPU_ENC_S(4) FGPU_ENC_S(6) FGPU_ENC_S(8) FGPU_ENC_S(16)
#undef FGPU_ENC_S
#undef FGPU_ENC
  return set_error(FGPU_ERR_UNSUPPORTED, "pq_encode: unsupported sub-dimension");
}

fgpu_status launch_pq_residuals(const float* x, int dim, const int32_t* rows, int nrows, const int32_t* assign,
                                const float* cent, int ncent, float* res, hipStream_t s) {
  return launch1d(pq_residuals_kernel, (int64_t)nrows * dim, 256, s, x, dim, rows, nrows, assign, cent, (uint32_t)ncent,
                  res);
}

fgpu_status launch_pq_init(const float* res, int nsample, int dim, int m, const int32_t* init_rows, float* codebook,
                           hipStream_t s) {
  (void)nsample;
  const int S = dim / m;
  return launch1d(pq_init_kernel, (int64_t)m * kPQK * S, 256, s, res, dim, m, S, init_rows, codebook);
}

// A subspace's assignments: ns bytes, rounded up to whole 16-byte loads.
static int pq_stride(int ns) { return (ns + 15) / 16 * 16; }
size_t pq_assign_bytes(int ns, int m) { return (size_t)pq_stride(ns) * m; }

// Workgroups of 256 threads up to which the E step takes one row a thread: three a
// CU run together.  Measured (us an iteration with its M step, two rows / one):
// 500 rows, 16 codes 37.5 / 25.6; 4000 rows, 48 codes 25.4 / 21.8 (768
// workgroups); 16000 rows, 16 codes 56.5 / 59.6 (1008).
constexpr int kEstepOneRow = 768;
fgpu_status launch_pq_estep(const float* res, int ns, int dim, int m, const float* codebook, uint8_t* assign_pq,
                            hipStream_t s) {
  const int S = dim / m;
  const int rows = (int64_t)((ns + 255) / 256) * m <= kEstepOneRow ? 1 : 2;
  const dim3 grid((unsigned)((ns + 256 * rows - 1) / (256 * rows)), (unsigned)m);
#define FGPU_EST(SS, RR)                                                                                      \
  if (S == SS && rows == RR) {                                                                                \
    hipLaunchKernelGGL((pq_estep_kernel<SS, RR>), grid, dim3(256), 0, s, res, ns, dim, m, codebook, assign_pq, \
                       pq_stride(ns));                                                                        \
    FGPU_HIP(hipGetLastError());                                                                              \
    return FGPU_OK;                                                                                           \
  }
  FGPU_EST(1, 1) FGPU_EST(2, 1) FGPU_EST(3, 1) FGPU_EST(4, 1) FGPU_EST(6, 1) FGPU_EST(8, 1) FGPU_EST(16, 1)
  FGPU_EST(1, 2) FGPU_EST(2, 2) FGPU_EST(3, 2) FGPU_EST(4, 2) FGPU_EST(6, 2) FGPU_EST(8, 2) FGPU_EST(16, 2)
#undef FGPU_EST
  return set_error(FGPU_ERR_UNSUPPORTED, "pq_estep: unsupported sub-dimension");
}

fgpu_status launch_pq_mstep(const float* res, int ns, int dim, int m, const uint8_t* assign_pq, float* codebook,
                            hipStream_t s) {
  const int S = dim / m;
#define FGPU_MST(SS)                                                                                                  \
  if (S == SS) {                                                                                                      \
    hipLaunchKernelGGL(pq_mstep_kernel<SS>, dim3(kPQK, (unsigned)m), dim3(kWave), 0, s, res, ns, dim, assign_pq,      \
                       pq_stride(ns), codebook);                                                                      \
    FGPU_HIP(hipGetLastError());                                                                                      \
    return FGPU_OK;                                                                                                   \
  }
  FGPU_MST(1) FGPU_MST(2) FGPU_MST(3) FGPU_MST(4) FGPU_MST(6) FGPU_MST(8) FGPU_MST(16)
#undef FGPU_MST
  return set_error(FGPU_ERR_UNSUPPORTED, "pq_mstep: unsupported sub-dimension");
}

size_t kmeans_pp_ws_bytes(int64_t n, int k) {
  const int64_t nb = (n + kPPBlock - 1) / kPPBlock;
  return carve_bytes<float>(n) + carve_bytes<uint64_t>(n) + carve_bytes<uint64_t>(nb) + carve_bytes<uint8_t>(n) +
         carve_bytes<int>(1) + carve_bytes<int32_t>(n) + carve_bytes<float>(k > 0 ? k : 1);
}

fgpu_status launch_kmeans_pp(const float* x, int64_t n, int dim, int k, uint64_t seed, float* cent, int32_t* rows,
                             void* ws, size_t ws_bytes, hipStream_t s) {
  Carve cv(ws, ws_bytes);
  float* d2 = cv.take<float>(n);
  uint64_t* w = cv.take<uint64_t>(n);
  const int nb = (int)((n + kPPBlock - 1) / kPPBlock);
  uint64_t* part = cv.take<uint64_t>(nb);
  uint8_t* chosen = cv.take<uint8_t>(n);
  int* shift = cv.take<int>(1);
  int32_t* asg = cv.take<int32_t>(n);
  float* cc = cv.take<float>(k > 0 ? k : 1);
  FGPU_CHECK(cv.ok(), FGPU_ERR_WORKSPACE, "kmeans++: workspace too small");
  FGPU_HIP(hipMemsetAsync(chosen, 0, n, s));
  hipLaunchKernelGGL(pp_first_kernel, dim3(1), dim3(1), 0, s, n, seed, rows, chosen);
  hipLaunchKernelGGL(pp_take_kernel, dim3(1), dim3(256), 0, s, x, dim, rows, 0, cent, chosen);
  FGPU_TRY(pp_update(x, n, dim, cent, 1, d2, nullptr, w, part, nb, asg, cc, 0, nullptr, chosen, s));  // asg := 0
  hipLaunchKernelGGL(pp_shift_kernel, dim3(1), dim3(1024), 0, s, d2, n, shift);
  FGPU_HIP(hipGetLastError());
  // weights for round 1 from the initial d2 (every row: no skip yet)
  FGPU_TRY(pp_update(x, n, dim, cent, 0, d2, shift, w, part, nb, nullptr, cc, 0, nullptr, chosen, s));
  for (int j = 1; j < k; ++j) {
    // the pick, the row as centre j and its distances to the earlier centres
    // (those only if a pass follows)
    const unsigned g = j + 1 < k ? (unsigned)((j + kPPBlock / kWave - 1) / (kPPBlock / kWave)) : 1u;
    hipLaunchKernelGGL(pp_pick_kernel, dim3(g), dim3(kPPBlock), 0, s, w, part, nb, n, seed, j, chosen, rows, x, dim, cent,
                       cc);
    if (j + 1 < k)
      FGPU_TRY(pp_update(x, n, dim, cent + (size_t)j * dim, 0, d2, shift, w, part, nb, asg, cc, j, rows + j, chosen, s));
  }
  FGPU_HIP(hipGetLastError());
  return FGPU_OK;
}


fgpu_status launch_list_radius(const float* codebook, int m, int sub, const uint8_t* codes, const int32_t* offsets,
                               int nlist, float* rmax, hipStream_t s) {
  if (nlist <= 0) return FGPU_OK;
  const size_t lds = (size_t)m * kPQK * sizeof(double);
  FGPU_CHECK(lds <= 128 * 1024, FGPU_ERR_UNSUPPORTED, "list_radius: pq_m too large");
  FGPU_HIP(hipFuncSetAttribute((const void*)list_radius_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(list_radius_kernel, dim3((unsigned)nlist), dim3(256), lds, s, codebook, m, sub, codes, offsets,
                     rmax);
  FGPU_HIP(hipGetLastError());
  return FGPU_OK;
}

}  // namespace fgpu
