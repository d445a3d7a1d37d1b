// knn.hip -- exact kNN of a query set over a large base (A18) on fp16 MFMA
// bounds.
//
// brute_force_search_kernel (tune_parameters.cu:49-96) inserts every exact
// distance into a per-thread top-k.  coarse.hip's form of it writes a matrix of
// fp32 estimates per 4096 base rows and reads it back.  Here no estimate is
// written: the base goes through the MFMA units once, each query keeps a short
// list of (row, estimate) candidates against a threshold that tightens as the
// base goes by, and only the candidates left at the end get the exact
// device-form distance, which alone decides ids, distances and order.
//
//   1. The base rows are taken in the order (a i + b) mod n, i = 0, 1, ..., with a
//      near n / golden ratio and prime to n: any range of i is a uniform sample of
//      the rows, whatever order the base is in.
//   2. Level 0: the estimates of the first kCap rows are every query's list.
//   3. After each level the list's k-th smallest estimate bounds, with the
//      margin below, the estimate of every row that can be in the top-k; the
//      entries above it are dropped and it becomes the next level's threshold.
//      Level l + 1 takes F times the rows so far, which adds about k (F - 1)
//      entries (times the margin's share), so that the list stays inside its
//      kCap slots.
//   4. The last lists (about 1.5 k entries) get exact distances; the k smallest
//      (distance, row) keys are the answer.
//   5. A query whose list overflows (many tied rows, or a margin as wide as the
//      distances) or whose norm is out of the scales (norms_in_range) gets every exact
//      distance.
//
// The estimate and its margin are assign.hip's, with the query as the row and
// bias 0: f = D + kappa + e, D the distance scaled by 2^(sx + sc), kappa one
// unknown constant a query with |kappa| <= s, |e| <= g sqrt(D) + hn.  If k rows
// have f <= fk, their D is at most (sqrt(fk + s + hn) + g)^2 = sd^2, and since
// the exact chain is within gamma(130) of D, a row of the top-k has
//     f <= fk + 2 (g sd + hn) + 2^-15 sd^2.
// The threshold T enters the MFMA sum through the query's constant, so a row
// passes when the sum is <= 0 (its rounding then runs over terms of at most
// 4.13 N: 160 u24 4.13 = 3.9e-5, hn takes 2^-14 N).  E_c is the largest rounding
// error of a base row at 11 significant bits, plus 2^-14 a coordinate for what
// fp16 flushes.
#include <algorithm>
#include <cmath>
#include <numeric>

#include "common.hpp"
#include "fp16_bounds.hpp"
#include "kernels.hpp"

namespace fgpu {
namespace {

constexpr int kQRows = 64;    // queries a wave: two MFMA row sets share each base fragment
constexpr int kQWaves = 8;    // waves a screen workgroup: 512 queries
constexpr int kQStage = 4;    // base tiles (of 32 rows) a stage
constexpr int kCap = 2048;    // list slots a query
constexpr int kStageBuf = 1024;  // a wave's staged entries (LDS): a row set's 32 x 32 tile always fits
constexpr int64_t kQueryBatch = 16384;
constexpr float kNever = 60000.0f;  // estimates of real rows stay below 2^15, the others' above 65504 - 2^15

struct KnnStat {  // of the base
  float n2;       // max ||c||^2
  float e;        // max rounding error norm at 11 significant bits
};
struct KnnQuery {  // of a query (the margin's terms)
  float g, hn, s;
  float thr;   // the level's threshold on f; -inf: the query takes every exact distance
  float kx;    // X^2 / u, f's constant
  float top;   // a threshold no real row's f exceeds
};

// Row of position i: (a i + b) mod n.
struct KnnOrder {
  uint64_t a, b, n;
};
__device__ __forceinline__ int order_row(KnnOrder o, int64_t i) { return (int)((o.a * (uint64_t)i + o.b) % o.n); }

// ---- the base's largest norm and rounding error: eight lanes a row -----------------
template <int D>
__global__ __launch_bounds__(256) void knn_stats_kernel(const float* __restrict__ c, int64_t n,
                                                        KnnStat* __restrict__ part) {
  const int lane = threadIdx.x & 63, sub = lane & 7, r8 = lane >> 3;
  float mn = 0.0f, me = 0.0f;
  for (int64_t r0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 8; r0 < n; r0 += (int64_t)gridDim.x * 32) {
    const int64_t r = min(r0 + r8, n - 1);
    float n2 = 0.0f, e2 = 0.0f;
#pragma unroll
    for (int l = 0; l < D / 32; ++l) {
      const float4 v = reinterpret_cast<const float4*>(c + r * D)[8 * l + sub];
      const float w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t u = __float_as_uint(w[i]);
        const float e = w[i] - __uint_as_float((u + 0xFFFu + ((u >> 13) & 1u)) & ~0x1FFFu);
        n2 = __builtin_fmaf(w[i], w[i], n2);
        e2 = __builtin_fmaf(e, e, e2);
      }
    }
#pragma unroll
    for (int m = 1; m < 8; m <<= 1) {
      n2 += __shfl_xor(n2, m, kWave);
      e2 += __shfl_xor(e2, m, kWave);
    }
    mn = fmaxf(mn, n2);  // passes over NaN
    me = fmaxf(me, e2);
  }
  __shared__ float sn[4], se[4];
  mn = wave_max_f(mn);
  me = wave_max_f(me);
  if (lane == 0) {
    sn[threadIdx.x >> 6] = mn;
    se[threadIdx.x >> 6] = me;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    part[blockIdx.x] = KnnStat{fmaxf(fmaxf(sn[0], sn[1]), fmaxf(sn[2], sn[3])),
                               fmaxf(fmaxf(se[0], se[1]), fmaxf(se[2], se[3]))};
}

__global__ __launch_bounds__(1024) void knn_stats_final_kernel(const KnnStat* __restrict__ part, int np,
                                                               KnnStat* __restrict__ out, int* __restrict__ ctr,
                                                               int nctr) {
  __shared__ float sn[16], se[16];
  float mn = 0.0f, me = 0.0f;
  for (int i = threadIdx.x; i < np; i += 1024) {
    mn = fmaxf(mn, part[i].n2);
    me = fmaxf(me, part[i].e);
  }
  for (int i = threadIdx.x; i < nctr; i += 1024) ctr[i] = 0;
  mn = wave_max_f(mn);
  me = wave_max_f(me);
  if ((threadIdx.x & 63) == 0) {
    sn[threadIdx.x >> 6] = mn;
    se[threadIdx.x >> 6] = me;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 16; ++i) {
      mn = fmaxf(mn, sn[i]);
      me = fmaxf(me, se[i]);
    }
    *out = KnnStat{mn, sqrtf(me) * 1.001f};
  }
}

// ---- queries: A fragments (tile of 32: fragment, lane) and margins, a wave a tile ----
template <int D>
__global__ __launch_bounds__(64) void knn_query_kernel(const float* __restrict__ x, int nq,
                                                       const KnnStat* __restrict__ stat, uint4* __restrict__ ablk,
                                                       KnnQuery* __restrict__ qc, int* __restrict__ cnt,
                                                       int* __restrict__ fcount, int* __restrict__ flist) {
  constexpr int NC = D / 16;
  const int lane = threadIdx.x, li = lane & 31, h = lane >> 5;
  const int q = 32 * blockIdx.x + li;
  const float cm = stat->n2;
  const int sc = column_scale(cm);
  const float* xr = x + (size_t)min(q, nq - 1) * D + 8 * h;
  float4 v[2 * NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    v[2 * k] = *reinterpret_cast<const float4*>(xr + 16 * k);
    v[2 * k + 1] = *reinterpret_cast<const float4*>(xr + 16 * k + 4);
  }
  float n2 = 0.0f;
#pragma unroll
  for (int k = 0; k < 2 * NC; ++k) n2 += v[k].x * v[k].x + v[k].y * v[k].y + v[k].z * v[k].z + v[k].w * v[k].w;
  n2 += __shfl_xor(n2, 32, kWave);
  const int sx = 13 - max(norm_exp(n2), norm_exp(cm)) - sc;  // X^2 / u and u C^2 below 2^13
  const bool ok = q < nq && norms_in_range(n2, cm) && sx - sc >= -14 && sx - sc <= 15 && sx >= -126 && sx <= 126;
  const float f = ok ? ldexpf(1.0f, sx) : 0.0f;
  float e2 = 0.0f;
  uint4* b = ablk + (size_t)blockIdx.x * (NC + 1) * kWave + lane;
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const float w[8] = {v[2 * k].x * f,     v[2 * k].y * f,     v[2 * k].z * f,     v[2 * k].w * f,
                        v[2 * k + 1].x * f, v[2 * k + 1].y * f, v[2 * k + 1].z * f, v[2 * k + 1].w * f};
    uint32_t p[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint16_t b0 = h_rn(-2.0f * w[2 * i]), b1 = h_rn(-2.0f * w[2 * i + 1]);
      const float e0 = -0.5f * h_float(b0) - w[2 * i], e1 = -0.5f * h_float(b1) - w[2 * i + 1];
      e2 += e0 * e0 + e1 * e1;
      p[i] = ok ? pack2(b0, b1) : 0u;
    }
    b[k * kWave] = make_uint4(p[0], p[1], p[2], p[3]);
  }
  e2 += __shfl_xor(e2, 32, kWave);
  const uint16_t ub = ok ? (uint16_t)((15 + sx - sc) << 10) : (uint16_t)0;  // u
  // the constant's parts (z, w) depend on the level's threshold: the screen adds them
  b[NC * kWave] = h ? make_uint4(0u, 0u, 0u, 0u) : make_uint4(pack2(ub, ub), pack2(ub, kHOne), 0u, 0u);
  if (h || q >= nq) return;
  const float u = ok ? h_float(ub) : 1.0f, su = sqrtf(u) * 1.001f;
  const float X = sqrtf(n2) * f * 1.001f, Ea = sqrtf(e2) * 1.001f + 0x1p-30f, C = sqrtf(cm) * ldexpf(1.001f, sc);
  const float ec = stat->e * ldexpf(1.001f, sc) + 0x1p-14f * sqrtf((float)D) * 1.001f;
  const float N = X * X / u + u * C * C;
  KnnQuery r;
  r.g = 2.002f * (Ea * 1.002f / su + ec * su);
  r.hn = 1.001f * (2.0f * Ea * ec + 0x1p-14f * N + 0x1p-13f * (1.0f + u));
  r.s = 2.002f * Ea * X / u + 0x1p-16f * N;  // 2^-16 N: the fp32 sum behind kx
  r.thr = ok ? 0.0f : -INFINITY;
  r.kx = ok ? ldexpf(n2, sx + sc) : 0.0f;
  r.top = 2.1f * N;
  qc[q] = r;
  cnt[q] = ok ? kCap : 0;  // level 0 fills every slot
  if (!ok) flist[atomicAdd(fcount, 1)] = q;
}

// ---- base tiles in MFMA operand order (positions i0 .. i0 + ncols - 1), 32 a wave -----
// Tile t, fragment c < D / 16: lane (li, h) holds dims 16 c + 8 h .. + 7 of the
// tile's row li; the last fragment is the extra block (h = 0: P's three parts, 0
// or 65504 for a row past the end or not finite, three ones).  Rows are read
// eight lanes a row (whole 128-byte lines), four rows a lane.
template <int D>
__global__ __launch_bounds__(256) void knn_base_kernel(const float* __restrict__ c, KnnOrder ord, int64_t i0, int ncols,
                                                       const KnnStat* __restrict__ stat, uint4* __restrict__ blk) {
  constexpr int NC = D / 16, L = D / 32;
  const int lane = threadIdx.x & 63, sub = lane & 7, r8 = lane >> 3;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (32 * t >= ncols) return;  // whole wave leaves
  const float f = ldexpf(1.0f, column_scale(stat->n2));
  const int col_l = 32 * t + (lane & 31);
  const int row_l = order_row(ord, i0 + min(col_l, ncols - 1));
  uint2 w[4][L];
  double n2[4], ce[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4* p = reinterpret_cast<const float4*>(c + (size_t)__shfl(row_l, 8 * i + r8, kWave) * D) + sub;
    float4 v[L];
#pragma unroll
    for (int l = 0; l < L; ++l) v[l] = p[8 * l];
    n2[i] = ce[i] = 0.0;
#pragma unroll
    for (int l = 0; l < L; ++l) {
      const float x[4] = {v[l].x * f, v[l].y * f, v[l].z * f, v[l].w * f};
      uint16_t hb[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        hb[e] = h_rn(x[e]);
        n2[i] += (double)x[e] * x[e];
        ce[i] += (double)x[e] * (h_val(hb[e]) - (double)x[e]);
      }
      w[i][l] = make_uint2(pack2(hb[0], hb[1]), pack2(hb[2], hb[3]));
    }
  }
  uint4* bt = blk + (size_t)t * (NC + 1) * kWave;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int m = 1; m < 8; m <<= 1) {
      n2[i] += __shfl_xor(n2[i], m, kWave);
      ce[i] += __shfl_xor(ce[i], m, kWave);
    }
    const int li = 8 * i + r8;
    const bool ok = 32 * t + li < ncols && n2[i] < 0x1p13;
#pragma unroll
    for (int l = 0; l < L; ++l) {
      uint4* d = bt + (2 * l + (sub >> 2)) * kWave + ((sub >> 1) & 1) * 32 + li;
      reinterpret_cast<uint2*>(d)[sub & 1] = ok ? w[i][l] : make_uint2(0u, 0u);
    }
    if (sub < 2) {
      uint16_t p1, p2, p3;
      split3<false>(ok ? n2[i] + 2.0 * ce[i] : 0.0, p1, p2, p3);
      bt[NC * kWave + sub * 32 + li] =
          sub ? make_uint4(0u, 0u, 0u, 0u)
              : make_uint4(ok ? pack2(p1, p2) : 0u, ok ? pack2(p3, 0u) : pack2(0u, kHBig), kOneOne, pack2(kHOne, 0u));
    }
  }
}

// ---- the screen ---------------------------------------------------------------------
struct KnnScreen {
  const uint4* ablk;
  const uint4* blk;
  const KnnQuery* qc;
  int nq, ntiles, per;  // base tiles of the launch, tiles a workgroup
  int ngroups, nchunks;
  int pos0;             // position of the launch's first base row
  uint2* cand;          // [nq][kCap] (position, f bits)
  int* cnt;             // [nq]
};

// A wave's staged entries to their queries' lists: counted per query in LDS,
// each query's slots reserved with one global atomic, then written (a list's
// order is free).  thr: the queries' thresholds, added back to the sums.
__device__ __forceinline__ void knn_flush(const KnnScreen& a, int q0, const uint2* wb, int* rcnt, const float* thr,
                                          int nb) {
  const int lane = threadIdx.x & 63;
  wave_lds_order();
  rcnt[lane] = 0;
  wave_lds_order();
  for (int i = lane; i < nb; i += kWave) atomicAdd(&rcnt[wb[i].x >> 26], 1);
  wave_lds_order();
  const int c = rcnt[lane];
  wave_lds_order();
  rcnt[lane] = c > 0 ? atomicAdd(&a.cnt[q0 + lane], c) : 0;  // the query's next slot
  wave_lds_order();
  for (int i = lane; i < nb; i += kWave) {
    const uint2 e = wb[i];
    const int row = (int)(e.x >> 26), slot = atomicAdd(&rcnt[row], 1);
    if (slot < kCap)
      a.cand[(size_t)(q0 + row) * kCap + slot] =
          make_uint2((uint32_t)a.pos0 + (e.x & 0x3FFFFFFu), __float_as_uint(__uint_as_float(e.y) + thr[row]));
  }
  wave_lds_order();
}

// One workgroup: 512 queries (a wave 64, their fragments in registers) against
// `per` base tiles, which pass through LDS as in assign.hip.  ALL (level 0): entry
// i of every list is position i.  Otherwise a tile's sums <= 0 are staged in the
// wave's LDS buffer.
// Workgroups go round-robin over the 8 XCDs; the query groups of one chunk of
// the base follow each other on one XCD and share its L2.
// What bounds it: the MFMA pipe; a tile is 2 (D / 16 + 1) MFMAs of 32 cycles against
// 32 VALU minima, and about 0.1 % of the pairs pass.  Measured, 10k queries x 1M
// rows x 128 dims, k = 100: 4.1 ms of screens (620 TFLOP/s; five levels) of 4.5 ms
// in all; the chunked estimates took 39.9 ms.
template <int D, bool ALL>
__device__ __forceinline__ void knn_stage(const uint4* __restrict__ cur, uint4* __restrict__ nxt,
                                          const uint4* __restrict__ src, int next_kb, int tile0, int nt,
                                          const f16x8 (&A)[2][D / 16 + 1], const KnnScreen& a, int q0, uint2* wb,
                                          int* rcnt, const float* thr, int& nb, int lane, int wave) {
  constexpr int NC = D / 16, kTileU4 = (NC + 1) * kWave;
  const int li = lane & 31, h = lane >> 5;
  for (int i = wave; i < next_kb; i += kQWaves)
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + i * kWave + lane),
                                     (__attribute__((address_space(3))) void*)(nxt + i * kWave), 16, 0, 0);
  const uint4* bt = cur + lane;
  uint4 b[NC + 1];
#pragma unroll
  for (int k = 0; k <= NC; ++k) b[k] = bt[k * kWave];
#pragma unroll 1
  for (int t = 0; t < nt; ++t) {
    f32x16 acc[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.0f;
#pragma unroll
    for (int k = 0; k <= NC; ++k) {
      const f16x8 bk = __builtin_bit_cast(f16x8, b[k]);
      acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[0][k], bk, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[1][k], bk, acc[1], 0, 0, 0);
    }
    bt += t + 1 < nt ? kTileU4 : 0;  // the last tile reloads itself
#pragma unroll
    for (int k = 0; k <= NC; ++k) b[k] = bt[k * kWave];
    const uint32_t col = (uint32_t)(32 * (tile0 + t) + li);
    // acc[s][r]: query 32 s + 8 (r / 4) + 4 h + r % 4 of the wave, base position `col`
    if constexpr (ALL) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int q = q0 + 32 * s + 8 * (r >> 2) + 4 * h + (r & 3);
          const float f = acc[s][r] < kNever ? acc[s][r] : INFINITY;
          if (q < a.nq) a.cand[(size_t)q * kCap + col] = make_uint2((uint32_t)a.pos0 + col, __float_as_uint(f));
        }
    } else {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        int mn = __float_as_int(acc[s][0]);  // <= 0: the bits as a signed int
#pragma unroll
        for (int r = 1; r < 16; ++r) mn = min(mn, __float_as_int(acc[s][r]));
        if (__ballot(mn <= 0)) {
          int total = 0;
#pragma unroll
          for (int r = 0; r < 16; ++r) total += __popcll(__ballot(__float_as_int(acc[s][r]) <= 0));
          if (nb + total > kStageBuf) {
            knn_flush(a, q0, wb, rcnt, thr, nb);
            nb = 0;
          }
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const bool pass = __float_as_int(acc[s][r]) <= 0;
            const uint64_t bm = __ballot(pass);
            if (bm) {
              const uint32_t row = (uint32_t)(32 * s + 8 * (r >> 2) + 4 * h + (r & 3));
              if (pass)
                wb[nb + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u))] =
                    make_uint2((row << 26) | col, __float_as_uint(acc[s][r]));
              nb += __popcll(bm);
            }
          }
        }
      }
    }
  }
}

template <int D, bool ALL>
__global__ __launch_bounds__(kQWaves * kWave, 2) void knn_screen_kernel(KnnScreen a) {
  constexpr int NC = D / 16;
  constexpr int kTileU4 = (NC + 1) * kWave;
  constexpr int kStageU4 = kQStage * kTileU4;
  __shared__ __align__(16) uint4 bs0[kStageU4];
  __shared__ __align__(16) uint4 bs1[kStageU4];
  __shared__ uint2 wb_s[ALL ? 1 : kQWaves][ALL ? 1 : kStageBuf];
  __shared__ int rcnt_s[kQWaves][kWave];
  __shared__ float thr_s[kQWaves][kWave];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, h = lane >> 5;
  const int i = (int)blockIdx.x >> 3, group = i % a.ngroups, chunk = (i / a.ngroups) * 8 + ((int)blockIdx.x & 7);
  if (chunk >= a.nchunks) return;
  const int t0 = chunk * a.per, ntiles = min(a.per, a.ntiles - t0), nst = (ntiles + kQStage - 1) / kQStage;
  const uint4* src = a.blk + (size_t)t0 * kTileU4;
  auto stage_kb = [&](int s) { return s < nst ? min(kQStage, ntiles - s * kQStage) * (NC + 1) : 0; };
  for (int k = wave; k < stage_kb(0); k += kQWaves)
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + k * kWave + lane),
                                     (__attribute__((address_space(3))) void*)(bs0 + k * kWave), 16, 0, 0);
  const int q0 = (group * kQWaves + wave) * kQRows;
  f16x8 A[2][NC + 1];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int q = q0 + 32 * s + li;
    const bool in = q0 + 32 * s < a.nq;  // the query tile exists
    const uint4* ab = a.ablk + (size_t)(in ? (q0 >> 5) + s : 0) * kTileU4 + lane;
#pragma unroll
    for (int k = 0; k < NC; ++k) A[s][k] = __builtin_bit_cast(f16x8, in ? ab[k * kWave] : make_uint4(0u, 0u, 0u, 0u));
    uint4 e = in ? ab[NC * kWave] : make_uint4(0u, 0u, 0u, 0u);
    // the constant kx - thr; a query that takes no rows (or none here): 65504
    const KnnQuery qc = a.qc[min(q, a.nq - 1)];
    const bool on = q < a.nq && qc.thr > -INFINITY;
    const float thr = on && !ALL ? qc.thr : 0.0f;
    uint16_t k1, k2, k3;
    split3<false>(on ? (double)qc.kx - (double)thr : 0.0, k1, k2, k3);
    e.z = h ? 0u : on ? pack2(k1, k2) : pack2(kHBig, 0u);
    e.w = h ? 0u : on ? pack2(k3, 0u) : 0u;
    A[s][NC] = __builtin_bit_cast(f16x8, e);
    if (h == 0) thr_s[wave][32 * s + li] = thr;
  }
  int nb = 0;  // staged entries
  uint2* wb = wb_s[ALL ? 0 : wave];
  for (int st = 0; st < nst; st += 2) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part of stage st
    __syncthreads();                                   // every part; stage st - 1 read by all
    knn_stage<D, ALL>(bs0, bs1, src + (size_t)(st + 1) * kStageU4, stage_kb(st + 1), t0 + st * kQStage,
                      min(kQStage, ntiles - st * kQStage), A, a, q0, wb, rcnt_s[wave], thr_s[wave], nb, lane, wave);
    if (st + 1 >= nst) break;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    knn_stage<D, ALL>(bs1, bs0, src + (size_t)(st + 2) * kStageU4, stage_kb(st + 2), t0 + (st + 1) * kQStage,
                      min(kQStage, ntiles - (st + 1) * kQStage), A, a, q0, wb, rcnt_s[wave], thr_s[wave], nb, lane,
                      wave);
  }
  if (!ALL && nb > 0) knn_flush(a, q0, wb, rcnt_s[wave], thr_s[wave], nb);
}

// ---- after a level: the k-th smallest estimate, the next threshold, the entries kept ----
// One wave a query, the list's estimates in registers; the k-th smallest is
// bisected from above (any value with at least k entries at or below it is a
// valid fk; 2^-12 of the list's range is far inside the margin).
__global__ __launch_bounds__(256) void knn_tighten_kernel(uint2* __restrict__ cand, int* __restrict__ cnt,
                                                          KnnQuery* __restrict__ qc, int nq, int k,
                                                          int* __restrict__ fcount, int* __restrict__ flist) {
  constexpr int R = kCap / kWave;
  const int lane = threadIdx.x & 63;
  const int q = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  if (q >= nq) return;
  const KnnQuery c = qc[q];
  if (!(c.thr > -INFINITY)) return;
  const int n = __builtin_amdgcn_readfirstlane(cnt[q]);
  uint2* l = cand + (size_t)q * kCap;
  if (n > kCap) {  // entries were lost: every exact distance for this query
    if (lane == 0) {
      qc[q].thr = -INFINITY;
      cnt[q] = 0;
      flist[atomicAdd(fcount, 1)] = q;
    }
    return;
  }
  uint2 e[R];
  uint32_t lo = 0xFFFFFFFFu, hi = 0u;
  int fin = 0;  // entries with a finite estimate
#pragma unroll
  for (int i = 0; i < R; ++i) {
    e[i] = make_uint2(0u, 0x7F800000u);
    if (64 * i < n) {
      if (64 * i + lane < n) e[i] = l[64 * i + lane];
      const bool f = __uint_as_float(e[i].y) < INFINITY;
      const uint32_t key = float_key(__uint_as_float(e[i].y));
      if (f) {
        lo = min(lo, key);
        hi = max(hi, key);
      }
      fin += __popcll(__ballot(f));
    }
  }
  float thr = c.top;
  if (fin >= k) {
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) {
      lo = min(lo, (uint32_t)shfl_xor_i((int)lo, m));
      hi = max(hi, (uint32_t)shfl_xor_i((int)hi, m));
    }
    const uint32_t stop = (hi - lo) >> 12;
    while (hi - lo > stop && hi > lo) {  // count(<= hi) >= k throughout
      const uint32_t mid = lo + ((hi - lo) >> 1);
      int m = 0;
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (64 * i < n) m += __popcll(__ballot(float_key(__uint_as_float(e[i].y)) <= mid));
      if (m >= k) hi = mid;
      else lo = mid + 1;
    }
    const float fk = key_float(hi);
    const float sd = sqrtf(fmaxf(fk + c.s + c.hn, 0.0f)) * 1.0001f + c.g;
    const float t = fk + 2.002f * (c.g * sd + c.hn) + 0x1.01p-15f * sd * sd;
    thr = fminf(t + fabsf(t) * 0x1p-20f, c.top);
  }
  int kept = 0;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (64 * i < n) {
      const bool f = __uint_as_float(e[i].y) <= thr;
      const uint64_t bm = __ballot(f);
      if (f)
        l[kept + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u))] =
            e[i];
      kept += __popcll(bm);
    }
  }
  if (lane == 0) {
    cnt[q] = kept;
    qc[q].thr = thr;
  }
}

// ---- exact distances --------------------------------------------------------------------
// The running top-k (k <= 128) as two sorted 64-key lists.
__device__ __forceinline__ void knn_merge(uint64_t& ak, uint64_t& bk, int k, uint64_t key) {  // key sorted
  if (k <= kWave) {
    wave_merge_sorted64_k(ak, key);
    return;
  }
  const uint64_t r = wave_reverse64(key);
  const bool low = r < ak;
  uint64_t h = low ? ak : r;
  ak = low ? r : ak;
  bitonic_pass_k<64>(ak, true);
  bitonic_pass_k<64>(h, true);
  wave_merge_sorted64_k(bk, h);
}
__device__ __forceinline__ void knn_write(uint64_t ak, uint64_t bk, int q, int k, int32_t* ids, float* d) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = lane + 64 * j;
    if (r < k) {
      const uint64_t key = j ? bk : ak;
      const bool pad = key_id(key) == kPadId;
      ids[(size_t)q * k + r] = pad ? -1 : key_id(key);
      d[(size_t)q * k + r] = pad ? FLT_MAX : key_dist(key);
    }
  }
}

// One wave a query: its list's rows, 64 at a time (read eight lanes a row).
template <int D>
__global__ __launch_bounds__(256) void knn_final_kernel(const float* __restrict__ x, const float* __restrict__ c,
                                                        KnnOrder ord, const uint2* __restrict__ cand,
                                                        const int* __restrict__ cnt, const KnnQuery* __restrict__ qc,
                                                        int nq, int k, int32_t* __restrict__ ids,
                                                        float* __restrict__ d) {
  __shared__ __align__(16) float tr_s[4][row_tr_floats()];
  __shared__ float qs_s[4][D];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int q = blockIdx.x * 4 + wave;
  if (q >= nq || !(qc[q].thr > -INFINITY)) return;  // whole wave leaves
  float* qs = qs_s[wave];
  for (int i = lane; i < D; i += kWave) qs[i] = x[(size_t)q * D + i];
  wave_lds_order();
  const int n = __builtin_amdgcn_readfirstlane(cnt[q]);
  uint64_t ak = kPadKey, bk = kPadKey;
  for (int b = 0; b < n; b += kWave) {
    const int row = order_row(ord, (int64_t)cand[(size_t)q * kCap + min(b + lane, n - 1)].x);
    const float dist = wave_rows_l2<D, kWave, 1>(c, row, qs, tr_s[wave]);
    uint64_t key = b + lane < n ? key_of(dist, row) : kPadKey;
    wave_sort64_k(key);
    knn_merge(ak, bk, k, key);
  }
  knn_write(ak, bk, q, k, ids, d);
}

// The listed queries against every base row: 16 queries a workgroup (one a
// wave), 64 base rows at a time in LDS, a lane a row.  With few queries the base
// is split over the workgroups and the last one of a query group merges.
constexpr int kBWaves = 16;
constexpr int kBGrid = 256;
constexpr int kBStride = 4;  // floats of padding a row: 16-byte reads down the rows spread over the banks
template <int D>
__global__ __launch_bounds__(kBWaves * kWave) void knn_brute_kernel(const float* __restrict__ x,
                                                                    const float* __restrict__ c, int64_t n, int k,
                                                                    const int* __restrict__ fcount,
                                                                    const int* __restrict__ flist, int nq,
                                                                    uint64_t* __restrict__ part, int* __restrict__ arr,
                                                                    int32_t* __restrict__ ids, float* __restrict__ d) {
  __shared__ __align__(16) float rs[kWave * (D + kBStride)];
  __shared__ __align__(16) float qs_s[kBWaves][D];
  __shared__ int s_last;
  const int count = min(*fcount, nq);
  if (count <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int groups = (count + kBWaves - 1) / kBWaves;
  const int S = max(1, kBGrid / groups);  // slices of the base; groups * S <= kBGrid unless S is 1
  const int64_t tiles = (n + kWave - 1) / kWave;
  for (int it = blockIdx.x; it < groups * S; it += gridDim.x) {
    const int g = it / S, sl = it % S;
    const int f = g * kBWaves + wave;
    const int q = f < count ? flist[f] : -1;
    const float* qs = qs_s[wave];
    for (int i = lane; i < D; i += kWave) qs_s[wave][i] = q >= 0 ? x[(size_t)q * D + i] : 0.0f;
    uint64_t ak = kPadKey, bk = kPadKey;
    for (int64_t t = tiles * sl / S; t < tiles * (sl + 1) / S; ++t) {
      __syncthreads();
      for (int i = tid; i < kWave * (D / 4); i += kBWaves * kWave) {
        const int r = i / (D / 4), w = i % (D / 4);
        const int64_t row = min(t * kWave + r, n - 1);
        *reinterpret_cast<float4*>(rs + r * (D + kBStride) + 4 * w) = reinterpret_cast<const float4*>(c + row * D)[w];
      }
      __syncthreads();
      float acc = 0.0f;
#pragma unroll 4
      for (int j = 0; j < D / 4; ++j) {
        const float4 v = *reinterpret_cast<const float4*>(rs + lane * (D + kBStride) + 4 * j);
        const float4 w = *reinterpret_cast<const float4*>(qs + 4 * j);
        float df = w.x - v.x;
        acc = __builtin_fmaf(df, df, acc);
        df = w.y - v.y;
        acc = __builtin_fmaf(df, df, acc);
        df = w.z - v.z;
        acc = __builtin_fmaf(df, df, acc);
        df = w.w - v.w;
        acc = __builtin_fmaf(df, df, acc);
      }
      const int64_t row = t * kWave + lane;
      uint64_t key = row < n ? key_of(acc, (int)row) : kPadKey;
      const uint64_t kth = k <= kWave ? readlane64(ak, k - 1) : readlane64(bk, k - kWave - 1);
      if (__ballot(key < kth)) {
        wave_sort64_k(key);
        knn_merge(ak, bk, k, key);
      }
    }
    if (S > 1) {
      uint64_t* p = part + ((size_t)it * kBWaves + wave) * 2 * kWave;
      p[lane] = ak;
      p[kWave + lane] = bk;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      __syncthreads();
      if (tid == 0) s_last = __hip_atomic_fetch_add(&arr[g], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == S - 1;
      __syncthreads();
      if (!s_last) continue;
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      for (int o = 0; o < S; ++o) {
        if (o == sl) continue;
        const uint64_t* po = part + ((size_t)(g * S + o) * kBWaves + wave) * 2 * kWave;
        const uint64_t ka = po[lane], kb = po[kWave + lane];
        knn_merge(ak, bk, k, ka);
        if (k > kWave) knn_merge(ak, bk, k, kb);
      }
    }
    if (q >= 0) knn_write(ak, bk, q, k, ids, d);
  }
}

constexpr int kStatGrid = 2048;

// The region's parts for a batch of nq queries; what is left holds base tiles.
struct KnnWs {
  KnnStat* part;
  KnnStat* stat;
  int* ctr;  // [1 + kBGrid]: listed queries, arrivals
  int* flist;
  int* cnt;
  KnnQuery* qc;
  uint4* ablk;
  uint2* cand;
  uint64_t* brute;
  uint4* blk;
  int64_t tiles;  // base tiles that fit
  bool carve(void* base, size_t bytes, int nq, int dim) {
    Carve cv(base, bytes);
    part = cv.take<KnnStat>(kStatGrid);
    stat = cv.take<KnnStat>(1);
    ctr = cv.take<int>(1 + kBGrid);
    flist = cv.take<int>((size_t)nq);
    cnt = cv.take<int>((size_t)nq);
    qc = cv.take<KnnQuery>((size_t)nq);
    ablk = cv.take<uint4>((size_t)((nq + 31) / 32) * (dim / 16 + 1) * kWave);
    cand = cv.take<uint2>((size_t)nq * kCap);
    brute = cv.take<uint64_t>((size_t)kBGrid * kBWaves * 2 * kWave);
    if (!cv.ok()) return false;
    blk = reinterpret_cast<uint4*>(cv.base + cv.used);
    tiles = (int64_t)((cv.cap - cv.used) / ((size_t)(dim / 16 + 1) * kWave * sizeof(uint4)));
    return true;
  }
};
// Base rows a launch takes at most (positions are 26 bits of a staged entry), and
// the workspace asked for holds.  Fewer rows a launch leave the screen's last
// workgroups alone more often.  Measured (us, 2^15 / 2^18 / 2^20 rows a launch, 1M
// rows): 128 dims, 1 query 618 / 476 / 437, 1000 queries 1015 / 797 / 690, 10k,
// k 100, 5771 / 4469 / 4343; 32 dims, 1 query 399 / 233 / 194.
constexpr int64_t kBaseRows = 1 << 20;
constexpr int64_t kMinTiles = 1024;  // base tiles the workspace has to hold

template <int D>
fgpu_status launch_knn_d(const float* x, int nq, const float* c, int64_t n, int k, KnnWs w, int32_t* ids, float* d,
                         hipStream_t s) {
  KnnOrder ord{0, 0, (uint64_t)n};
  ord.a = (uint64_t)((double)n * 0.6180339887498949) | 1u;
  while (std::gcd(ord.a, ord.n) != 1) ord.a += 2;
  ord.a %= ord.n;
  ord.b = ord.n / 3;
  hipLaunchKernelGGL(knn_stats_kernel<D>, dim3(kStatGrid), dim3(256), 0, s, c, n, w.part);
  hipLaunchKernelGGL(knn_stats_final_kernel, dim3(1), dim3(1024), 0, s, w.part, kStatGrid, w.stat, w.ctr, 1 + kBGrid);
  hipLaunchKernelGGL(knn_query_kernel<D>, dim3((unsigned)((nq + 31) / 32)), dim3(64), 0, s, x, nq, w.stat, w.ablk, w.qc,
                     w.cnt, w.ctr, w.flist);
  // Levels: kCap rows, then each F times the rows before it, F such that the
  // list's share of a level stays below about 900 of the kCap slots.
  const double F = std::min(64.0, std::max(2.0, 900.0 / (2.1 * k)));
  const int levels = std::max(1, (int)std::ceil(std::log((double)n / kCap) / std::log(F)));
  const int64_t span = std::min<int64_t>(kBaseRows, w.tiles * 32);
  int64_t done = 0;
  for (int lv = 0; lv <= levels; ++lv) {
    int64_t end = lv == 0 ? kCap : lv == levels ? n : (int64_t)(kCap * std::pow((double)n / kCap, (double)lv / levels));
    end = std::min(n, (end + 31) / 32 * 32);
    for (; done < end; done += std::min(span, end - done)) {
      const int nb = (int)std::min(span, end - done);
      KnnScreen a{w.ablk, w.blk, w.qc, nq, (nb + 31) / 32, 0, 0, 0, (int)done, w.cand, w.cnt};
      a.ngroups = (nq + kQWaves * kQRows - 1) / (kQWaves * kQRows);
      // About 12 workgroups a CU; at least a stage of tiles each, at most 128.
      a.per = (int)std::min<int64_t>(128, std::max<int64_t>(kQStage, (int64_t)a.ntiles * a.ngroups / (256 * 12)));
      a.nchunks = (a.ntiles + a.per - 1) / a.per;
      const dim3 grid((unsigned)(8 * a.ngroups * ((a.nchunks + 7) / 8)));
      hipLaunchKernelGGL(knn_base_kernel<D>, dim3((unsigned)((a.ntiles + 3) / 4)), dim3(256), 0, s, c, ord, done, nb,
                         w.stat, w.blk);
      if (lv == 0)
        hipLaunchKernelGGL((knn_screen_kernel<D, true>), grid, dim3(kQWaves * kWave), 0, s, a);
      else
        hipLaunchKernelGGL((knn_screen_kernel<D, false>), grid, dim3(kQWaves * kWave), 0, s, a);
    }
    hipLaunchKernelGGL(knn_tighten_kernel, dim3((unsigned)((nq + 3) / 4)), dim3(256), 0, s, w.cand, w.cnt, w.qc, nq, k,
                       w.ctr, w.flist);
  }
  hipLaunchKernelGGL(knn_final_kernel<D>, dim3((unsigned)((nq + 3) / 4)), dim3(256), 0, s, x, c, ord, w.cand, w.cnt,
                     w.qc, nq, k, ids, d);
  hipLaunchKernelGGL(knn_brute_kernel<D>, dim3(kBGrid), dim3(kBWaves * kWave), 0, s, x, c, n, k, w.ctr, w.flist, nq,
                     w.brute, w.ctr + 1, ids, d);
  FGPU_HIP(hipGetLastError());
  return FGPU_OK;
}

}  // namespace

size_t knn_screen_ws_bytes(int nq, int64_t n) {
  const int64_t q = std::min<int64_t>(nq, kQueryBatch);
  return carve_bytes<KnnStat>(kStatGrid) + carve_bytes<KnnStat>(1) + carve_bytes<int>(1 + kBGrid) +
         2 * carve_bytes<int>(q) + carve_bytes<KnnQuery>(q) + carve_bytes<uint4>((q + 31) / 32 * 9 * kWave) +
         carve_bytes<uint2>((size_t)q * kCap) + carve_bytes<uint64_t>((size_t)kBGrid * kBWaves * 2 * kWave) +
         (size_t)std::max<int64_t>(kMinTiles, (std::min<int64_t>(n, kBaseRows) + 31) / 32) * 9 * kWave * sizeof(uint4);
}

bool knn_screen_takes(const float* x, int nq, const float* c, int64_t n, int dim, size_t ws_bytes) {
  if (((uintptr_t)x & 15) || ((uintptr_t)c & 15) || n < kKnnScreenMinRows) return false;
  if (dim != 32 && dim != 64 && dim != 96 && dim != 128) return false;
  KnnWs w;
  return w.carve(nullptr, ws_bytes, (int)std::min<int64_t>(nq, kQueryBatch), dim) && w.tiles >= kMinTiles;
}

fgpu_status launch_knn_screen(const float* x, int nq, const float* c, int64_t n, int dim, int k, void* ws,
                              size_t ws_bytes, int32_t* ids, float* d, hipStream_t s) {
  for (int64_t b = 0; b < nq; b += kQueryBatch) {
    const int nb = (int)std::min<int64_t>(kQueryBatch, nq - b);
    KnnWs w;
    FGPU_CHECK(w.carve(ws, ws_bytes, nb, dim) && w.tiles >= kMinTiles, FGPU_ERR_WORKSPACE,
               "knn_exact: workspace too small");
    const float* xb = x + b * dim;
    int32_t* ib = ids + b * k;
    float* db = d + b * k;
    if (dim == 128) FGPU_TRY(launch_knn_d<128>(xb, nb, c, n, k, w, ib, db, s));
    else if (dim == 96) FGPU_TRY(launch_knn_d<96>(xb, nb, c, n, k, w, ib, db, s));
    else if (dim == 64) FGPU_TRY(launch_knn_d<64>(xb, nb, c, n, k, w, ib, db, s));
    else FGPU_TRY(launch_knn_d<32>(xb, nb, c, n, k, w, ib, db, s));
  }
  return FGPU_OK;
}

}  // namespace fgpu
