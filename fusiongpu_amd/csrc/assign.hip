// assign.hip -- the nearest column of every row by exact L2 (the k-means
// assignment, A13): one fp16 MFMA pass that keeps a few candidate columns a
// row in registers, then their exact distances.
//
// The reference ranks with a cuBLAS -2 X C^T GEMM plus norms and takes the
// argmin (kmeans_gpu.cuh:59-76, 197-229).  Here, as in coarse.hip, an estimate
// with a proven margin picks a superset of the nearest columns and the exact
// device-form distance (a sequential fused chain) decides, so ids and distances
// do not depend on the estimate's rounding.  Unlike coarse.hip no estimate is
// written to memory: with 4096 columns the fp16 estimate matrix of the
// two-kernel form is 8 GB a million rows, written and read back.
//
// The estimate.  With x~ = x 2^sx (sx per row) and c~ = c 2^sc (sc from max ||c||),
// u = 2^(sx - sc), X = ||x~||, C >= ||c~||, the scaled distance is
//     D_j = 2^(sx + sc) ||x - c_j||^2 = X^2 / u + u ||c~_j||^2 - 2 <x~, c~_j>,
// the scales such that X^2 / u and u C^2 stay below 2^13 and C <= 64.
// v_mfma_f32_32x32x16_f16 forms it from x' = x~ + da and c' = c~ + dc (fp16,
// nearest) and one extra K block of three-part fp16 splits: u times P_j =
// ||c~_j||^2 + 2 <c~_j, dc_j>, and the row's K = X^2 / u + bias; a column past the
// end gets 65504.  What it computes is then
//     f_j = D_j + (bias - 2 <da, x~> / u)
//           - 2 <da, c~_j - x~/u> - 2 <x~ - u c~_j, dc_j> - 2 <da, dc_j> + rounding:
// the first bracket is the same for all columns of a row, and since
// ||x~ - u c~_j||^2 = u D_j the rest is at most g sqrt(D_j) + hn with the measured
// E_a = ||da||, E_c = max ||dc_j||, N = X^2 / u + u C^2 >= 2 X C and
//     g = 2 (E_a / sqrt(u) + E_c sqrt(u)),
//     hn = 2 E_a E_c + 2^-15 N + 2^-13 (1 + u)
// (160 fp32 roundings over terms summing to at most 2.03 N: 1.94e-5 N; the
// splits' last parts).  The operands' errors thus count against the distance
// itself, not against the norms: near columns share them.  bias = 1.01 (2 E_a X /
// u + g^2 + 2 hn) keeps every f_j positive, so floats order as integers, and the
// column's tile number replaces the low 7 mantissa bits (2^-16 f_j).
// A column b that the exact chain (within gamma(130) < 2^-16 of the distance)
// can rank first against m, the smallest key's column, has D_b <= D_m (1 + 2^-15),
// so its key is at most
//     f_m (1 + 2^-16) + 2.001 (g sqrt(D_m) + hn) + 2^-15 D_m,
// with sqrt(D_m) <= sqrt(Y) + g, Y = f_m (1 + 2^-16) - (bias - 2 E_a X / u - hn).
// Rows or centroids outside the scales (norms_in_range; or not finite) get a NaN
// bound, which makes every column a candidate, and rows that are not finite -inf.
//
// Candidates.  A lane sees the columns of one class (column mod 32) and keeps
// the class's smallest key, whose low bits name the tile, and its second
// smallest.  A class whose smallest key passes gives that column; one whose
// second smallest passes too gives all its columns.  At most 32 entries a row,
// about 1.3 on mixture data.
#include "common.hpp"
#include "fp16_bounds.hpp"
#include "kernels.hpp"

namespace fgpu {
namespace {

constexpr int kARows = 64;                  // rows a wave: two MFMA row sets share each column fragment
constexpr int kAWaves = 8;                  // waves a workgroup (two a SIMD at 256 VGPRs)
constexpr int kAStage = 4;                  // column tiles (of 32) a stage
constexpr int kASlots = 32;                 // candidate entries a row (one a column class)
constexpr uint16_t kAClass = 0x8000u;       // entry: every column of the class

// Column tiles in MFMA operand order: tile t, fragment c < D / 16: lane (li, h)
// holds dims 16 c + 8 h .. + 7 of column 32 t + li; the last fragment is the
// extra block (h = 0: P's three parts, 0 or 65504 past the end, three ones).
// emax[t]: the tile's largest ||c' - c~||.
template <int D>
__global__ __launch_bounds__(64) void assign_prep_kernel(const float* __restrict__ c, int nc,
                                                         const float* __restrict__ cn_max, uint4* __restrict__ blk,
                                                         float* __restrict__ emax) {
  constexpr int NC = D / 16;
  const int lane = threadIdx.x, li = lane & 31, h = lane >> 5, t = blockIdx.x;
  const int col = 32 * t + li;
  const float f = ldexpf(1.0f, column_scale(*cn_max));
  uint4* b = blk + (size_t)t * (NC + 1) * kWave + lane;
  double n2 = 0.0, e2 = 0.0, ce = 0.0;
  uint4 w[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    uint16_t v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float t = col < nc ? c[(size_t)col * D + 16 * k + 8 * h + i] * f : 0.0f;
      v[i] = h_rn(t);
      const double e = h_val(v[i]) - (double)t;
      n2 += (double)t * t;
      e2 += e * e;
      ce += (double)t * e;
    }
    w[k] = make_uint4(pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7]));
  }
  n2 += __shfl_xor(n2, 32, kWave);
  e2 += __shfl_xor(e2, 32, kWave);
  ce += __shfl_xor(ce, 32, kWave);
  // A column that is not finite can win no row: it counts as one past the end
  // (max ||c||^2 passes over NaN; with an infinite one no margin is finite).
  const bool ok = col < nc && n2 < 0x1p13;
  uint16_t p1, p2, p3;
  split3<false>(ok ? n2 + 2.0 * ce : 0.0, p1, p2, p3);
#pragma unroll
  for (int k = 0; k < NC; ++k) b[k * kWave] = ok ? w[k] : make_uint4(0u, 0u, 0u, 0u);
  b[NC * kWave] = h ? make_uint4(0u, 0u, 0u, 0u)
                    : make_uint4(ok ? pack2(p1, p2) : 0u, ok ? pack2(p3, 0u) : pack2(0u, kHBig), kOneOne,
                                 pack2(kHOne, 0u));
  const float em = wave_max_f(ok ? f_above(sqrt(e2) * (1.0 + 0x1p-40)) : 0.0f);
  if (lane == 0) emax[t] = em;
}

// One stage of column tiles for a wave: the next stage's loads go out straight
// to LDS, then each tile's MFMAs and the insertion of its values into the
// lane's two smallest keys of each row.  A tile's fragments are read while the
// tile before it is inserted.  cur and nxt are different buffers, and __restrict__
// says so: otherwise the compiler waits for the loads into nxt before the first
// read of cur.
template <int D>
__device__ __forceinline__ void assign_stage(const uint4* __restrict__ cur, uint4* __restrict__ nxt,
                                             const uint4* __restrict__ src, int next_kb, int tile0, int nt,
                                             const f16x8 (&A)[2][D / 16 + 1], uint32_t (&m1)[2][16],
                                             float (&m2)[2][16], int lane, int wave) {
  constexpr int NC = D / 16, kTileU4 = (NC + 1) * kWave;
  for (int i = wave; i < next_kb; i += kAWaves)
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + i * kWave + lane),
                                     (__attribute__((address_space(3))) void*)(nxt + i * kWave), 16, 0, 0);
  uint32_t mask = ~0x7Fu;
  asm volatile("" : "+s"(mask));
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
    uint32_t tile = (uint32_t)(tile0 + t);
    asm volatile("" : "+v"(tile));  // in a vector register: one v_and_or_b32 a key
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t key = (__float_as_uint(acc[s][r]) & mask) | tile;
        m2[s][r] = __builtin_amdgcn_fmed3f(__uint_as_float(m1[s][r]), m2[s][r], __uint_as_float(key));
        m1[s][r] = min(m1[s][r], key);  // positive floats
      }
  }
}

// Each workgroup takes 512 rows: a wave keeps its 64 rows' fragments (two sets
// of 32) and its lanes' two smallest keys per row in registers while the
// column tiles pass through LDS (loaded straight into LDS, two buffers of four
// tiles taking turns), and at the end writes each row's candidate entries.
// What bounds it: the MFMA pipe, then VALU issue.  A tile of 32 columns is
// 2 (D / 16 + 1) MFMAs of 32 cycles (576 at D = 128) against 96 VALU
// instructions of 4 for the two smallest keys (insert the tile number, median,
// minimum), which the other wave of the SIMD overlaps.  Two row sets halve the
// LDS reads an MFMA needs.  Measured, 1M rows x 4096 columns x 128 dims: 1.13 ms
// = 930 TFLOP/s (1050 with the extra block; a large bf16 product reaches 1177 on
// the same card), the rescore 0.20 ms; one Lloyd step 10.4 -> 1.46 ms against the
// estimate + select pair (three bf16 products, 8 GB of estimates).
template <int D>
__global__ __launch_bounds__(kAWaves * kWave, 2) void assign_kernel(const float* __restrict__ x, int64_t n, int nc,
                                                                    const uint4* __restrict__ blk,
                                                                    const float* __restrict__ emax,
                                                                    const float* __restrict__ cn_max,
                                                                    uint16_t* __restrict__ cand,
                                                                    uint8_t* __restrict__ cnt) {
  constexpr int NC = D / 16;
  constexpr int kTileU4 = (NC + 1) * kWave;        // uint4 a tile
  constexpr int kStageU4 = kAStage * kTileU4;
  __shared__ __align__(16) uint4 bs0[kStageU4];
  __shared__ __align__(16) uint4 bs1[kStageU4];
  __shared__ float g_s[kAWaves][kARows], q_s[kAWaves][kARows], h_s[kAWaves][kARows];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, h = lane >> 5;
  const int ntiles = (nc + 31) / 32, nst = (ntiles + kAStage - 1) / kAStage;
  const int64_t row0 = (int64_t)blockIdx.x * (kAWaves * kARows) + wave * kARows;
  // KB of stage s (tiles are (NC + 1) KB each)
  auto stage_kb = [&](int s) { return s < nst ? min(kAStage, ntiles - s * kAStage) * (NC + 1) : 0; };
  for (int i = wave; i < stage_kb(0); i += kAWaves)
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(blk + i * kWave + lane),
                                     (__attribute__((address_space(3))) void*)(bs0 + i * kWave), 16, 0, 0);

  float ec = 0.0f;
  for (int t = lane; t < ntiles; t += kWave) ec = fmaxf(ec, emax[t]);
  ec = wave_max_f(ec);
  const float cm = *cn_max;
  const int sc = column_scale(cm), ce = norm_exp(cm);

  f16x8 A[2][NC + 1];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int64_t row = min(row0 + 32 * s + li, n - 1);
    const float* xr = x + row * D + 8 * h;
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
    const int sx = 13 - max(norm_exp(n2), ce) - sc;  // X^2 / u and u C^2 below 2^13
    const bool ok = norms_in_range(n2, cm) && sx - sc >= -14 && sx - sc <= 15 && sx >= -126 && sx <= 126;
    const float f = ok ? ldexpf(1.0f, sx) : 0.0f;
    float e2 = 0.0f;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const float w[8] = {v[2 * k].x * f,     v[2 * k].y * f,     v[2 * k].z * f,     v[2 * k].w * f,
                          v[2 * k + 1].x * f, v[2 * k + 1].y * f, v[2 * k + 1].z * f, v[2 * k + 1].w * f};
      uint32_t p[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // the operand is -2 x', and x' half of it, exactly
        const uint16_t b0 = h_rn(-2.0f * w[2 * i]), b1 = h_rn(-2.0f * w[2 * i + 1]);
        const float e0 = -0.5f * h_float(b0) - w[2 * i], e1 = -0.5f * h_float(b1) - w[2 * i + 1];
        e2 += e0 * e0 + e1 * e1;
        p[i] = ok ? pack2(b0, b1) : 0u;
      }
      A[s][k] = __builtin_bit_cast(f16x8, make_uint4(p[0], p[1], p[2], p[3]));
    }
    e2 += __shfl_xor(e2, 32, kWave);
    const uint16_t ub = ok ? (uint16_t)((15 + sx - sc) << 10) : (uint16_t)0;  // u
    const float u = ok ? h_float(ub) : 1.0f, su = sqrtf(u) * 1.001f;
    const float X = sqrtf(n2) * f * 1.001f, Ea = sqrtf(e2) * 1.001f + 0x1p-30f, C = sqrtf(cm) * ldexpf(1.001f, sc);
    const float N = X * X / u + u * C * C;
    const float g = 2.002f * (Ea * 1.002f / su + ec * su);
    const float hn = 1.001f * (2.0f * Ea * ec + 0x1p-15f * N + 0x1p-13f * (1.0f + u));
    const float shift = 2.002f * Ea * X / u, bias = 1.01f * (shift + g * g + 2.0f * hn);
    uint16_t k1, k2, k3;
    split3<true>(ok ? ldexp((double)n2, sx + sc) + (double)bias : 0.0, k1, k2, k3);
    A[s][NC] = __builtin_bit_cast(f16x8, h ? make_uint4(0u, 0u, 0u, 0u)
                                           : make_uint4(pack2(ub, ub), pack2(ub, kHOne), pack2(k1, k2), pack2(k3, 0u)));
    if (h == 0) {
      // f is 0 if not ok, and e2 then 0, or NaN if the row is not finite: no column is its nearest
      g_s[wave][32 * s + li] = ok ? g : e2 == 0.0f ? __builtin_nanf("") : 0.0f;
      q_s[wave][32 * s + li] = bias - shift - hn;
      h_s[wave][32 * s + li] = ok ? hn : -INFINITY;
    }
  }

  uint32_t m1[2][16];
  float m2[2][16];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      m1[s][r] = __float_as_uint(0x1p127f);
      m2[s][r] = 0x1p127f;
    }
  for (int st = 0; st < nst; st += 2) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part of stage st
    __syncthreads();                                   // every part; stage st - 1 read by all
    assign_stage<D>(bs0, bs1, blk + (size_t)(st + 1) * kStageU4, stage_kb(st + 1), st * kAStage,
                    min(kAStage, ntiles - st * kAStage), A, m1, m2, lane, wave);
    if (st + 1 >= nst) break;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    assign_stage<D>(bs1, bs0, blk + (size_t)(st + 2) * kStageU4, stage_kb(st + 2), (st + 1) * kAStage,
                    min(kAStage, ntiles - (st + 1) * kAStage), A, m1, m2, lane, wave);
  }

  // m1[s][r] of lane (li, h): row 32 s + 8 (r / 4) + 4 h + r % 4, column class li.
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      uint32_t v = m1[s][r];
      v = min(v, (uint32_t)xchg<1>((int)v));
      v = min(v, (uint32_t)xchg<2>((int)v));
      v = min(v, (uint32_t)xchg<4>((int)v));
      v = min(v, (uint32_t)xchg<8>((int)v));
      v = min(v, (uint32_t)xchg<16>((int)v));
      const int rl = 32 * s + 8 * (r >> 2) + 4 * h + (r & 3);
      const float g = g_s[wave][rl], fm = __uint_as_float(v) * (1.0f + 0x1.1p-16f);
      const float sd = sqrtf(fmaxf(fm - q_s[wave][rl], 0.0f)) * 1.0001f + g;
      const float thr = (fm + 2.002f * (g * sd + h_s[wave][rl]) + 0x1.01p-15f * sd * sd) * (1.0f + 0x1p-20f);
      const bool f = !(__uint_as_float(m1[s][r]) > thr);
      const uint64_t bm = __ballot(f);
      const uint32_t hm = h ? (uint32_t)(bm >> 32) : (uint32_t)bm;
      const int64_t row = row0 + rl;
      if (row < n) {
        if (f)
          cand[row * kASlots + __popc(hm & ((1u << li) - 1u))] =
              (uint16_t)(32 * (m1[s][r] & 0x7Fu) + li) | (!(m2[s][r] > thr) ? kAClass : (uint16_t)0);
        if (li == 0) cnt[row] = (uint8_t)__popc(hm);
      }
    }
}

// Exact squared L2 of 64 (row, column) pairs, one a lane: each 128-byte line
// of both rows is read eight lanes a row, subtracted there, and the differences
// change hands through LDS to the lane that owns the pair, which runs the
// sequential fused chain (wave_rows_l2's hand-over, with the subtraction
// before it: the same fl(x - c)).
template <int D>
__device__ __forceinline__ float wave_pairs_l2(const float* __restrict__ x, const float* __restrict__ c, int64_t xrow,
                                               int col, float* tr) {
  const int lane = lane_id(), sub = lane & 7, r8 = lane >> 3;
  const int xlo = (int)xrow, xhi = (int)(xrow >> 32);
  float acc = 0.0f;
#pragma unroll
  for (int l = 0; l < D / 32; ++l) {
    // The empty asm keeps a line's loads after the line before it: hoisted,
    // every line is live at once and spills.
    asm volatile("" : "+v"(col));
    float4 v[8], w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int src = 8 * i + r8;
      const int64_t xr = ((int64_t)__shfl(xhi, src, kWave) << 32) | (uint32_t)__shfl(xlo, src, kWave);
      const int cr = __shfl(col, src, kWave);
      v[i] = reinterpret_cast<const float4*>(x + xr * D)[8 * l + sub];
      w[i] = reinterpret_cast<const float4*>(c + (size_t)cr * D)[8 * l + sub];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      *reinterpret_cast<float4*>(tr + (8 * i + r8) * kRowTrStride + 4 * sub) =
          make_float4(v[i].x - w[i].x, v[i].y - w[i].y, v[i].z - w[i].z, v[i].w - w[i].w);
    wave_lds_order();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float4 d = *reinterpret_cast<const float4*>(tr + lane * kRowTrStride + 4 * j);
      acc = __builtin_fmaf(d.x, d.x, acc);
      acc = __builtin_fmaf(d.y, d.y, acc);
      acc = __builtin_fmaf(d.z, d.z, acc);
      acc = __builtin_fmaf(d.w, d.w, acc);
    }
    asm volatile("" : "+v"(acc));
    wave_lds_order();
  }
  return acc;
}

// Every column's exact distance for the wave's 64 rows, a lane a row: each lane's
// smallest (distance, column) key, kNoKey if every distance is NaN.  A column's
// values are the same for the whole wave and come through scalar loads; the row is
// read once every kDenseCols columns.  VALU bounds it: 84 G pairs of 128 dims a
// second (200,000 rows x 1024 columns 2.43 ms), pair by pair about 20 G.
constexpr uint64_t kNoKey = ((uint64_t)0x7F800000u << 32) | (uint32_t)kPadId;  // above every key that is not NaN
constexpr int kDenseCols = 16;
template <int D>
__device__ __forceinline__ uint64_t wave_all_columns(const float* __restrict__ xr, const float* __restrict__ c, int nc) {
  uint64_t best = kNoKey;
#pragma unroll 1
  for (int c0 = 0; c0 < nc; c0 += kDenseCols) {
    float acc[kDenseCols];
#pragma unroll
    for (int j = 0; j < kDenseCols; ++j) acc[j] = 0.0f;
#pragma unroll 1
    for (int l = 0; l < D / 32; ++l) {
      float4 v[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) v[t] = reinterpret_cast<const float4*>(xr)[8 * l + t];
#pragma unroll
      for (int j = 0; j < kDenseCols; ++j) {
        const float4* cr = reinterpret_cast<const float4*>(c + (size_t)min(c0 + j, nc - 1) * D + 32 * l);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
          const float4 w = cr[t];
          float df = v[t].x - w.x;
          acc[j] = __builtin_fmaf(df, df, acc[j]);
          df = v[t].y - w.y;
          acc[j] = __builtin_fmaf(df, df, acc[j]);
          df = v[t].z - w.z;
          acc[j] = __builtin_fmaf(df, df, acc[j]);
          df = v[t].w - w.w;
          acc[j] = __builtin_fmaf(df, df, acc[j]);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kDenseCols; ++j) {
      const uint64_t key = key_of(acc[j], c0 + j);
      best = c0 + j < nc && key < best ? key : best;
    }
  }
  return best;
}

// The candidates' exact distances: a wave takes 64 rows, packs their candidate
// columns 64 at a time and keeps each row's smallest (distance, column) key.
// A row all of whose distances overflow has its first column, at distance inf; one
// that is not finite itself (no candidates) has none (kPadKey).
// Where the wave's entries name more than a kDenseShare-th of its pairs (data whose
// common offset is far larger than its differences, equal columns) every pair is
// computed instead: 200,000 rows x 1024 columns 20 -> 2.4 ms, 50,000 x 4096 (one
// wave a SIMD) 26 -> 9.4, both 11.2 with the estimate + select pair.  (Both forms
// cost the same near a quarter of the pairs with many waves, later with one a SIMD.)
// The lambdas are always_inline: left to the compiler, what they capture lay in
// scratch memory and each batch waited for it, 384 us against 201 (1M rows x 4096
// columns, 128 dims).
constexpr int kRWaves = 4;
constexpr int kDenseShare = 3;
template <int D>
__global__ __launch_bounds__(kRWaves * kWave, 4) void assign_rescore_kernel(
    const float* __restrict__ x, int64_t n, const float* __restrict__ c, int nc, const uint16_t* __restrict__ cand,
    const uint8_t* __restrict__ cnt, int32_t* __restrict__ ids, float* __restrict__ dist) {
  __shared__ __align__(16) float tr_s[kRWaves][row_tr_floats()];
  __shared__ unsigned long long best_s[kRWaves][kWave];
  __shared__ uint32_t q_s[kRWaves][2 * kWave];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row0 = ((int64_t)blockIdx.x * kRWaves + wave) * kWave;
  if (row0 >= n) return;  // whole wave leaves; no workgroup barrier follows
  float* tr = tr_s[wave];
  unsigned long long* best = best_s[wave];
  uint32_t* q = q_s[wave];  // row << 16 | column
  const int64_t row = row0 + lane;
  int ncand = row < n ? (int)cnt[row] : 0;
  best[lane] = kNoKey;
  int nq = 0;
  auto score = [&](int m) __attribute__((always_inline)) {
    wave_lds_order();
    const uint32_t e = q[lane < m ? lane : 0];
    const int rl = (int)(e >> 16), col = (int)(e & 0xFFFFu);
    const float d = wave_pairs_l2<D>(x, c, row0 + rl, col, tr);
    if (lane < m) atomicMin(&best[rl], (unsigned long long)key_of(d, col));
    wave_lds_order();
  };
  // Append a column for each lane with `f`; a full wave of them is scored.
  auto push = [&](bool f, uint32_t e) __attribute__((always_inline)) {
    const uint64_t bm = __ballot(f);
    if (f) q[nq + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u))] = e;
    nq += __popcll(bm);
    if (nq >= kWave) {
      score(kWave);
      const uint32_t m = q[kWave + lane];
      wave_lds_order();
      q[lane] = m;
      nq -= kWave;
    }
  };
  // Counted only where a third of the rows have candidates in half the classes.
  if (__builtin_expect(__popcll(__ballot(ncand >= kASlots / 2)) * kDenseShare >= kWave, 0)) {
    int cols = 0;
    for (int s = 0; s < ncand; ++s) cols += cand[row * kASlots + s] & kAClass ? (nc + 31) / 32 : 1;
    if (wave_sum_i(cols) * kDenseShare > nc * kWave) {
      const uint64_t b = wave_all_columns<D>(x + min(row, n - 1) * D, c, nc);
      if (ncand > 0) best[lane] = b;
      ncand = 0;
    }
  }
  for (int s = 0; __ballot(s < ncand); ++s) {
    const uint32_t e = s < ncand ? cand[row * kASlots + s] : 0u;
    const bool cls = s < ncand && (e & kAClass);
    const int col = (int)(e & (kAClass - 1u));
    push(s < ncand && !cls && col < nc, ((uint32_t)lane << 16) | (uint32_t)col);
    uint64_t m = __ballot(cls);
    while (m) {
      const int b = __builtin_ctzll(m);
      m &= m - 1;
      const int li = __builtin_amdgcn_readlane((int)e, b) & 31;
      for (int t0 = 0; t0 * 32 < nc; t0 += kWave) {
        const int cc = 32 * (t0 + lane) + li;
        push(cc < nc, ((uint32_t)b << 16) | (uint32_t)cc);
      }
    }
  }
  if (nq > 0) score(nq);
  if (row < n) {
    const uint64_t b = best[lane], k = b == kNoKey ? kPadKey : b;
    ids[row] = key_id(k);
    dist[row] = key_dist(k);
  }
}

template <int D>
fgpu_status launch_assign_d(const float* x, int64_t n, const float* c, int nc, const float* cn_max, void* ws,
                            size_t ws_bytes, int32_t* ids, float* d, hipStream_t s) {
  const int ntiles = (nc + 31) / 32;
  Carve cv(ws, ws_bytes);
  uint4* blk = cv.take<uint4>((size_t)ntiles * (D / 16 + 1) * kWave);
  float* emax = cv.take<float>(ntiles);
  FGPU_CHECK(cv.ok(), FGPU_ERR_WORKSPACE, "assign: workspace too small");
  constexpr int kRowBytes = kASlots * (int)sizeof(uint16_t) + 1;
  constexpr int64_t kGroup = kAWaves * kARows;
  const int64_t fit = (int64_t)((ws_bytes - cv.used) / kRowBytes) - 512;  // 512: the two arrays' alignment
  const int64_t rows = std::min<int64_t>(fit / kGroup * kGroup, (n + kGroup - 1) / kGroup * kGroup);
  FGPU_CHECK(rows >= kGroup, FGPU_ERR_WORKSPACE, "assign: workspace too small");
  uint16_t* cand = cv.take<uint16_t>((size_t)rows * kASlots);
  uint8_t* cnt = cv.take<uint8_t>((size_t)rows);
  FGPU_CHECK(cv.ok(), FGPU_ERR_WORKSPACE, "assign: workspace too small");
  hipLaunchKernelGGL(assign_prep_kernel<D>, dim3((unsigned)ntiles), dim3(kWave), 0, s, c, nc, cn_max, blk, emax);
  for (int64_t b = 0; b < n; b += rows) {
    const int64_t nb = std::min<int64_t>(rows, n - b);
    hipLaunchKernelGGL(assign_kernel<D>, dim3((unsigned)((nb + kGroup - 1) / kGroup)), dim3(kAWaves * kWave), 0, s,
                       x + b * D, nb, nc, blk, emax, cn_max, cand, cnt);
    hipLaunchKernelGGL(assign_rescore_kernel<D>, dim3((unsigned)((nb + kRWaves * kWave - 1) / (kRWaves * kWave))),
                       dim3(kRWaves * kWave), 0, s, x + b * D, nb, c, nc, cand, cnt, ids + b, d + b);
  }
  FGPU_HIP(hipGetLastError());
  return FGPU_OK;
}

}  // namespace

bool assign_takes(const float* x, int64_t n, const float* c, int nc, int dim, size_t ws_bytes) {
  if (((uintptr_t)x & 15) || ((uintptr_t)c & 15) || nc < kAssignMinCols || nc > kAssignMaxCols ||
      n < kAssignMinRows)
    return false;
  if (dim != 32 && dim != 64 && dim != 96 && dim != 128) return false;
  const int64_t tiles = (nc + 31) / 32;
  const int64_t need = tiles * (dim / 16 + 1) * 1024 + tiles * 4 + 65 * 1024 + 4096;  // 512 rows and alignment
  return (int64_t)ws_bytes >= need;
}

fgpu_status launch_assign(const float* x, int64_t n, const float* c, int nc, int dim, const float* cn_max, void* ws,
                          size_t ws_bytes, int32_t* ids, float* d, hipStream_t s) {
  if (dim == 128) return launch_assign_d<128>(x, n, c, nc, cn_max, ws, ws_bytes, ids, d, s);
  if (dim == 96) return launch_assign_d<96>(x, n, c, nc, cn_max, ws, ws_bytes, ids, d, s);
  if (dim == 64) return launch_assign_d<64>(x, n, c, nc, cn_max, ws, ws_bytes, ids, d, s);
  if (dim == 32) return launch_assign_d<32>(x, n, c, nc, cn_max, ws, ws_bytes, ids, d, s);
  return set_error(FGPU_ERR_UNSUPPORTED, "assign: dim must be 32, 64, 96 or 128");
}

}  // namespace fgpu
