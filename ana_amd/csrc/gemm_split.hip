// ANA_FAST_FP32 prefill products on the bf16 matrix cores (gfx950).
//
// Y[m][n] = sum_k A[m][k] W[n][k] in fp32 precision: every operand is the
// exact sum of three bf16 values (8 mantissa bits each, so 24 together), and
// a product of two fp32 values is the sum of the six products of their parts
// that matter, each exact in the matrix core's fp32 accumulation. The three
// left out (the second part times the third, twice, and the third times the
// third) are at most 2^-25 of the product, below the rounding of one fp32
// multiply. Six bf16 products cost 6/16 of the matrix-core time of one fp32
// product (v_mfma_f32_16x16x4f32 does 1/16 of v_mfma_f32_16x16x32_bf16's
// rate).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "ana_internal.h"
#include "mfma.h"
#include "wave.h"

namespace ana {

namespace {

// An operand in parts: 16 rows x 32 k make one block of three planes (the
// first parts, the second, the third), each 1 KB in the matrix core's lane
// order (lane l holds row l % 16 at k = 8 (l / 16) .. + 7), blocks ordered
// (row tile, k step): a tile's k range streams as consecutive 1 KB pieces
// and a fragment is one 16-byte LDS read a lane at 16 l, no bank conflicts.
constexpr uint32_t kBlk = 3 * 512;

// x as the sum of three bf16 values: the value rounded (clamped to bf16's
// largest finite one, as fp32's last binade rounds past it), the remainder
// rounded, the remainder of that (exact: 24 bits are 8 + 8 + 8). Infinities
// and NaN stay whole in the first part (their products are then infinite or
// NaN in the sum; an infinity can come out as NaN).
__device__ __forceinline__ void split3(float x, __bf16* a, __bf16* b, __bf16* c) {
  constexpr float M = 0x1.fep127f;
  const __bf16 h = (__bf16)__builtin_amdgcn_fmed3f(x, -M, M);
  const float r = x - (float)h;
  const __bf16 m = (__bf16)r;
  const __bf16 l = (__bf16)(r - (float)m);
  const bool fin = fabsf(x) < __builtin_inff();
  *a = fin ? h : (__bf16)x;
  *b = fin ? m : (__bf16)0.0f;
  *c = fin ? l : (__bf16)0.0f;
}

// The weights of a product in parts, times the norm's gains (each product
// rounded once, as the packed decode weights have them): 16-row tiles over
// the segments in turn, or with SiLU gate tile j then up tile j.
__global__ __launch_bounds__(256) void k_pack3(GemvArgs a, uint32_t nk, uint64_t pieces, uint4* __restrict__ dst) {
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < pieces; i += (uint64_t)gridDim.x * 256) {
    const uint32_t lane = (uint32_t)(i & 63), r = lane & 15;
    const uint64_t ts = i >> 6;
    const uint32_t s = (uint32_t)(ts % nk), t = (uint32_t)(ts / nk), k = 32 * s + 8 * (lane >> 4);
    const float* w;
    if (a.mode == GM_SILU) {
      w = ((t & 1) ? a.seg[1].W : a.seg[0].W) + (size_t)(16 * (t >> 1) + r) * a.K;
    } else {
      const uint32_t v = 16 * t + r;
      w = v < a.seg[0].rows ? a.seg[0].W + (size_t)v * a.K : a.seg[1].W + (size_t)(v - a.seg[0].rows) * a.K;
    }
    __bf16 p[3][8];
#pragma unroll
    for (int e = 0; e < 8; e++) split3(a.ng ? w[k + e] * a.ng[k + e] : w[k + e], &p[0][e], &p[1][e], &p[2][e]);
#pragma unroll
    for (int q = 0; q < 3; q++) dst[ts * 192 + q * 64 + lane] = *reinterpret_cast<const uint4*>(p[q]);
  }
}

// The activations of a product in parts, and with rsc each row's norm scale
// 1 / sqrt(sum x^2 / K + 1e-5): a workgroup a 16-row tile, its four waves
// taking the k steps in turn, a lane's eight values at a time. Bound by its
// traffic, 4 bytes a value read and 6 written. Rows past B are zero.
__global__ __launch_bounds__(256) void k_split3(const float* __restrict__ X, uint32_t ldx, uint32_t K, uint32_t B,
                                                 uint4* __restrict__ dst, float* __restrict__ rsc) {
  __shared__ float sums[4][16];
  const uint32_t lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nk = K / 32;
  const uint32_t m = 16 * blockIdx.x + (lane & 15);
  const float* x = X + (size_t)(m < B ? m : 0) * ldx + 8 * (lane >> 4);
  float ss = 0.0f;
  for (uint32_t s = wv; s < nk; s += 4) {
    float4 v[2] = {*reinterpret_cast<const float4*>(x + 32 * s), *reinterpret_cast<const float4*>(x + 32 * s + 4)};
    const float f[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
    __bf16 p[3][8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float y = m < B ? f[e] : 0.0f;
      ss = fmaf(y, y, ss);
      split3(y, &p[0][e], &p[1][e], &p[2][e]);
    }
#pragma unroll
    for (int q = 0; q < 3; q++)
      dst[((size_t)blockIdx.x * nk + s) * 192 + q * 64 + lane] = *reinterpret_cast<const uint4*>(p[q]);
  }
  if (!rsc) return;
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  if (lane < 16) sums[wv][lane] = ss;
  __syncthreads();
  if (threadIdx.x < 16 && m < B) {
    const float t = (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
    rsc[m] = 1.0f / sqrtf(t / (float)K + 1.0e-5f);
  }
}

struct X3Args {
  const __bf16 *A, *W;      // the operands in parts
  uint32_t nk, B, MT, NT;   // k steps, rows, 16-row tiles of each
  float *Y0, *Y1;           // output rows of the two segments (rows0 columns in the first)
  uint32_t ld0, ld1, rows0;
  const float* R;           // residual rows (nullptr: none)
  uint32_t ldr;
  const float* rsc;         // the rows' norm scales (nullptr: none)
  __bf16* H;                // SiLU: the hidden rows in parts
  uint32_t hk;              // and their k steps
};

// A (WM MJ 16)-row x (WN NI 16)-column tile of WM x WN waves, each MJ x NI
// 16 x 16 tiles. K goes in stages of 32 through two LDS objects (so the
// compiler sees that a stage's reads miss the loads in flight into the
// other), each filled one stage ahead by global_load_lds, 3 KB of a row tile
// at a time; a wave reads its tiles' parts (24 fragments of 1 KB at 4 x 4)
// and runs six matrix-core instructions a 16 x 16 tile, 96 for 24 KB of
// reads, the smallest products first. The weights are the left operand, so
// a lane's four results are four consecutive columns of one row: the
// outputs, the residuals and the hidden rows' parts move 16 (8) bytes a
// lane.
// With two waves a SIMD a stage is 3072 cycles of matrix-core time at 4 x 4
// against about 2400 to bring its 72 KB in and 2060 of LDS traffic, so the
// matrix cores bound it where the tiles fill the CUs. Measured at the 115M's
// shapes and 8192 rows, with k_gemm_big's fp32 matrix-core products before:
// q|k|v|z 388 -> 173 us, gate|up 519 -> 241 us, Wo and down 211 -> 93 us on
// average; the matrix cores busy 62% of the time (the clock at 2.1 GHz under
// this load), 1.28 PFLOP/s of bf16 products in gate|up.
template <int WM, int WN, int MJ, int NI, bool SILU>
__global__ __launch_bounds__(WM * WN * 64) void k_gemm_x3(X3Args a) {
  constexpr int NW = WM * WN, AT = WM * MJ, TT = AT + WN * NI, H = (TT + NW - 1) / NW;
  static_assert(!SILU || NI % 2 == 0, "gate and up tiles in pairs");
  __shared__ __align__(1024) __bf16 st0[TT * kBlk], st1[TT * kBlk];
  auto stage = [&](auto B) -> __bf16* {
    if constexpr (decltype(B)::value == 0) return st0;
    else return st1;
  };
  const uint32_t lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t wm = wv / WN, wn = wv % WN, r16 = lane & 15, g4 = lane >> 4;
  uint32_t ntile, mtile;
  xcd_tile(&ntile, &mtile);
  const uint32_t nt0 = ntile * (WN * NI), mt0 = mtile * AT;
  // the row tiles this wave brings in (tiles past the operand's end load its
  // last one; nothing reads their results)
  const __bf16* src[H];
#pragma unroll
  for (int h = 0; h < H; h++) {
    const uint32_t t = wv + NW * h;
    src[h] = t < (uint32_t)AT ? a.A + (size_t)min(mt0 + t, a.MT - 1) * a.nk * kBlk
                              : a.W + (size_t)min(nt0 + t - AT, a.NT - 1) * a.nk * kBlk;
  }
  auto issue = [&](uint32_t s, auto B) {
#pragma unroll
    for (int h = 0; h < H; h++) {
      const uint32_t t = wv + NW * h;
      if ((h + 1) * NW > TT && t >= (uint32_t)TT) break;
      const __bf16* p = src[h] + (size_t)s * kBlk + 8 * lane;
#pragma unroll
      for (int q = 0; q < 3; q++)
        __builtin_amdgcn_global_load_lds((const void*)(p + 512 * q), (lds_void*)(stage(B) + t * kBlk + 512 * q), 16, 0, 0);
    }
  };
  // the first parts' products in one sum, the five smaller ones (2^-8 of it
  // and less) in another: the large sum is then rounded once a stage
  f32x4_t acc[NI][MJ], low[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int j = 0; j < MJ; j++) acc[i][j] = low[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  // fragments of two parts at a time: the first parts' (fw0, fa0), and the
  // second's, then the third's, in the same registers (fw, fa)
  bf16x8_t fw0[NI], fa0[MJ], fw[NI], fa[MJ];
  auto read_w = [&](auto B, int q, bf16x8_t (&f)[NI]) {
    const __bf16* p = stage(B) + (AT + wn * NI) * kBlk + 8 * lane + 512 * q;
#pragma unroll
    for (int i = 0; i < NI; i++) f[i] = *reinterpret_cast<const bf16x8_t*>(p + i * kBlk);
  };
  auto read_a = [&](auto B, int q, bf16x8_t (&f)[MJ]) {
    const __bf16* p = stage(B) + wm * MJ * kBlk + 8 * lane + 512 * q;
#pragma unroll
    for (int j = 0; j < MJ; j++) f[j] = *reinterpret_cast<const bf16x8_t*>(p + j * kBlk);
  };
  auto term = [&](f32x4_t (&c)[NI][MJ], const bf16x8_t (&w)[NI], const bf16x8_t (&x)[MJ]) {
#pragma unroll
    for (int i = 0; i < NI; i++)
#pragma unroll
      for (int j = 0; j < MJ; j++) c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], x[j], c[i][j], 0, 0, 0);
  };
  auto keep = [&]() { __builtin_amdgcn_sched_barrier(0); };   // (nothing moved across)
  // a stage: every read goes out a product or more before its use, the
  // first ones before the last product of the stage before (held over the
  // barrier), so the matrix cores work while the reads land
  auto step = [&](uint32_t s, auto B, auto Bn, auto first) {
    // this wave's loads of stage s are done and so are its reads of the
    // other object; the barrier says so for every wave
    keep();
    asm volatile("" ::: "memory");
    ANA_LGKMCNT0();
    ANA_VMCNT(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    keep();
    if (s + 1 < a.nk) issue(s + 1, Bn);
    read_w(B, 1, fw);
    read_a(B, 1, fa);
    keep();
    if constexpr (!decltype(first)::value) term(acc, fw0, fa0);
    keep();
    read_a(B, 0, fa0);
    read_w(B, 0, fw0);
    keep();
    term(low, fw, fa);
    keep();
    term(low, fw, fa0);
    keep();
    read_w(B, 2, fw);
    keep();
    term(low, fw0, fa);
    keep();
    read_a(B, 2, fa);
    keep();
    term(low, fw, fa0);
    keep();
    term(low, fw0, fa);
    keep();
  };
  constexpr std::integral_constant<int, 0> S0{};
  constexpr std::integral_constant<int, 1> S1{};
  issue(0, S0);
  step(0, S0, S1, std::true_type{});
  for (uint32_t s = 1; s < a.nk; s += 2) {
    step(s, S1, S0, std::false_type{});
    if (s + 1 < a.nk) step(s + 1, S0, S1, std::false_type{});
  }
  term(acc, fw0, fa0);
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int j = 0; j < MJ; j++) acc[i][j] += low[i][j];
  // this lane's results: row (mt0 + wm MJ + j) 16 + r16, columns
  // (nt0 + wn NI + i) 16 + 4 g4 .. + 3
  const uint32_t mt = mt0 + wm * MJ, nt = nt0 + wn * NI;
  float sc[MJ];
#pragma unroll
  for (int j = 0; j < MJ; j++) sc[j] = a.rsc ? a.rsc[min((mt + j) * 16 + r16, a.B - 1)] : 1.0f;
  if constexpr (SILU) {
#pragma unroll
    for (int i = 0; i < NI; i += 2) {
      if (nt + i >= a.NT) continue;
      const uint32_t n = ((nt + i) >> 1) * 16 + 4 * g4;
      const uint32_t at = (n >> 5) * kBlk + (r16 + 16 * ((n & 31) >> 3)) * 8 + (n & 7);
#pragma unroll
      for (int j = 0; j < MJ; j++) {
        if (mt + j >= a.MT) continue;
        __bf16 p[3][4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float h = fast_silu(acc[i][j][r] * sc[j]) * (acc[i + 1][j][r] * sc[j]);
          split3(h, &p[0][r], &p[1][r], &p[2][r]);
        }
        __bf16* y = a.H + (size_t)(mt + j) * a.hk * kBlk + at;
#pragma unroll
        for (int q = 0; q < 3; q++) *reinterpret_cast<uint2*>(y + 512 * q) = *reinterpret_cast<const uint2*>(p[q]);
      }
    }
  } else {
    float4 res[NI][MJ];
    if (a.R) {
#pragma unroll
      for (int i = 0; i < NI; i++)
#pragma unroll
        for (int j = 0; j < MJ; j++)
          res[i][j] = *reinterpret_cast<const float4*>(a.R + (size_t)min((mt + j) * 16 + r16, a.B - 1) * a.ldr +
                                                       min(nt + i, a.NT - 1) * 16 + 4 * g4);
    }
#pragma unroll
    for (int i = 0; i < NI; i++) {
      if (nt + i >= a.NT) continue;
      const uint32_t n = (nt + i) * 16 + 4 * g4;
      const bool s1 = n >= a.rows0;
      float* const Y = s1 ? a.Y1 + (n - a.rows0) : a.Y0 + n;
      const uint32_t ld = s1 ? a.ld1 : a.ld0;
#pragma unroll
      for (int j = 0; j < MJ; j++) {
        const uint32_t m = (mt + j) * 16 + r16;
        if (m >= a.B) continue;
        float4 y = make_float4(acc[i][j][0] * sc[j], acc[i][j][1] * sc[j], acc[i][j][2] * sc[j], acc[i][j][3] * sc[j]);
        if (a.R) y = make_float4(res[i][j].x + y.x, res[i][j].y + y.y, res[i][j].z + y.z, res[i][j].w + y.w);
        *reinterpret_cast<float4*>(Y + (size_t)m * ld) = y;
      }
    }
  }
}

uint32_t w_rows(const GemvArgs& a) {
  return a.mode == GM_SILU ? 2 * a.seg[0].rows : a.seg[0].rows + (a.nseg > 1 ? a.seg[1].rows : 0);
}

// The tile for a product: the one whose workgroups finish first by what the
// shapes measured at K = 768 (us; every one grows with K alike). `per`
// workgroups share a CU: a full round of them takes `round`, a last round
// of one or two a CU part[1] or part[2]. So 96 columns where 128 leave a
// round part empty (Wo at 8192 rows: 192 workgroups of 256 x 128 on 256 CUs
// 62 us, 256 of 256 x 96 54 us), and 64 x 64 where the larger ones leave CUs
// idle (Wo at 1919 rows 43 us with 256 x 96, 31 with 128 x 128, 20 with
// 64 x 64; gate|up at 256 rows 48, 28 and 17).
struct Tile { uint32_t bm, bn, per; float round, part[3]; };
constexpr Tile kTiles[] = {{256, 128, 1, 57.0f, {}}, {256, 96, 1, 47.0f, {}}, {128, 128, 1, 33.0f, {}},
                           {64, 64, 3, 29.0f, {0.0f, 15.0f, 20.0f}}};

}  // namespace

int x3_tile(uint32_t B, uint32_t rows, bool silu, uint32_t cus) {
  int best = 0;
  float least = 0.0f;
  for (int t = 0; t < 4; t++) {
    const Tile& k = kTiles[t];
    if (silu && k.bn == 96) continue;
    const uint32_t wgs = (B + k.bm - 1) / k.bm * ((rows + k.bn - 1) / k.bn), w = (wgs + cus - 1) / cus;
    const float cost = (float)(w / k.per) * k.round + k.part[w % k.per];
    if (t == 0 || cost < least) {
      best = t;
      least = cost;
    }
  }
  return best;
}

bool x3_fits(const GemvArgs& a) {
  return a.K % 32 == 0 && a.seg[0].rows % 16 == 0 && (a.nseg < 2 || a.seg[1].rows % 16 == 0) &&
         (a.mode != GM_SILU || a.seg[0].rows % 32 == 0);
}

uint64_t x3_bytes(uint32_t rows, uint32_t K) { return (uint64_t)((rows + 15) / 16) * (K / 32) * kBlk * sizeof(__bf16); }

uint64_t x3_weight_bytes(const GemvArgs& a) { return x3_bytes(w_rows(a), a.K); }

hipError_t launch_pack3(const GemvArgs& a, void* dst, hipStream_t st) {
  if (!x3_fits(a)) return hipErrorInvalidValue;
  const uint64_t pieces = (uint64_t)(w_rows(a) / 16) * (a.K / 32) * 64;
  hipLaunchKernelGGL(k_pack3, dim3((uint32_t)std::min<uint64_t>((pieces + 255) / 256, 8192)), dim3(256), 0, st, a, a.K / 32,
                     pieces, static_cast<uint4*>(dst));
  return hipGetLastError();
}

hipError_t launch_split3(const float* X, uint32_t ldx, uint32_t K, uint32_t B, void* dst, float* rsc, hipStream_t st) {
  if (B == 0 || K % 32 || ldx % 4) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_split3, dim3((B + 15) / 16), dim3(256), 0, st, X, ldx, K, B, static_cast<uint4*>(dst), rsc);
  return hipGetLastError();
}

hipError_t launch_gemm_x3(const GemvArgs& g, const void* A, const void* W, const float* rsc, void* H, hipStream_t st) {
  const bool silu = g.mode == GM_SILU;
  if (!x3_fits(g) || g.B == 0 || g.amax || (g.ng && !rsc) || (silu && !H)) return hipErrorInvalidValue;
  if (!silu && (g.seg[0].ldy % 4 || (g.nseg > 1 && g.seg[1].ldy % 4) || (g.mode == GM_RESID && (g.ldr % 4 || g.nseg != 1))))
    return hipErrorInvalidValue;
  const uint32_t rows = w_rows(g);
  X3Args a{};
  a.A = static_cast<const __bf16*>(A);
  a.W = static_cast<const __bf16*>(W);
  a.nk = g.K / 32;
  a.B = g.B;
  a.MT = (g.B + 15) / 16;
  a.NT = rows / 16;
  a.Y0 = g.seg[0].Y; a.ld0 = g.seg[0].ldy; a.rows0 = g.seg[0].rows;
  if (g.nseg > 1) { a.Y1 = g.seg[1].Y; a.ld1 = g.seg[1].ldy; }
  if (g.mode == GM_RESID) { a.R = g.R; a.ldr = g.ldr; }
  a.rsc = g.ng ? rsc : nullptr;
  a.H = static_cast<__bf16*>(H);
  a.hk = silu ? g.seg[0].rows / 32 : 0;
  static const uint32_t cus = device_cus();
  const int t = x3_tile(g.B, rows, silu, cus);
  const dim3 grid((rows + kTiles[t].bn - 1) / kTiles[t].bn, (g.B + kTiles[t].bm - 1) / kTiles[t].bm);
#define L_(WM, WN, MJ, NI, S) hipLaunchKernelGGL((k_gemm_x3<WM, WN, MJ, NI, S>), grid, dim3(WM * WN * 64), 0, st, a)
  switch (t) {
    case 0: if (silu) L_(4, 2, 4, 4, true); else L_(4, 2, 4, 4, false); break;
    case 1: L_(4, 2, 4, 3, false); break;
    case 2: if (silu) L_(4, 2, 2, 4, true); else L_(4, 2, 2, 4, false); break;
    default: if (silu) L_(2, 2, 2, 2, true); else L_(2, 2, 2, 2, false); break;
  }
#undef L_
  return hipGetLastError();
}

}  // namespace ana
