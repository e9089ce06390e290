// The fast modes' products over packed weights (gfx950): decode batches of
// 5 .. 1023 rows (kPwMaxB) and prefill steps of 5 .. 127.
#include <hip/hip_runtime.h>

#include "ana_internal.h"
#include "mfma.h"

namespace ana {

// ------------------------------------------------------------------ packed weights

// A product's weights re-laid for the decode-batch GEMM (k_gemm_pw): tile t
// (16 weight rows in Segs order, 8 gate + 8 up rows with SiLU) and step s
// (32 k) form one block, blocks ordered (t, s), so a wave streams its k range
// of a tile as consecutive 1 KB pieces. In a block, lane l of a wave owns
// weight row l % 16 at k = 32 s + 8 (l / 16) .. + 7: fp32 (2 KB) as two 1 KB
// halves, half h holding k + 4 h .. + 3 of every lane at 16 l; bf16 (1 KB)
// the lane's eight values at 16 l. Rows past the segments are zero. With
// `ng` (the product's RMSNorm gains) each weight is stored as g[k] * W[n][k]
// (then rounded to bf16, nearest even, in the bf16 form), so the product
// needs only the raw x and its rows' norm scales.
__global__ void k_pack(GemvArgs a, uint32_t tiles, uint4* __restrict__ dst, int bf) {
  const Segs sgs(a);
  const uint32_t K = a.K, nsa = K >> 5;
  const uint64_t n = (uint64_t)tiles * nsa * (bf ? 64 : 128);
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t lane = (uint32_t)(i & 63);
    const uint32_t h = bf ? 0u : (uint32_t)((i >> 6) & 1);
    const uint64_t ts = bf ? i >> 6 : i >> 7;
    const uint32_t s = (uint32_t)(ts % nsa), t = (uint32_t)(ts / nsa);
    const float* w;
    uint32_t sg, lr;
    const bool ok = sgs.row(16, t, lane & 15, &w, &sg, &lr);
    const uint32_t k = 32 * s + 8 * (lane >> 4) + 4 * h;
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const uint32_t ke = k + (bf || e < 4 ? e : 0);
      x[e] = ok ? w[ke] * (a.ng ? a.ng[ke] : 1.0f) : 0.0f;
    }
    uint4 v;
    if (bf) {
      uint32_t b[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const uint32_t u = __float_as_uint(x[e]);
        b[e] = (u & 0x7fffffffu) > 0x7f800000u ? ((u >> 16) | 0x40u) : ((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
      }
      v = make_uint4(b[0] | (b[1] << 16), b[2] | (b[3] << 16), b[4] | (b[5] << 16), b[6] | (b[7] << 16));
    } else {
      v = make_uint4(__float_as_uint(x[0]), __float_as_uint(x[1]), __float_as_uint(x[2]), __float_as_uint(x[3]));
    }
    dst[i] = v;
  }
}

uint64_t pack_bytes(const GemvArgs& a, int bf) {
  return (uint64_t)pk_tiles(a) * (a.K / 32) * (bf ? 1024 : 2048);
}

hipError_t launch_pack(const GemvArgs& a, void* dst, int bf, hipStream_t st) {
  if (a.K % 32) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_pack, dim3(2048), dim3(256), 0, st, a, pk_tiles(a), static_cast<uint4*>(dst), bf);
  return hipGetLastError();
}

// Decode batches of 5..1023 rows and prefill steps of 5..127 in the fast modes:
// Y[m][n] = sum_k X[m][k] W[n][k] over packed weights (the norm gains folded
// in when `ng` is set). A workgroup owns NT 16-row weight tiles and 16 batch
// rows (each x fragment serves the NT tiles); K = 128 NS, and its four
// waves take a quarter of K each (NS steps of 32 k), every wave on its own.
// Per step a wave issues its weight pieces (coalesced 1 KB loads into a ring
// of D register sets) and two global_load_lds_dwordx4 of the 16 rows' x for that step (each 1 KB: 8 rows
// x 128 bytes, a row's 16-byte units at unit ^ (row & 7), so the fragment
// reads of 16 rows at one k fall in distinct bank groups) into an LDS block
// of its own. Its loads retire in issue order: before step s it waits until
// only the ops of steps s + 1 .. s + D - 1 are outstanding (a count fixed at
// compile time) and reads the step's x with no barrier. MFMA operands: lane
// l holds row l % 16 of x and of the tile at k = 8 (l / 16) + e of the step;
// fp32 (WT 0) takes v_mfma_f32_16x16x4f32 once per e, bf16 (WT 1) one
// v_mfma_f32_16x16x32_bf16 on x rounded to bf16. With `ng`
// each wave also sums its rows' x^2 from the same fragments. The waves'
// partial tiles and sums meet in LDS, where wave w adds result row r = w of
// every lane's four in wave order and applies the norm scale 1/sqrt(ss/K + 1e-5) and the epilogue (plain,
// residual, SiLU with tile rows 0..7 gate j and 8..15 up j): with all of it
// left to wave 0 a launch took 0.5 us more on average (B = 64, in a chain of
// a layer's four products: fp32 8.68 -> 8.14 us a product, bf16 6.70 ->
// 6.20). The result tile: lane l holds batch rows 4 (l / 16) + r, weight row
// l % 16. Bound by each wave's serial steps, not by bytes: tiles of 32 batch
// rows (two thirds of the traffic), four weight tiles, or eight waves a
// workgroup were all slower at B = 64 (chains of 9.1 to 13.5 us fp32).
template <int WT, int NS, int D, int NT>
__global__ __launch_bounds__(256) void k_gemm_pw(GemvArgs a, const uint4* __restrict__ pk, uint32_t tiles) {
  constexpr int WP = WT == 1 ? 1 : 2, OPS = NT * WP + 2;
  __shared__ __align__(1024) float xs[4][NS][512];
  __shared__ float red[4][NT][4][64];
  __shared__ float ssr[4][16];
  const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r16 = lane & 15, g4 = lane >> 4;
  const uint32_t K = 128 * NS, nsa = 4 * NS;
  const uint32_t m0 = blockIdx.y * 16;
  const bool norm = a.ng != nullptr;
  // the workgroup's tiles NT x .. NT x + NT - 1; one past the last reads the
  // last tile again and stores nothing
  const uint4* wsrc[NT];
#pragma unroll
  for (int j = 0; j < NT; j++)
    wsrc[j] = pk + ((size_t)min(NT * blockIdx.x + j, tiles - 1) * nsa + wv * NS) * (64 * WP) + lane;
  // this lane's x piece in each half of a step: row 8 h + (lane >> 3), its
  // unit (lane & 7) ^ row
  const uint32_t dr = lane >> 3, sl = (lane & 7) ^ dr;
  uint32_t xo[2];
#pragma unroll
  for (int h = 0; h < 2; h++) xo[h] = min(m0 + 8 * h + dr, a.B - 1) * a.ldx + wv * (K / 4) + 4 * sl;
  // the residuals of this wave's share of the epilogue first: they depend on
  // nothing, and loaded after the stores each would wait on the one before
  const Segs sgs(a);
  const uint32_t m = m0 + 4 * g4 + wv;
  float res[NT];
#pragma unroll
  for (int j = 0; j < NT; j++) {
    const uint32_t t = NT * blockIdx.x + j;
    const float* w_;
    uint32_t sg, lr;
    res[j] = 0.0f;
    if (a.mode == GM_RESID && t < tiles && sgs.row(16, t, r16, &w_, &sg, &lr) && m < a.B) res[j] = a.R[(size_t)m * a.ldr + lr];
  }
  uint4 wr[D][NT][WP];
  auto issue = [&](auto S) {
    constexpr int s = decltype(S)::value;
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int p = 0; p < WP; p++) wr[s % D][j][p] = wsrc[j][s * 64 * WP + 64 * p];
#pragma unroll
    for (int h = 0; h < 2; h++)
      __builtin_amdgcn_global_load_lds((const void*)(a.X + xo[h] + 32 * s), (lds_void*)&xs[wv][s][256 * h], 16, 0, 0);
  };
  static_for<(D < NS ? D : NS)>(issue);
  f32x4_t acc[NT];
#pragma unroll
  for (int j = 0; j < NT; j++) acc[j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float ss = 0.0f;
  const uint32_t fo0 = (r16 >> 3) * 256 + (r16 & 7) * 32 + 4 * ((2 * g4) ^ (r16 & 7));
  const uint32_t fo1 = (r16 >> 3) * 256 + (r16 & 7) * 32 + 4 * ((2 * g4 + 1) ^ (r16 & 7));
  static_for<NS>([&](auto S) {
    constexpr int s = decltype(S)::value;
    constexpr int last = s + D - 1 < NS - 1 ? s + D - 1 : NS - 1;
    ANA_VMCNT(OPS * (last - s));
    const float4 x0 = *reinterpret_cast<const float4*>(&xs[wv][s][fo0]);
    const float4 x1 = *reinterpret_cast<const float4*>(&xs[wv][s][fo1]);
    const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    if (norm) {
#pragma unroll
      for (int e = 0; e < 8; e++) ss += x[e] * x[e];
    }
    if constexpr (WT == 0) {
#pragma unroll
      for (int j = 0; j < NT; j++) {
        const uint4 w0 = wr[s % D][j][0], w1 = wr[s % D][j][WP - 1];
        const float w[8] = {__uint_as_float(w0.x), __uint_as_float(w0.y), __uint_as_float(w0.z),
                            __uint_as_float(w0.w), __uint_as_float(w1.x), __uint_as_float(w1.y),
                            __uint_as_float(w1.z), __uint_as_float(w1.w)};
#pragma unroll
        for (int e = 0; e < 8; e++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], w[e], acc[j], 0, 0, 0);
      }
    } else {
      bf16x8_t hi;
#pragma unroll
      for (int e = 0; e < 8; e++) hi[e] = (__bf16)x[e];
#pragma unroll
      for (int j = 0; j < NT; j++) {
        const bf16x8_t wb8 = __builtin_bit_cast(bf16x8_t, wr[s % D][j][0]);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, wb8, acc[j], 0, 0, 0);
      }
    }
    if constexpr (s + D < NS) issue(std::integral_constant<int, s + D>{});
  });
#pragma unroll
  for (int j = 0; j < NT; j++)
#pragma unroll
    for (int r = 0; r < 4; r++) red[wv][j][r][lane] = acc[j][r];
  if (norm) {
    float v = ss;
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    if (g4 == 0) ssr[wv][r16] = v;
  }
  __syncthreads();
  const uint32_t mi = 4 * g4 + wv;
  const float rs = norm ? 1.0f / sqrtf((((ssr[0][mi] + ssr[1][mi]) + ssr[2][mi]) + ssr[3][mi]) / (float)K + 1.0e-5f) : 1.0f;
#pragma unroll
  for (int j = 0; j < NT; j++) {
    const uint32_t t = NT * blockIdx.x + j;
    const float* w_;
    uint32_t sg, lr;
    const bool ok = t < tiles && sgs.row(16, t, r16, &w_, &sg, &lr) && m < a.B;
    float y = ((red[0][j][wv][lane] + red[1][j][wv][lane]) + red[2][j][wv][lane]) + red[3][j][wv][lane];
    if (norm) y *= rs;
    if (a.mode == GM_SILU) {
      const float up = __shfl_xor(y, 8, 64);
      if (r16 < 8 && ok) a.seg[0].Y[(size_t)m * a.seg[0].ldy + lr] = fast_silu(y) * up;
    } else if (ok) {
      if (a.mode == GM_RESID) y = res[j] + y;
      if (sg) a.seg[1].Y[(size_t)m * a.seg[1].ldy + lr] = y;
      else a.seg[0].Y[(size_t)m * a.seg[0].ldy + lr] = y;
    }
  }
}

bool gemm_pk_fits(const GemvArgs& a) {
  return !a.amax && a.B > 0 && a.K % 128 == 0 && a.K <= 2048 && (a.ldx & 3) == 0 &&
         (reinterpret_cast<uintptr_t>(a.X) & 15) == 0;
}

// two weight tiles a workgroup when the one-tile grid has 4 to 16
// workgroups a CU (measured at B = 64: gate|up 10.3 -> 8.9 us fp32, 7.9 ->
// 6.4 us bf16; with fewer, q|k|v|z and Wo lose the spread over the CUs,
// with more, the head gains nothing), and K <= 1024 (the register ring of
// two tiles' weights)
constexpr uint32_t kPwTwoTileMin = 1024, kPwTwoTileMax = 4096;

// The register ring holds D steps: three for K <= 1024, four above (a sweep
// at B = 16 and 64 with the weights evicted between launches: one step
// ahead starves the loads; six or eight ahead, every load issued at once,
// cost 0.3-1.1 us more a product than three)
template <int NS>
static hipError_t pw_go(const GemvArgs& a, const uint4* p, int bf, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  constexpr int D = NS < 3 ? NS : NS <= 8 ? 3 : 4;
  const uint32_t tiles = pk_tiles(a), mt = (a.B + 15) / 16;
  if constexpr (NS <= 8) {
    if (tiles * mt >= kPwTwoTileMin && tiles * mt <= kPwTwoTileMax) {
      const dim3 grid((tiles + 1) / 2, mt);
      if (bf) ANA_LAUNCH_F((k_gemm_pw<1, NS, D, 2>), grid, dim3(256), 0, st, e0, e1, a, p, tiles);
      else ANA_LAUNCH_F((k_gemm_pw<0, NS, D, 2>), grid, dim3(256), 0, st, e0, e1, a, p, tiles);
      return hipGetLastError();
    }
  }
  const dim3 grid(tiles, mt);
  if (bf) ANA_LAUNCH_F((k_gemm_pw<1, NS, D, 1>), grid, dim3(256), 0, st, e0, e1, a, p, tiles);
  else ANA_LAUNCH_F((k_gemm_pw<0, NS, D, 1>), grid, dim3(256), 0, st, e0, e1, a, p, tiles);
  return hipGetLastError();
}

template <int... I>
static hipError_t pw_dispatch(const GemvArgs& a, const uint4* p, int bf, hipStream_t st, hipEvent_t e0, hipEvent_t e1,
                              std::integer_sequence<int, I...>) {
  hipError_t e = hipErrorInvalidValue;
  ((a.K == 128u * (I + 1) ? (void)(e = pw_go<I + 1>(a, p, bf, st, e0, e1)) : (void)0), ...);
  return e;
}

hipError_t launch_gemm_pk(const GemvArgs& a, const void* pk, int bf, hipStream_t st, hipEvent_t e0, hipEvent_t e1) {
  if (!gemm_pk_fits(a) || !pk) return hipErrorInvalidValue;
  return pw_dispatch(a, static_cast<const uint4*>(pk), bf, st, e0, e1, std::make_integer_sequence<int, 16>{});
}

}  // namespace ana
