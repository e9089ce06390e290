// Decode attention of more than kSmallB rows in the fast modes (gfx950).
#include <hip/hip_runtime.h>

#include "ana_internal.h"
#include "mfma.h"
#include "wave.h"

namespace ana {

// the sum over each group of L consecutive lanes (L = 4, 8 or 16), in every
// lane of the group, by DPP
template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
  static_assert(L == 4 || L == 8 || L == 16, "a quad, a half row or a row");
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  if constexpr (L >= 8) v += dpp<0x141>(v);
  if constexpr (L >= 16) v += dpp<0x140>(v);
  return v;
}

// Decode attention of more than kSmallB rows in the fast modes: one
// workgroup per (head, row) over the row's live slots 0 .. npos. The row's
// k (qk-normed when on) and v go to its slot first; its own slot's score
// and product come from registers. A slot is L = HD / 4 lanes (a float4 of
// its K and V row each, so a slot's row is one 16 L-byte piece), the
// workgroup G = 256 / L slot groups, a stage U slots a group. A stage's K
// and V come in together, D stages in flight in registers from before the
// row's q is known, and each group keeps a running max m, sum l and sum
// e V of its own (scaled once a stage), so no barrier and no wait but the
// loads' stand between the stages; the groups meet in LDS at the end. Bound
// by the K and V rows' bytes: 59 MB a layer at B = 64 and ~150 slots 18.5 us,
// 379 MB at B = 32 and ~1900 in 256-slot pieces 77.2 us with the combine's
// 4.8 (two passes over the window, the scores in LDS between them: 19.4,
// 78.0 and 6.5; a kernel that only reads those rows, in pieces of 256 bytes
// or of 1 KB: 14.7 and 67). U = 2 and D = 3 against 4 and 3: fewer
// registers, 18.5 against 20.2 us. With
// a split grid (gridDim.z > 1) workgroup z takes slots z SL .. z SL + SL - 1
// of the live ones (SL = kRowsSplit), and leaves its max m, its sum l = sum e
// and its o = sum e V (e = exp(sc s - m), no sink) in part for
// k_attn_rows_comb.
template <int HD>
__global__ __launch_bounds__(256) void k_attn_rows(AttnArgs a) {
  constexpr int L = HD / 4, G = 256 / L, U = 2, D = 3, ST = U * G;
  constexpr float kLow = -3.0e38f;   // below every score, and finite (exp(-inf - kLow) is 0)
  __shared__ float nrm[2], ms[G], ls[G], ws[G];
  __shared__ __align__(16) float kv[2][HD];
  __shared__ float4 op[G][L];
  const uint32_t h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const uint32_t d = a.d, ctx = a.ctx;
  const uint32_t pos = a.pos[b];
  const uint32_t slot = pos % ctx, npos = pos < ctx - 1 ? pos : ctx - 1;
  const uint32_t nsp = gridDim.z, sp = blockIdx.z;
  const uint32_t s0 = nsp > 1 ? sp * kRowsSplit : 0u;
  const uint32_t s1 = nsp > 1 ? min(npos + 1, s0 + kRowsSplit) : npos + 1;   // slots s0 .. s1 - 1
  float* part = nsp > 1 ? a.part + (((size_t)b * a.heads + h) * nsp + sp) * (HD + 2) : nullptr;
  if (s0 >= s1) {
    // no live slot in this split
    if (tid < HD) part[2 + tid] = 0.0f;
    if (tid == 0) {
      part[0] = -INFINITY;
      part[1] = 0.0f;
    }
    return;
  }
  float* Kr = a.KV.base + (size_t)a.seq[b] * a.KV.seq_stride + a.KV.layer_off;
  float* Vr = Kr + (size_t)ctx * d;
  const uint32_t li = tid % L, g = tid / L;
  // stage i's pieces (slots past the last load the last one again)
  const float* kb = Kr + h * HD + 4 * li;
  const float* vb = Vr + h * HD + 4 * li;
  float4 kr[D][U], vr[D][U];
  auto issue = [&](auto I, uint32_t t0) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const size_t o = (size_t)min(t0 + g + u * G, s1 - 1) * d;
      kr[decltype(I)::value][u] = *reinterpret_cast<const float4*>(kb + o);
      vr[decltype(I)::value][u] = *reinterpret_cast<const float4*>(vb + o);
    }
  };
  static_for<D>([&](auto I) { issue(I, s0 + ST * decltype(I)::value); });
  // the row's q, k and v: every group holds q in its lanes; k and v for the
  // ring
  const float* x = a.QKV + (size_t)b * 3 * d + h * HD;
  float4 q4 = *reinterpret_cast<const float4*>(x + 4 * li);
  float4 k4 = *reinterpret_cast<const float4*>(x + d + 4 * li);
  const float4 v4 = *reinterpret_cast<const float4*>(x + 2 * d + 4 * li);
  if (a.gq) {
    // M.qkn (bend/Dense/Model.bend:39-42)
    auto qkn = [&](float4 t, const float* gain) {
      const float n = 1.0f / sqrtf(lanes_sum<L>((t.x * t.x + t.y * t.y) + (t.z * t.z + t.w * t.w)) / (float)HD + 1.0e-5f);
      const float4 gn = *reinterpret_cast<const float4*>(gain + 4 * li);
      return make_float4((t.x * n) * (1.0f + gn.x), (t.y * n) * (1.0f + gn.y), (t.z * n) * (1.0f + gn.z),
                         (t.w * n) * (1.0f + gn.w));
    };
    q4 = qkn(q4, a.gq);
    k4 = qkn(k4, a.gk);
  }
  const float sc = 1.0f / sqrtf((float)HD);
  auto dot = [&](float4 k) { return sc * lanes_sum<L>((q4.x * k.x + q4.y * k.y) + (q4.z * k.z + q4.w * k.w)); };
  float m = kLow, l = 0.0f;
  float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  // group 0 of the workgroup that has the row's own slot starts from it
  if (g == 0 && slot >= s0 && slot < s1) {
    *reinterpret_cast<float4*>(Kr + (size_t)slot * d + h * HD + 4 * li) = k4;
    *reinterpret_cast<float4*>(Vr + (size_t)slot * d + h * HD + 4 * li) = v4;
    m = fmaxf(dot(k4), kLow);
    l = expf(dot(k4) - m);
    o = make_float4(l * v4.x, l * v4.y, l * v4.z, l * v4.w);
  }
  auto stage = [&](auto I, uint32_t t0) {
    constexpr int i = decltype(I)::value;
    float s[U], mn = m;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const uint32_t t = t0 + g + u * G;
      s[u] = dot(kr[i][u]);
      if (t >= s1 || t == slot) s[u] = -INFINITY;
      mn = fmaxf(mn, s[u]);
    }
    const float c = expf(m - mn);
    m = mn;
    l *= c;
    o.x *= c;
    o.y *= c;
    o.z *= c;
    o.w *= c;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const float e = expf(s[u] - m);
      l += e;
      o.x = fmaf(e, vr[i][u].x, o.x);
      o.y = fmaf(e, vr[i][u].y, o.y);
      o.z = fmaf(e, vr[i][u].z, o.z);
      o.w = fmaf(e, vr[i][u].w, o.w);
    }
  };
  for (uint32_t t0 = s0; t0 < s1; t0 += D * ST)
    static_for<D>([&](auto I) {
      const uint32_t t = t0 + ST * decltype(I)::value;
      if (t < s1) {
        stage(I, t);
        issue(I, t + D * ST);
      }
    });
  if (li == 0) {
    ms[g] = m;
    ls[g] = l;
  }
  op[g][li] = o;
  __syncthreads();
  const float sink = a.sink ? a.sink[h] : 0.0f;
  float mx = a.sink && nsp == 1 ? sink : kLow;
#pragma unroll
  for (int j = 0; j < G; j++) mx = fmaxf(mx, ms[j]);
  if (tid < G) ws[tid] = expf(ms[tid] - mx);
  __syncthreads();
  if (tid < HD) {
    const uint32_t c = tid / 4, e = tid % 4;
    float acc = 0.0f, den = 0.0f;
#pragma unroll 8
    for (int j = 0; j < G; j++) {
      const float4 p4 = op[j][c];
      acc = fmaf(ws[j], e == 0 ? p4.x : e == 1 ? p4.y : e == 2 ? p4.z : p4.w, acc);
      den = fmaf(ws[j], ls[j], den);
    }
    if (nsp > 1) {
      part[2 + tid] = acc;
      if (tid == 0) {
        part[0] = mx;
        part[1] = den;
      }
      return;
    }
    if (a.sink) den += expf(sink - mx);
    a.O[(size_t)b * d + h * HD + tid] = acc / den;
  }
}

// the splits of k_attn_rows for one (head, row), with the sink:
// M = max(m_i, sink), den = sum l_i e^(m_i - M) + e^(sink - M),
// o = sum o_i e^(m_i - M) / den. A lane a split for the maxima and sums
// (at most 64 splits), every split's column loaded before the first is
// added eight at a time: one load round trip in place of one a split.
template <int HD>
__global__ __launch_bounds__(64) void k_attn_rows_comb(AttnArgs a, uint32_t nsp) {
  __shared__ float w[64];
  const uint32_t h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  const float* part = a.part + ((size_t)b * a.heads + h) * nsp * (HD + 2);
  const float mi = tid < nsp ? part[tid * (HD + 2)] : -INFINITY;
  const float li = tid < nsp ? part[tid * (HD + 2) + 1] : 0.0f;
  const uint32_t c = tid < (uint32_t)HD ? tid : 0;
  float v[8];
#pragma unroll
  for (uint32_t i = 0; i < 8; i++) v[i] = part[min(i, nsp - 1) * (HD + 2) + 2 + c];
  const float sink = a.sink ? a.sink[h] : -INFINITY;
  const float M = fmaxf(wmax(mi), sink);
  const float e = tid < nsp ? expf(mi - M) : 0.0f;
  w[tid] = e;
  const float den = wsum(li * e) + (a.sink ? expf(sink - M) : 0.0f);
  __syncthreads();
  float acc = 0.0f;
#pragma unroll
  for (uint32_t i = 0; i < 8; i++)
    if (i < nsp) acc = fmaf(v[i], w[i], acc);
  for (uint32_t i = 8; i < nsp; i++) acc = fmaf(part[i * (HD + 2) + 2 + c], w[i], acc);
  if (tid < (uint32_t)HD) a.O[(size_t)b * a.d + h * HD + tid] = acc / den;
}

hipError_t launch_attn_rows(const AttnArgs& a, bool split, hipStream_t st) {
  const uint32_t hd = a.heads ? a.d / a.heads : 0;
  if (!a.seq || !a.pos || !a.write_kv || a.ctx == 0 || hd * a.heads != a.d) return hipErrorInvalidValue;
  if (split && !a.part) return hipErrorInvalidValue;
  const uint32_t nsp = split ? (a.ctx + kRowsSplit - 1) / kRowsSplit : 1u;
  if (nsp > 64 || (split && (size_t)a.B * a.heads * nsp * (hd + 2) > a.part_cap)) return hipErrorInvalidValue;
#define L_(H)                                                                                       \
  hipLaunchKernelGGL(k_attn_rows<H>, dim3(a.heads, a.B, nsp), dim3(256), 0, st, a);                \
  if (split) hipLaunchKernelGGL(k_attn_rows_comb<H>, dim3(a.heads, a.B), dim3(64), 0, st, a, nsp)
  switch (hd) {
    case 64: L_(64); break;
    case 32: L_(32); break;
    case 16: L_(16); break;
    default: return hipErrorInvalidValue;
  }
#undef L_
  return hipGetLastError();
}

}  // namespace ana
