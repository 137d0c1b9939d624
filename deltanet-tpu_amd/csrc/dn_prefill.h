// Device helpers shared by the prefill kernels (dn_prefill.hip,
// dn_prefill_long.hip): gate activations and head maps, segment ids, and the
// prologue of a token row.
#pragma once
#include "dn_common.h"
#include "dn_host.h"

namespace dn {

constexpr int KD = 128;   // key / value head dim (gdn2.py:1897)

// diag blocks whose in-block log2-decay span exceeds this use the
// overflow-free hierarchical path (e^{69} stays far inside the fp32 range)
constexpr float kDiagSafeLog2 = 100.f;

// ---------------------------------------------------------------------------
// gate activations (gdn2.py:38-47, 133-142, 1970-1974): g = -exp(min(g, 5)),
// b, w = sigmoid.  The sigmoid uses the hardware reciprocal (v_rcp_f32, 1 ulp):
// 1 + e^{-x} >= 1, and an infinite denominator gives exactly 0.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float sigmoid_fast(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }

// head of a K-side gate (g, b) used by execution head h
__device__ __forceinline__ int kgate_head(const PF& p, int H, int h) {
  if (H == 1) return 0;
  if (p.gates_at_hv) return (H == p.Hv) ? h : h / p.G;
  return h;
}
// head of a value-side gate (w) used by value head hv
__device__ __forceinline__ int vgate_head(const PF& p, int H, int hv) {
  if (H == 1) return 0;
  return (H == p.Hv) ? hv : hv / p.G;
}

// A segment id as its two 32-bit words; an int32 id repeats its one word in
// hi (no select on the loaded value, so nothing waits for the load until the
// ids are compared; equality is unchanged)
struct SegId {
  int32_t lo, hi;
  __device__ __forceinline__ bool operator!=(const SegId& o) const { return lo != o.lo || hi != o.hi; }
};
__device__ __forceinline__ SegId seg_raw(const PF& p, int b, int t) {
  const int64_t i = p.seg_batched ? (int64_t)b * p.L + t : (int64_t)t;
  const bool w64 = p.seg_dt == DT_I64;
  const int32_t* s32 = (const int32_t*)p.seg + (w64 ? 2 * i : i);
  return SegId{s32[0], s32[w64 ? 1 : 0]};
}

// q, k and b * k of one token row in fragment order (slab s: elements
// 8s..8s+7), after the prologue: L2 normalisation (gdn2.py:1990-1996, the
// normalised q and k rounded back to the input type), the q scale, the b
// activation or clamp, and zeros for tokens past the end.
template <class TIn>
__device__ __forceinline__ void row_inputs(const PF& p, const Raw8<TIn> (&rq)[4], const Raw8<TIn> (&rk)[4],
                                           const Raw8<float> (&rb)[4], float b_scalar, bool valid, float (&qv)[32],
                                           float (&kv)[32], float (&bet)[32]) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    rq[s].to(qv + 8 * s);
    rk[s].to(kv + 8 * s);
  }
  if (p.b_c == 1) {
#pragma unroll
    for (int e = 0; e < 32; ++e) bet[e] = b_scalar;
  } else {
#pragma unroll
    for (int s = 0; s < 4; ++s) rb[s].to(bet + 8 * s);
  }
  float ssq = 0.f, ssk = 0.f;
#pragma unroll
  for (int e = 0; e < 32; ++e) { ssq += qv[e] * qv[e]; ssk += kv[e] * kv[e]; }
  ssq += __shfl_xor(ssq, 16); ssq += __shfl_xor(ssq, 32);
  ssk += __shfl_xor(ssk, 16); ssk += __shfl_xor(ssk, 32);
  if (p.fuse) {
    const float rq = rsqrtf(ssq + 1e-6f) , rk = rsqrtf(ssk + 1e-6f);
#pragma unroll
    for (int e = 0; e < 32; ++e) {
      qv[e] = (qv[e] * rq) * p.scale;
      kv[e] = kv[e] * rk;
      bet[e] = sigmoid_fast(bet[e]);
    }
  } else if (p.l2norm) {
    const float rq = rsqrtf(ssq + 1e-6f), rk = rsqrtf(ssk + 1e-6f);
#pragma unroll
    for (int e = 0; e < 32; ++e) { qv[e] = round_as<TIn>((qv[e] * rq) * p.scale); kv[e] = round_as<TIn>(kv[e] * rk); }
  } else {
#pragma unroll
    for (int e = 0; e < 32; ++e) qv[e] = round_as<TIn>(qv[e] * p.scale);
  }
  if (p.guard && !p.fuse) {
#pragma unroll
    for (int e = 0; e < 32; ++e) bet[e] = fmaxf(bet[e], 0.f);
  }
#pragma unroll
  for (int e = 0; e < 32; ++e) {
    qv[e] = valid ? qv[e] : 0.f;
    kv[e] = valid ? kv[e] : 0.f;
    bet[e] = valid ? bet[e] * kv[e] : 0.f;
  }
}

}  // namespace dn
