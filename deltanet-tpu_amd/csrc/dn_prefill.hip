// Chunked WY prefill for GDN-2 / Gated DeltaNet on gfx950 (MI355X).
//
// Reference algorithm (maelie-labs/deltanet-tpu v0.3.0, src/deltanet_tpu/):
//   prepass   gdn2.py:115-240   (Lambda, A, M, T = (I+A)^-1, W, U, qe, ke)
//   state     gdn2.py:585-652   (Vnew = U - W S, O = qe S + M Vnew,
//                                S <- [same doc] diag(e^Lend) S + ke^T Vnew)
//   flags     gdn2.py:1291-1302 (is_new_doc, all_same_doc per chunk)
//   wrapper   gdn2.py:1970-2125 (clamps, scale, L2-norm, gate broadcast,
//                                segment canonicalisation, padding)
//
// The MI355X design runs 64-token chunks in two launches per token block.  Per
// chunk, with be = b k e^Lambda, qe = q e^Lambda, ke = k e^{Lend - Lambda}
// (tokens of the chunk's first / first / last document) and T = (I + A)^-1:
//     Vn = T (w v - be S),   O = qe S + M Vn,
//     S <- [same doc] diag(e^Lend) S + ke^T Vn
//   k_prepass (one workgroup of 4 waves per (batch, exec head, chunk) unit)
//       everything that depends neither on the values nor on the state:
//       prologue, Lambda, be, qe, ke^T, A and M on MFMA, T by blocked
//       substitution on fp32 MFMA.
//   k_chain   (grid: 16-column tiles x exec head x batch, 8 waves)
//       the sequential scan over chunks with the fp32 state in VGPRs, three
//       dependent products per chunk, and each chunk's output beside it.
// T is applied inside the scan: folding it into per-chunk operators of the
// state (W = T be, U = T (w v), an affine map of S) made every unit read v and
// w, run five more products and write operators as wide as the values; the
// scan now reads v and w itself and the operators do not grow with the number
// of value heads.
//
// Intermediates live in a caller-provided workspace sized for one token
// block; every array is stored in the MFMA lane order of its consumer.
#include <mutex>

#include "dn_common.h"
#include "dn_host.h"
#include "dn_prefill.h"

namespace dn {

constexpr int CH = 64;    // chunk size (the reference's 128 is a TPU tile size; the recurrence is the same)
constexpr int NB = CH / 16;   // 16-token blocks of a chunk
constexpr int XP = 132;   // fp32 LDS pitch (floats) of the Lambda rows: conflict-free 16-lane column groups
constexpr int AP = 68;    // fp32 LDS pitch of A and T
constexpr int kMaxBlockChunks = 1024;   // chunks per token block (chain's LDS flag table)

// a 16 x 32 slab of an operand with two slabs per tile (reduction over the
// chunk's 64 tokens)
__device__ __forceinline__ int fofs2(int tile, int slab, int lane) { return ((tile * 2 + slab) * 64 + lane) * 8; }

// T and M (64 x 64, lower triangular): the six slabs that are not all zero
__device__ __forceinline__ int tofs(int tile, int slab, int lane) { return ((tile + tile / 3 + slab) * 64 + lane) * 8; }
constexpr int TM = 6 * 64 * 8;   // elements of T or M

// One unit of a prepass launch: (batch, execution head, chunk) with the
// XCD-aware remap (the hardware deals linear block ids to the 8 XCDs
// round-robin; consecutive chunks of a head share one XCD's L2).
struct Unit {
  int b, h, c, hk;
  int tb, t_end;   // first token, end of the valid tokens
  int64_t u;
};
__device__ __forceinline__ Unit unit_of(const PF& p) {
  Unit x;
  const int units = p.B * p.Hx * p.NCb;
  int id = blockIdx.x;
  if ((units & 7) == 0) id = (id & 7) * (units >> 3) + (id >> 3);
  x.c = id % p.NCb;
  id /= p.NCb;
  x.h = id % p.Hx;
  x.b = id / p.Hx;
  x.hk = p.gates_at_hv ? x.h / p.G : x.h;
  x.tb = p.t0 + x.c * CH;
  x.t_end = min(p.t0 + p.nt, p.L);
  x.u = ((int64_t)x.b * p.Hx + x.h) * p.NCb + x.c;
  return x;
}

// Segment ids of a chunk: wave 0 loads token l's id and its predecessor's,
// and the ids at the chunk's edge and at token 0 (every lane loads, so nothing
// is consumed inside a divergent branch before it is needed).
struct ChunkSeg {
  SegId t{0, 0}, tp{0, 0}, s0{0, 0}, a{0, 0}, b{0, 0};
  int32_t iseg = 0;
  __device__ __forceinline__ void load(const PF& p, const Unit& x, int l) {
    if (p.seg != nullptr) {
      t = seg_raw(p, x.b, min(x.tb + l, x.t_end - 1));
      tp = seg_raw(p, x.b, max(min(x.tb + l - 1, x.t_end - 1), 0));
      s0 = seg_raw(p, x.b, 0);
      a = seg_raw(p, x.b, x.tb);
      b = seg_raw(p, x.b, max(x.tb - 1, 0));
    }
    if (p.init_seg != nullptr) iseg = p.init_seg[x.b];
  }
  // The in-chunk document index (segment canonicalisation: doc[i] = number of
  // segment starts among tokens 1..i, one wave ballot) into LDS, and the
  // chunk's flags (gdn2.py:1291-1302) from the lane of its last token.
  __device__ __forceinline__ void finish(const PF& p, const Unit& x, int l, int* doc) {
    const uint64_t bal = __ballot(l > 0 && p.seg != nullptr && (t != tp));
    const int d = __popcll(bal & ((2ull << l) - 1ull));   // lanes 0..l (l = 63: all)
    doc[l] = d;
    if (l != 63 || x.h != 0) return;
    int is_new;
    if (x.tb == 0) {
      if (p.has_init) {
        is_new = 0;
        // initial_state_segment_id is int32; a wider first id differs from it
        // when its high word is not the sign extension of its low word
        if (p.init_seg != nullptr) is_new = (s0.lo != iseg) || (p.seg_dt == DT_I64 && s0.hi != (iseg < 0 ? -1 : 0));
      } else {
        is_new = 1;
      }
    } else if (x.c == 0 && !p.has_init) {
      is_new = 1;
    } else {
      is_new = p.seg ? (a != b) : 0;
    }
    p.flags[((int64_t)x.b * p.NCb + x.c) * 2 + 0] = is_new;
    p.flags[((int64_t)x.b * p.NCb + x.c) * 2 + 1] = (d == 0);
  }
};

// T = (I + A)^-1 of one chunk (A strictly lower, fp32 in X with pitch AP, the
// tiles right of even diagonal blocks zeroed), by blocked forward
// substitution; Tt is 64 x AP floats of scratch that nobody reads any more.
// Wave w inverts diagonal block w, then per block row a wave bt < a forms
// T[a][bt] = -D_a sum_{cc = bt}^{a-1} A[a][cc] T[cc][bt].  Each 16x16x16
// product runs as 4 steps of the 16x16x4 fp32 MFMA with lane (r, q) holding
// reduction index 4q + kk at step kk, so a lane's A operand (row of A) and B
// operand (row of T^T, kept in Tt) are one 16-byte LDS read each.  T goes to
// the workspace as fragments (wave w: row tile w), split in bf16 mode.
template <bool BF>
__device__ __forceinline__ void invert_and_store(float* X, float* Tt, typename Store<BF>::ST* g_Th,
                                                 typename Store<BF>::ST* g_Tl, int w, int l) {
  using SS = Store<BF>;
  const int r16 = l & 15, q = l >> 4;
  {
    // every lane group q works on the same columns (LDS reads broadcast); the
    // group w stores, so the four waves write four different diagonal blocks
    const int a = w;
    float tc[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) tc[m] = (m == r16) ? 1.f : 0.f;
#pragma unroll
    for (int ii = 1; ii < 16; ++ii) {
      float acc = 0.f;
#pragma unroll
      for (int m = 0; m < ii; ++m) acc += X[(16 * a + ii) * AP + 16 * a + m] * tc[m];
      if (ii > r16) tc[ii] = -acc;
    }
    if (q == 0) {
#pragma unroll
      for (int ii = 0; ii < 16; ++ii) X[(16 * a + ii) * AP + 16 * a + r16] = tc[ii];
    } else if (q == 1) {
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        *reinterpret_cast<f32x4*>(&Tt[(16 * a + r16) * AP + 16 * a + 4 * i4]) =
            f32x4{tc[4 * i4], tc[4 * i4 + 1], tc[4 * i4 + 2], tc[4 * i4 + 3]};
    }
  }
  lds_barrier();
#pragma unroll
  for (int a = 1; a < NB; ++a) {
    const int bt = w;
    f32x4 res = zero4();
    if (bt < a) {
      f32x4 acc0 = zero4(), acc1 = zero4();
#pragma unroll
      for (int cc = 0; cc < a; ++cc) {
        if (cc >= bt) {
          const f32x4 Ar = *reinterpret_cast<const f32x4*>(&X[(16 * a + r16) * AP + 16 * cc + 4 * q]);
          const f32x4 Br = *reinterpret_cast<const f32x4*>(&Tt[(16 * bt + r16) * AP + 16 * cc + 4 * q]);
#pragma unroll
          for (int kk = 0; kk < 4; ++kk) {
            if (cc & 1) acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(Ar[kk], Br[kk], acc1, 0, 0, 0);
            else acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(Ar[kk], Br[kk], acc0, 0, 0, 0);
          }
        }
      }
      const f32x4 Dr = *reinterpret_cast<const f32x4*>(&X[(16 * a + r16) * AP + 16 * a + 4 * q]);
      // lane (j, q) holds P[4q + ii][j]: the B operand of step kk is acc[kk]
      f32x4 r = zero4();
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        r = __builtin_amdgcn_mfma_f32_16x16x4f32(Dr[kk], acc0[kk] + acc1[kk], r, 0, 0, 0);
      res = -r;
    }
    lds_barrier();   // row a of A is read
    if (bt < a) {
      // lane (j, q) holds T[16a + 4q + ii][16bt + j]
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) X[(16 * a + 4 * q + ii) * AP + 16 * bt + r16] = res[ii];
      *reinterpret_cast<f32x4*>(&Tt[(16 * bt + r16) * AP + 16 * a + 4 * q]) = res;
    }
    lds_barrier();
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (s <= (w >> 1)) {
      float x[8];
      row8<float>(&X[(16 * w + r16) * AP + 32 * s], q, x);
      SS::st8s(g_Th + tofs(w, s, l), g_Tl + tofs(w, s, l), x);
    }
  }
}

// ===========================================================================
// k_prepass: the operands of one chunk that depend neither on the values nor
// on the state (wave w owns token block w).
//
// Lambda is kept block-local: X[i] = sum of g over the 16-token block of i up
// to and including i (log2 units, double-float hi in X / lo in Y), so a
// difference of two Lambdas is never the difference of two large cumulative
// sums (no fp32 cancellation after a strongly decayed stretch).  Cross-block
// factors come from the per-block totals (sums of the totals before / after
// block a, kept as the exponentials Ea / Sa).
//
// Bound by the latency of its dependent phases, so two independent workgroups
// share a CU (80 KB of LDS, 256 VGPRs each).  2048 tokens, 12 key heads: 27 us for
// 384 units, against 59 for the 192 of 128 tokens with the value products.
// ===========================================================================
template <bool BF, class TIn>
__global__ __launch_bounds__(256, 2) void k_prepass(const PF p) {
  using P = Pol<BF>;
  using F3 = typename P::F3;
  using SS = Store<BF>;
  using ST = typename SS::ST;
  __shared__ __align__(16) float X[CH * XP];   // Lambda hi -> A -> T (fp32)
  __shared__ __align__(16) float Y[CH * XP];   // Lambda lo -> column factors -> T^T
  __shared__ float Ftab[NB * KD];     // e^{total of block b}
  __shared__ float Mid0[NB * KD];     // e^{g at the first token of block a}
  __shared__ float Ea[NB * KD];       // e^{Lambda at the first token of block a} (chunk-global)
  __shared__ float Sa[NB * KD];       // e^{sum of the totals of blocks > a}
  __shared__ float Fa[NB * KD];       // e^{Lambda(last) - Lambda(first token) of block a}
  __shared__ float Gt[NB * KD];       // e^{Lambda(first token of block a) - Lambda(row 32)}
  __shared__ int doc[CH];
  __shared__ int unsafe_part[2][NB];  // per 64-channel half: block needs the hierarchical path
  __shared__ int wide_part[2];        // per 64-channel half: the chunk-reference path is unsafe

  const int tid = threadIdx.x;
  // (the wave index as a scalar: tile indices over waves stay in scalar registers)
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, r16 = l & 15, q = l >> 4;
  const Unit x0 = unit_of(p);
  const int tb = x0.tb, t_end = x0.t_end, b = x0.b, h = x0.h;
  const int64_t u = x0.u;
  ST* g_be = (ST*)p.BeA + u * (CH * KD);
  ST* g_qh = (ST*)p.QeAh + u * (CH * KD);
  ST* g_ql = (ST*)p.QeAl + u * (CH * KD);
  ST* g_keh = (ST*)p.KeTh + u * (CH * KD);
  ST* g_kel = (ST*)p.KeTl + u * (CH * KD);
  ST* g_Th = (ST*)p.TAh + u * TM;
  ST* g_Tl = (ST*)p.TAl + u * TM;
  ST* g_Mh = (ST*)p.MAh + u * TM;
  ST* g_Ml = (ST*)p.MAl + u * TM;
  float* g_dv = p.dvec + u * KD;

  // Global loads are issued up front, in the order their values are needed
  // (the vector-memory counter drains in order, so a load is only ever waited
  // for together with the loads issued before it).
  ChunkSeg sg;
  if (w == 0) sg.load(p, x0, l);
  // gates g: lane (half, cg) holds tokens 16w + 8 half .. + 7 of channels
  // 4cg..4cg+3 (a gate with one channel repeats it; out-of-range tokens read
  // the last valid token and are zeroed below)
  const int half = l >> 5, cg = l & 31;
  f32x4 gl[8];
  {
    const int hg = kgate_head(p, p.g_h, h);
    const int t8 = tb + 16 * w + 8 * half;
    const float* gp = (const float*)p.g + ((int64_t)b * p.L * p.g_h + hg) * p.g_c;
    const int64_t gs = (int64_t)p.g_h * p.g_c;
    if (p.g_c == 1) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float* r = gp + min(t8 + i, t_end - 1) * gs;
        gl[i] = f32x4{r[0], r[0], r[0], r[0]};
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) gl[i] = *reinterpret_cast<const f32x4*>(gp + min(t8 + i, t_end - 1) * gs + 4 * cg);
    }
  }
  Raw8<TIn> rq[4], rk[4];
  Raw8<float> rb[4];
  float b_scalar = 0.f;
  {
    const int hbg = kgate_head(p, p.b_h, h);
    const int t = tb + 16 * w + r16;
    const int tt = t < t_end ? t : tb;
    const TIn* qp = (const TIn*)p.q + (((int64_t)b * p.L + tt) * p.Hk + x0.hk) * KD;
    const TIn* kp = (const TIn*)p.k + (((int64_t)b * p.L + tt) * p.Hk + x0.hk) * KD;
    const float* bp = (const float*)p.b + (((int64_t)b * p.L + tt) * p.b_h + hbg) * p.b_c;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      rq[s].load(qp + 32 * s, q);
      rk[s].load(kp + 32 * s, q);
    }
    if (p.b_c == 1) {
      b_scalar = bp[0];
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) rb[s].load(bp + 32 * s, q);
    }
  }

  // ---- phase 1: block-local Lambda (double-float: X = hi, Y = lo) ----------
  {
    const float gmax = p.guard ? -1e-6f : 0.f;
    const int nvalid = t_end - (tb + 16 * w + 8 * half);   // of this lane's tokens (may be <= 0)
    f32x4 hi[8], lo[8];
    f32x4 h = zero4(), lw = zero4();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float gv = gl[i][e];
        gv = p.fuse ? -__expf(fminf(gv, 5.f)) : fminf(gv, 0.f);   // _nonpositive (NaN -> 0)
        gv = i < nvalid ? fminf(gv, gmax) : 0.f;
        // error-free accumulation (TwoSum)
        const float sum = h[e] + gv;
        const float bb = sum - h[e];
        lw[e] += (h[e] - (sum - bb)) + (gv - bb);
        h[e] = sum;
      }
      hi[i] = h;
      lo[i] = lw;
    }
    // the second half of the block continues the first (held by lane - 32)
    f32x4 h1, l1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float hp = __shfl_xor(h[e], 32), lp = __shfl_xor(lw[e], 32);
      h1[e] = half ? hp : 0.f;
      l1[e] = half ? lp : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      f32x4 xo, yo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float sum = h1[e] + hi[i][e];
        const float bb = sum - h1[e];
        const float lt = l1[e] + lo[i][e] + ((h1[e] - (sum - bb)) + (hi[i][e] - bb));
        // an exact split of hi * log2(e)
        const float ph = sum * kLog2e;
        xo[e] = ph;
        yo[e] = fmaf(sum, kLog2e, -ph) + lt * kLog2e;
      }
      const int row = 16 * w + 8 * half + i;
      *reinterpret_cast<f32x4*>(&X[row * XP + 4 * cg]) = xo;
      *reinterpret_cast<f32x4*>(&Y[row * XP + 4 * cg]) = yo;
    }
  }
  if (w == 0) sg.finish(p, x0, l, doc);
  lds_barrier();
  if (tid < KD) {
    float tot[NB];
#pragma unroll
    for (int a = 0; a < NB; ++a) tot[a] = X[(16 * a + 15) * XP + tid] + Y[(16 * a + 15) * XP + tid];
    float acc = 0.f, rl[NB + 1], span[NB];
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      const int sa = 16 * a, ea = sa + 15;
      const float lsa = X[sa * XP + tid] + Y[sa * XP + tid];
      // span of the block after its first token: Lambda(sa) - Lambda(ea) >= 0
      span[a] = (X[sa * XP + tid] - X[ea * XP + tid]) + (Y[sa * XP + tid] - Y[ea * XP + tid]);
      // Lambda at the first token of block a relative to the chunk's first
      // token (not a difference of chunk-global values: a large decay at the
      // chunk's first token would cancel in it)
      rl[a] = a == 0 ? 0.f : rl[a] + lsa;
      rl[a + 1] = rl[a] - span[a];
      Ea[a * KD + tid] = fast_exp2(acc + lsa);   // chunk-global Lambda at the first token of block a
      Mid0[a * KD + tid] = fast_exp2(lsa);
      acc += tot[a];
    }
    g_dv[tid] = fast_exp2(acc);   // e^{Lambda_end}
    // chunk reference row 32: every off-diagonal A / M entry factors as
    // (row i: e^{Lambda_i - Lambda_32}) (column j: e^{Lambda_32 - Lambda_j}),
    // both within 2^{+-100} when the spans on either side of row 32 are
    bool wide = (rl[0] - rl[NB / 2] > kDiagSafeLog2) || (rl[NB / 2] - rl[NB] > kDiagSafeLog2);
#pragma unroll
    for (int a = 0; a < NB; ++a) Gt[a * KD + tid] = fast_exp2(rl[a] - rl[NB / 2]);
    acc = 0.f;
#pragma unroll
    for (int a = NB - 1; a >= 0; --a) { Sa[a * KD + tid] = fast_exp2(acc); acc += tot[a]; }
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      Ftab[a * KD + tid] = fast_exp2(tot[a]);
      Fa[a * KD + tid] = fast_exp2(-span[a]);
      const bool un = __any(span[a] > kDiagSafeLog2);
      if (l == 0) unsafe_part[w][a] = un;
      wide = wide || un;
    }
    wide = __any(wide);
    if (l == 0) wide_part[w] = wide;
  }
  lds_barrier();
  // no block needs the hierarchical path and the chunk reference is safe:
  // phase 2 leaves the column factors of every block as split fragments in
  // Y, and phase 3 is MFMA products of stored fragments only
  const bool chunk_ref = __builtin_amdgcn_readfirstlane(!(wide_part[0] | wide_part[1]));

  // ---- phase 2: per-row operands, diagonal A/M blocks ----------------------
  F3 Rf[4], Qf[4];
  f32x4 Adiag;
  {
    const int a = w;
    const int i = 16 * a + r16;
    const bool valid = tb + i < t_end;
    float qv[32], kv[32], bet[32];
    row_inputs<TIn>(p, rq, rk, rb, b_scalar, valid, qv, kv, bet);
    const bool first = doc[i] == 0;
    const bool last = doc[i] == doc[CH - 1];
    const bool blk_unsafe = unsafe_part[0][a] | unsafe_part[1][a];
    // accA: A tile (lane = column token); accM: M^T tile (lane = row token)
    f32x4 accA = zero4(), accM = zero4();
    // Blocks with a large in-block decay span take the hierarchical path
    // first, while the slab loop's fragments are not yet live.
    if (blk_unsafe) {
      float dq = 0.f;
#pragma unroll
      for (int e = 0; e < 32; ++e) dq += qv[e] * kv[e];
      dq += __shfl_xor(dq, 16);
      dq += __shfl_xor(dq, 32);
      // Overflow-free hierarchical factorisation: the pair (i, j) is split at
      // the highest bit where the in-block indices differ; rows above and
      // columns below the split point are scaled toward it, so every
      // exponent is <= 0.  (accM holds the transposed tile, as above.)
#pragma unroll
      for (int hl = 3; hl >= 0; --hl) {
        const int hh = 1 << hl;
        const int sp = (r16 / (2 * hh)) * 2 * hh + hh;
        const bool upper = r16 >= sp;
        const int srow = 16 * a + sp;
        f32x4 tA = zero4(), tM = zero4();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          float lam[8], lsp[8], laml[8], lspl[8], xa[8], xm[8], xb[8];
          row8<float>(&X[i * XP + 32 * s], q, lam);
          row8<float>(&X[srow * XP + 32 * s], q, lsp);
          row8<float>(&Y[i * XP + 32 * s], q, laml);
          row8<float>(&Y[srow * XP + 32 * s], q, lspl);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float d = (lam[e] - lsp[e]) + (laml[e] - lspl[e]);
            const float x = fast_exp2(upper ? d : -d);
            xa[e] = upper ? bet[8 * s + e] * x : 0.f;
            xm[e] = upper ? qv[8 * s + e] * x : 0.f;
            xb[e] = upper ? 0.f : kv[8 * s + e] * x;
          }
          const F3 fb = P::f3(xb);
          P::m33(tA, P::f3(xa), fb);
          P::m33(tM, fb, P::f3(xm));
        }
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) {
          const int il = 4 * q + ii;
          const int hb = 31 - __builtin_clz((il ^ r16) | 1);  // il == r16 selects nothing
          if (il > r16 && hb == hl) accA[ii] = tA[ii];
          if (r16 > il && hb == hl) accM[ii] = tM[ii];
        }
      }
#pragma unroll
      for (int ii = 0; ii < 4; ++ii)
        if (4 * q + ii == r16) accM[ii] = dq;
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      float lam[8], lsa[8], laml[8], lsal[8], ea[8], sa[8];
      row8<float>(&X[i * XP + 32 * s], q, lam);
      row8<float>(&X[(16 * a) * XP + 32 * s], q, lsa);
      row8<float>(&Y[i * XP + 32 * s], q, laml);
      row8<float>(&Y[(16 * a) * XP + 32 * s], q, lsal);
      row8<float>(&Ea[a * KD + 32 * s], q, ea);
      row8<float>(&Sa[a * KD + 32 * s], q, sa);
      float rA[8], rM[8], bd[8], kc[8], qe[8], bt[8], kt[8];
      if (!blk_unsafe) {
        // every factor within 2^{+-100}: the exponentials of the row's
        // decay relative to the block's first token and their products
        float fa[8];
        row8<float>(&Fa[a * KD + 32 * s], q, fa);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float qh = qv[8 * s + e], kh = kv[8 * s + e], be = bet[8 * s + e];
          const float d_i_sa = (lam[e] - lsa[e]) + (laml[e] - lsal[e]);   // <= 0
          const float er = fast_exp2(d_i_sa);
          const float rr = fast_exp2(-d_i_sa);
          rA[e] = be * er;
          rM[e] = qh * er;
          const float ekc = fa[e] * rr;                 // e^{Lambda(ea) - Lambda(i)}
          kc[e] = kh * ekc;
          const float eL = ea[e] * er;                  // e^{Lambda(i)} (chunk-global)
          bt[e] = first ? be * eL : 0.f;
          kt[e] = last ? kc[e] * sa[e] : 0.f;
          bd[e] = kh * rr;
          qe[e] = first ? qh * eL : 0.f;
        }
      } else {
        float ta[8], tal[8];
        row8<float>(&X[(16 * a + 15) * XP + 32 * s], q, ta);
        row8<float>(&Y[(16 * a + 15) * XP + 32 * s], q, tal);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float qh = qv[8 * s + e], kh = kv[8 * s + e], be = bet[8 * s + e];
          const float d_i_sa = (lam[e] - lsa[e]) + (laml[e] - lsal[e]);   // <= 0
          const float d_ea_i = (ta[e] - lam[e]) + (tal[e] - laml[e]);     // <= 0
          const float er = fast_exp2(d_i_sa);
          rA[e] = be * er;
          rM[e] = qh * er;
          const float ekc = fast_exp2(d_ea_i);
          kc[e] = kh * ekc;
          const float eL = ea[e] * er;
          bt[e] = first ? be * eL : 0.f;
          kt[e] = last ? kh * ekc * sa[e] : 0.f;
          bd[e] = 0.f;   // unused: the hierarchical path formed this block's A and M
          qe[e] = first ? qh * eL : 0.f;
        }
      }
      SS::st8(g_be + fofs(a, s, l), bt);
      SS::st8s(g_qh + fofs(a, s, l), g_ql + fofs(a, s, l), qe);
      {
        // ke^T in fragment layout (row = key, k = token)
        const F3 fkt = P::f3(kt);
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          const auto id = ident_frag<BF>(hf, r16, q);
          f32x4 chi = zero4();
          mma(chi, P::hi(fkt), id);
          const int o = fofs2(2 * s + hf, a >> 1, l) + 4 * (a & 1);
          const float xh[4] = {chi[0], chi[1], chi[2], chi[3]};
          SS::st4(g_keh + o, xh);
          if constexpr (BF) {
            f32x4 clo = zero4();
            mma(clo, fkt.lo, id);
            const float xl[4] = {clo[0], clo[1], clo[2], clo[3]};
            SS::st4(g_kel + o, xl);
          }
        }
      }
      if (chunk_ref) {
        // rows relative to row 32 instead of the block's first token
        float gt[8];
        row8<float>(&Gt[a * KD + 32 * s], q, gt);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          rA[e] *= gt[e];
          rM[e] *= gt[e];
          bd[e] *= __builtin_amdgcn_rcpf(gt[e]);
        }
      }
      Rf[s] = P::f3(rA);
      Qf[s] = P::f3(rM);
      if (!blk_unsafe) {
        // A_aa, M_aa = (R, Qr) (k e^{Lambda_ref - Lambda})^T: every factor stays
        // within 2^{+-100} of 1, so the factorisation cannot overflow.
        const F3 fb = P::f3(bd);
        P::m33(accA, Rf[s], fb);
        P::m33(accM, fb, Qf[s]);
        if (chunk_ref) {
          // the column factors replace this slab's 16 rows x 32 columns of
          // Lambda low words (2 KB, once all lanes of the wave have read
          // them) as the split fragment of lane l: row l / 4, 32 bytes at
          // (l % 4) * 32 of the slab's 128 bytes in that row
          ST* fp = reinterpret_cast<ST*>(&Y[(16 * a + (l >> 2)) * XP + 32 * s]) + (l & 3) * (32 / sizeof(ST));
          SS::stf(fp, P::hi(fb));
          if constexpr (BF) SS::stf(fp + 8, fb.lo);
        }
      }
      if (!chunk_ref) {
        // Kc replaces this slab of the row's Lambda low words once all lanes
        // of the wave have read it (the other slabs' columns are untouched)
        st4<float>(&Y[i * XP + 32 * s + 4 * q], kc);
        st4<float>(&Y[i * XP + 32 * s + 16 + 4 * q], kc + 4);
      }
    }
    // diagonal blocks: A (row-major, LDS) and M (fragment-native, rows = token)
    float mv[4];
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const int il = 4 * q + ii, ia = 16 * a + il, ja = 16 * a + r16;
      const bool same = doc[ia] == doc[ja];
      Adiag[ii] = (il > r16 && same) ? accA[ii] : 0.f;        // A[ia][ja]
      mv[ii] = (r16 >= il && same) ? accM[ii] : 0.f;          // M[ja][ia]
    }
    const int mo = tofs(a, a >> 1, l) + 4 * (a & 1);
    SS::st4s(g_Mh + mo, g_Ml + mo, mv);
    if ((a & 1) == 0) {
      const float z[4] = {0.f, 0.f, 0.f, 0.f};
      SS::st4s(g_Mh + mo + 4, g_Ml + mo + 4, z);
    }
  }
  lds_barrier();

  // ---- phase 3: off-diagonal A/M blocks (X becomes A) -----------------------
  // Wave a forms the pairs (a, bb < a).
  {
    const int a = w;
    // one pair's A tile (rows of block a) and M^T tile, masked by document
    auto pair_out = [&](int bb, const f32x4& accA, const f32x4& accM) {
      float mv[4];
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        const int ia = 16 * a + 4 * q + ii, jb = 16 * bb + r16;
        X[ia * AP + jb] = (doc[ia] == doc[jb]) ? accA[ii] : 0.f;
        mv[ii] = (doc[16 * a + r16] == doc[16 * bb + 4 * q + ii]) ? accM[ii] : 0.f;
      }
      const int mo = tofs(a, bb >> 1, l) + 4 * (bb & 1);
      SS::st4s(g_Mh + mo, g_Ml + mo, mv);
    };
    if (chunk_ref) {
      for (int bb = a - 1; bb >= 0; --bb) {
        // two accumulators per tile (leading and correction products) halve
        // the dependent MFMA chains
        f32x4 accA = zero4(), accM = zero4(), accA2 = zero4(), accM2 = zero4();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const ST* fp = reinterpret_cast<const ST*>(&Y[(16 * bb + (l >> 2)) * XP + 32 * s]) + (l & 3) * (32 / sizeof(ST));
          if constexpr (BF) {
            const F3 fb = SS::fa3(fp, fp + 8);
            mma(accA, Rf[s].hi, fb.hi);   // A[16a + 4q + ii][16bb + r16]
            mma(accM, fb.hi, Qf[s].hi);   // M[16a + r16][16bb + 4q + ii]
            mma(accA2, Rf[s].hi, fb.lo);
            mma(accM2, fb.hi, Qf[s].lo);
            mma(accA2, Rf[s].lo, fb.hi);
            mma(accM2, fb.lo, Qf[s].hi);
          } else {
            const F3 fb = SS::fa(fp);
            P::m33(s & 1 ? accA2 : accA, Rf[s], fb);
            P::m33(s & 1 ? accM2 : accM, fb, Qf[s]);
          }
        }
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) { accA[ii] += accA2[ii]; accM[ii] += accM2[ii]; }
        pair_out(bb, accA, accM);
      }
    } else {
      float mloc[32];
#pragma unroll
      for (int s = 0; s < 4; ++s) row8<float>(&Mid0[a * KD + 32 * s], q, mloc + 8 * s);
      for (int bb = a - 1; bb >= 0; --bb) {
        f32x4 accA = zero4(), accM = zero4();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          float x[8], f[8];
          row8<float>(&Y[(16 * bb + r16) * XP + 32 * s], q, x);
          row8<float>(&Ftab[bb * KD + 32 * s], q, f);
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] *= mloc[8 * s + e];
          const F3 fb = P::f3(x);
          P::m33(accA, Rf[s], fb);   // A[16a + 4q + ii][16bb + r16]
          P::m33(accM, fb, Qf[s]);   // M[16a + r16][16bb + 4q + ii]
#pragma unroll
          for (int e = 0; e < 8; ++e) mloc[8 * s + e] *= f[e];
        }
        pair_out(bb, accA, accM);
      }
    }
    // this wave's diagonal block
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const int ia = 16 * a + 4 * q + ii;
      X[ia * AP + 16 * a + r16] = Adiag[ii];
      if ((a & 1) == 0) X[ia * AP + 16 * a + 16 + r16] = 0.f;
    }
  }
  lds_barrier();
  invert_and_store<BF>(X, Y, g_Th, g_Tl, w, l);
}

// ===========================================================================
// k_prepass_sc: the prepass for one decay, one b and one w per (token, head)
// (the Gated DeltaNet form, chunk_gdn: gdn.py:66-110 broadcasts them over the
// channels), precision "bf16" with bf16 q and k.  The per-channel machinery
// collapses:
//   * Lambda is one cumulative sum per token (double-float, log2 units);
//   * the normalised q and k are exactly bf16 (they are rounded back to the
//     input type), so the Gram matrices k k^T and q k^T are single bf16 MFMAs
//     with fp32 accumulation, and
//       A[i][j] = b_i e^{Lambda_i - Lambda_j} (k k^T)[i][j]   (i > j),
//       M[i][j] =     e^{Lambda_i - Lambda_j} (q k^T)[i][j]   (i >= j),
//     one exponential per pair, whose exponent is <= 0 for every unmasked
//     pair (no factorisation, no overflow path);
//   * be, qe and ke are row scalars times k, q and k: the scan takes the
//     normalised rows once per key head (k, q and k^T fragments, single bf16
//     words, exact) and the row scalars per execution head.
// Bound by memory: 4 x 8192 tokens, 32 heads 382 us for 1.67 GB (4.4 TB/s; 338 to
// 416 us within a dozen calls in a row), against 1510 us for the 128-token
// form's phases, which write operands per head.
// ===========================================================================
template <class TIn>
__global__ __launch_bounds__(256, 3) void k_prepass_sc(const PF p) {
  using P = Pol<true>;
  using F1 = P::F1;
  using SS = Store<true>;
  __shared__ __align__(16) float X[CH * AP];           // A -> T (fp32)
  __shared__ __align__(16) bf16 Kf[2 * CH * KD];       // k, then q fragments [block][slab][lane][8]; -> T^T
  __shared__ float lam_h[CH], lam_l[CH];               // Lambda (log2 units), double-float
  __shared__ float bet_s[CH];                          // b per token (0 past the end)
  __shared__ int doc[CH];
  bf16* Qf = Kf + CH * KD;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, r16 = l & 15, q = l >> 4;
  const Unit x0 = unit_of(p);
  const int tb = x0.tb, t_end = x0.t_end, b = x0.b, h = x0.h;
  const int64_t u = x0.u;
  const int64_t ku = ((int64_t)b * p.Hk + x0.hk) * p.NCb + x0.c;   // key-head unit of the k, q operands
  const bool rows_out = !p.gates_at_hv || h % p.G == 0;           // one unit per key head stores them

  ChunkSeg sg;
  if (w == 0) sg.load(p, x0, l);
  float g_tok = 0.f;
  if (w == 0)
    g_tok = ((const float*)p.g)[((int64_t)b * p.L + min(tb + l, t_end - 1)) * p.g_h + kgate_head(p, p.g_h, h)];
  Raw8<TIn> rq[4], rk[4];
  float b_scalar;
  {
    const int t = tb + 16 * w + r16;
    const int tt = t < t_end ? t : tb;
    const TIn* qp = (const TIn*)p.q + (((int64_t)b * p.L + tt) * p.Hk + x0.hk) * KD;
    const TIn* kp = (const TIn*)p.k + (((int64_t)b * p.L + tt) * p.Hk + x0.hk) * KD;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      rq[s].load(qp + 32 * s, q);
      rk[s].load(kp + 32 * s, q);
    }
    b_scalar = ((const float*)p.b)[((int64_t)b * p.L + tt) * p.b_h + kgate_head(p, p.b_h, h)];
  }

  // ---- Lambda: inclusive scan of g over the chunk (wave 0) -----------------
  if (w == 0) {
    sg.finish(p, x0, l, doc);
    float gv = fminf(g_tok, 0.f);   // _nonpositive (NaN -> 0)
    gv = fminf(gv, p.guard ? -1e-6f : 0.f);
    float hi = (tb + l < t_end) ? gv : 0.f, lo = 0.f;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float h2 = __shfl_up(hi, off), l2 = __shfl_up(lo, off);
      if (l >= off) {
        // error-free hi + h2 (TwoSum), the rounding error joins the low words
        const float sum = hi + h2;
        const float bb = sum - hi;
        lo += l2 + ((hi - (sum - bb)) + (h2 - bb));
        hi = sum;
      }
    }
    const float ph = hi * kLog2e;
    lam_h[l] = ph;
    lam_l[l] = fmaf(hi, kLog2e, -ph) + lo * kLog2e;
  }
  // ---- rows of token block w ------------------------------------------------
  {
    const int i = 16 * w + r16;
    const bool valid = tb + i < t_end;
    float qv[32], kv[32], bet[32];
    const Raw8<float> none[4] = {};
    row_inputs<TIn>(p, rq, rk, none, b_scalar, valid, qv, kv, bet);
    float bsc = b_scalar;
    if (p.guard) bsc = fmaxf(bsc, 0.f);
    if (q == 0) bet_s[i] = valid ? bsc : 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      // the normalised rows are bf16 values: their fragments are exact
      const F1 fk = P::f1(kv + 8 * s), fq = P::f1(qv + 8 * s);
      SS::stf(Kf + fofs(w, s, l), fk);
      SS::stf(Qf + fofs(w, s, l), fq);
      if (rows_out) {
        SS::stf((bf16*)p.BeA + ku * (CH * KD) + fofs(w, s, l), fk);
        SS::stf((bf16*)p.QeAh + ku * (CH * KD) + fofs(w, s, l), fq);
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          f32x4 c = zero4();
          mma(c, fk, ident_frag<true>(hf, r16, q));
          const float x[4] = {c[0], c[1], c[2], c[3]};
          SS::st4((bf16*)p.KeTh + ku * (CH * KD) + fofs2(2 * s + hf, w >> 1, l) + 4 * (w & 1), x);
        }
      }
    }
  }
  lds_barrier();
  // ---- row scalars: b e^Lambda, e^Lambda (first document), e^{Lend - Lambda} (last)
  const float le_h = lam_h[CH - 1], le_l = lam_l[CH - 1];
  if (w == 0) {
    const bool first = doc[l] == 0, last = doc[l] == doc[CH - 1];
    const float eL = first ? fast_exp2(lam_h[l] + lam_l[l]) : 0.f;                      // e^{Lambda_i} <= 1
    const float eK = last ? fast_exp2((le_h - lam_h[l]) + (le_l - lam_l[l])) : 0.f;     // e^{Lambda_end - Lambda_i} <= 1
    float* rs = p.rows + u * (4 * CH);
    rs[l] = bet_s[l] * eL;
    rs[CH + l] = eL;
    rs[2 * CH + l] = eK;
    rs[3 * CH + l] = fast_exp2(le_h + le_l);   // e^{Lambda_end}
  }
  // ---- A and M tiles (a, bb), bb <= a: 10 tiles dealt round-robin ------------
  bf16* g_Mh = (bf16*)p.MAh + u * TM;
  bf16* g_Ml = (bf16*)p.MAl + u * TM;
  for (int t = w; t < 10; t += 4) {
    const int a = t >= 6 ? 3 : (t >= 3 ? 2 : (t >= 1 ? 1 : 0));
    const int bb = t - a * (a + 1) / 2;
    f32x4 gk = zero4(), gq = zero4();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const F1 ka = SS::fa(Kf + fofs(a, s, l));
      const F1 kb = SS::fa(Kf + fofs(bb, s, l));
      const F1 qa = SS::fa(Qf + fofs(a, s, l));
      mma(gk, ka, kb);   // (k k^T)[16a + 4q + ii][16bb + r16]
      mma(gq, kb, qa);   // (q k^T)[16a + r16][16bb + 4q + ii]
    }
    float mv[4];
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      {
        const int i = 16 * a + 4 * q + ii, j = 16 * bb + r16;
        const float d = (lam_h[i] - lam_h[j]) + (lam_l[i] - lam_l[j]);
        const bool on = i > j && doc[i] == doc[j];
        X[i * AP + j] = on ? bet_s[i] * fast_exp2(fminf(d, 0.f)) * gk[ii] : 0.f;
        if (bb == a && (a & 1) == 0) X[i * AP + j + 16] = 0.f;
      }
      {
        const int i = 16 * a + r16, j = 16 * bb + 4 * q + ii;
        const float d = (lam_h[i] - lam_h[j]) + (lam_l[i] - lam_l[j]);
        const bool on = i >= j && doc[i] == doc[j];
        mv[ii] = on ? fast_exp2(fminf(d, 0.f)) * gq[ii] : 0.f;
      }
    }
    const int mo = tofs(a, bb >> 1, l) + 4 * (bb & 1);
    SS::st4s(g_Mh + mo, g_Ml + mo, mv);
    if (bb == a && (a & 1) == 0) {
      const float z[4] = {0.f, 0.f, 0.f, 0.f};
      SS::st4s(g_Mh + mo + 4, g_Ml + mo + 4, z);
    }
  }
  lds_barrier();
  invert_and_store<true>(X, reinterpret_cast<float*>(Kf), (bf16*)p.TAh + u * TM, (bf16*)p.TAl + u * TM, w, l);
}

// Output rows of one value head, written through a buffer resource that ends
// with the last valid token's row: lanes past it are dropped by the hardware,
// without a branch (a branch would leave the compiler unsure how many
// vector-memory operations are pending, and the waits for prefetched operands
// would then cover the stores too).
template <class TV> struct OutRows {
  TV* base;
  int rowb, ofs;
  __amdgpu_buffer_rsrc_t rs;
  __device__ __forceinline__ OutRows(const PF& p, int b, int hv, int row, int col) {
    base = (TV*)p.out + (((int64_t)b * p.L + p.t0) * p.Hv + hv) * KD;
    rowb = p.Hv * KD * (int)sizeof(TV);
    ofs = row * rowb + col * (int)sizeof(TV);
  }
  __device__ __forceinline__ void chunk(const PF& p, int c) {
    const int rows = min(CH, min(p.nt, p.L - p.t0) - c * CH);   // >= 1
    rs = __builtin_amdgcn_make_buffer_rsrc(base + (int64_t)c * CH * p.Hv * KD, (short)0,
                                           (rows - 1) * rowb + KD * (int)sizeof(TV), 0x00020000);
  }
  // columns col + dc .. + 3 of row + dr
  __device__ __forceinline__ void st(const f32x4& v, int dc, int dr = 0) const {
    if constexpr (sizeof(TV) == 4) {
      typedef unsigned u4 __attribute__((ext_vector_type(4)));
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), rs, ofs + dr * rowb + dc * 4, 0, 0);
    } else {
      typedef unsigned u2 __attribute__((ext_vector_type(2)));
      bf16x4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = (bf16)v[e];
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, x), rs, ofs + dr * rowb + dc * 2, 0, 0);
    }
  }
};

// ===========================================================================
// k_chain: the scan over chunks for NTL 16-column value tiles of one exec
// head, and each chunk's output.  One workgroup of 8 waves in two roles that
// meet at three LDS barriers per chunk:
//   waves 0-3 (recurrence): wave w owns state rows 32w..32w+31 (fp32, in
//     VGPRs) and publishes them to LDS as slab w of the S_c^T fragment (split
//     high / low bf16 in bf16 mode); after barrier 1 it forms token tile w of
//     be S and of R = w v - be S; after barrier 2 token tile w of Vn = T R;
//     after barrier 3 its state rows' ke^T Vn.
//   waves 4-7 (output): wave 4 + t computes token tile t of the chunk as
//     O^T = S^T qe^T + Vn^T M^T, beside the recurrence on the other wave slot
//     of each SIMD.
// With SC (k_prepass_sc) be, qe and ke are row scalars times k, q and k:
// be S = diag(b e^Lambda) (k S), and Vn is scaled before its product with k^T.
// The scalars are applied in fp32, so only S and Vn enter as split words.
// An operand's registers are loaded again for the next chunk as soon as their
// product is issued, in the shadow of the LDS reads that follow a barrier, so
// a load has most of a step to arrive and the loads are spread over the step
// (the output role, which has registers to spare, keeps whole sets).
// LDS fragments are read in bursts ahead of the products that use them.
// The role is a scalar (wave-uniform) branch.
// Bound by the step's six dependent products beside 110 KB of loads per CU (64
// bytes a clock): 1.5 us a chunk with 192 workgroups, 1.0 with every load taken
// out.  2048 tokens, 24 value heads 48 us, against 26 for the 128-token form's
// scan, whose prepass costs 32 more.
// ===========================================================================

// NTL: 16-column tiles per workgroup.  One tile per workgroup spreads a
// head's columns over the most CUs; when the tiles outnumber the CUs, a
// workgroup takes NTL tiles of one value head, so each chunk's operands are
// loaded once for all of them.  Index n of tile j is column NTL n + j of the
// workgroup's 16 NTL: a lane's NTL values of one row are neighbours in memory.
template <class T, int N> struct RowVec { typedef T V __attribute__((ext_vector_type(N))); };
template <class T> struct RowVec<T, 1> { typedef T V; };
template <class T, int N> __device__ __forceinline__ T row_el(const typename RowVec<T, N>::V& v, int j) {
  if constexpr (N == 1) return v; else return v[j];
}

// products of a split operand pair over two accumulators: the leading one
// and the corrections (independent chains; fp32: alternating by slab)
template <bool BF, class A, class B>
__device__ __forceinline__ void mma2(f32x4& c0, f32x4& c1, int s, const A& a, const B& b) {
  using P = Pol<BF>;
  if constexpr (!BF) {
    P::m33(s & 1 ? c1 : c0, a, b);
  } else if constexpr (std::is_same<A, typename P::F1>::value) {
    mma(c0, a, b.hi);
    mma(c1, a, b.lo);
  } else if constexpr (std::is_same<B, typename P::F1>::value) {
    mma(c0, a.hi, b);
    mma(c1, a.lo, b);
  } else {
    mma(c0, a.hi, b.hi);
    mma(c1, a.hi, b.lo);
    mma(c1, a.lo, b.hi);
  }
}

// (WCH: one write gate per value channel, not one per token -- a template
// argument so that no branch stands between the loads of the loop)
template <bool BF, bool SC, bool WCH, class TV, int NTL>
__global__ __launch_bounds__(512) void k_chain(const PF p) {
  using P = Pol<BF>;
  using F1 = typename P::F1;
  using F3 = typename P::F3;
  using SS = Store<BF>;
  using ST = typename SS::ST;
  using WV = typename RowVec<float, NTL>::V;
  constexpr int NT = 512;
  constexpr int FS = 4 * 64 * 8;   // elements of one tile's S^T fragment
  constexpr int FV = 2 * 64 * 8;   // elements of one tile's R / Vn fragment
  __shared__ __align__(16) ST Sh_s[NTL][FS], Sl_s[NTL][BF ? FS : 8];
  __shared__ __align__(16) ST Rh_s[NTL][FV], Rl_s[NTL][BF ? FV : 8];
  __shared__ __align__(16) ST Vh_s[NTL][FV], Vl_s[NTL][BF ? FV : 8];
  __shared__ __align__(16) ST Kh_s[SC ? NTL : 1][SC ? FV : 8], Kl_s[SC ? NTL : 1][SC ? FV : 8];   // Vn e^{Lend - Lambda}
  __shared__ __align__(16) float wv_s[4][NTL][64 * 4];   // w v: token tile, column tile, lane (index r16, tokens 4q..)
  __shared__ int flg[2 * kMaxBlockChunks];   // is_new_doc, all_same_doc per chunk
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, r16 = l & 15, q = l >> 4;
  int ctg, h, b;
  xcd_block(ctg, h, b);
  const int ct0 = NTL * ctg;       // first tile; the NTL tiles lie in one value head
  const int hv = p.gates_at_hv ? h : h * p.G + (16 * ct0) / KD;
  const int hk = p.gates_at_hv ? h / p.G : h;
  const int vc0 = (16 * ct0) % KD;   // first column of the tiles inside head hv
  const int t_end = min(p.t0 + p.nt, p.L);
  // chunk flags into LDS once, so testing them never waits on vector loads
  for (int i = tid; i < 2 * p.NCb; i += NT) flg[i] = p.flags[(int64_t)b * p.NCb * 2 + i];
  // unit of chunk c (clamped to the last) for the per-head operands, and for
  // the k / q operands that SC keeps once per key head
  auto unit = [&](int c) { return ((int64_t)b * p.Hx + h) * p.NCb + min(c, p.NCb - 1); };
  auto kunit = [&](int c) { return SC ? ((int64_t)b * p.Hk + hk) * p.NCb + min(c, p.NCb - 1) : unit(c); };
  auto lo_p = [](ST* hi, ST* lo) { return BF ? lo : hi; };
  auto ld_s = [&](int j, F3 (&f)[4]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int o = (s * 64 + l) * 8;
      f[s] = SS::fa3(&Sh_s[j][o], lo_p(&Sh_s[j][0], &Sl_s[j][0]) + o);
    }
  };

  if (wid < 4) {
    // ---------------- recurrence: state rows 32w.. ----------------
    // (its dependent products set the step: first in line for the LDS and for
    // load issue: 2048 tokens, 16 value heads 54.5 to 53.6 us)
    __builtin_amdgcn_s_setprio(3);
    const int w = wid;
    const int64_t sbase = ((int64_t)b * p.Hv + hv) * KD * KD + vc0 + NTL * r16;
    f32x4 S[NTL][2];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        WV x;
        if (p.has_init) x = *reinterpret_cast<const WV*>(p.init + sbase + (int64_t)(32 * w + 16 * r + 4 * q + ii) * KD);
        else x = WV{};
#pragma unroll
        for (int j = 0; j < NTL; ++j) S[j][r][ii] = row_el<float, NTL>(x, j);
      }
    using FK = std::conditional_t<SC, F1, F3>;
    F1 be[4];            // be (SC: k) rows of token tile w
    F3 tr[2];            // T rows of token tile w
    FK kt[2][2];         // ke^T (SC: k^T) state row tiles 2w, 2w + 1
    f32x4 dv[2];         // e^{Lend} of the state rows (SC: one value)
    f32x4 bl, eK;        // SC: row scalars of tokens 16w + 4q + ii
    // operands of chunk c's first product
    auto load_a = [&](int c) {
      const ST* bp = (const ST*)p.BeA + kunit(c) * (CH * KD);
      if constexpr (SC) bl = *reinterpret_cast<const f32x4*>(p.rows + unit(c) * (4 * CH) + 16 * w + 4 * q);
#pragma unroll
      for (int s = 0; s < 4; ++s) be[s] = SS::fa(bp + fofs(w, s, l));
    };
    auto load_t = [&](int c) {
      const ST* th = (const ST*)p.TAh + unit(c) * TM;
      const ST* tl = (const ST*)p.TAl + unit(c) * TM;
      // (slab 1 of T's upper row tiles is all zero and not stored)
#pragma unroll
      for (int s = 0; s < 2; ++s) tr[s] = SS::fa3(th + tofs(w, min(s, w >> 1), l), tl + tofs(w, min(s, w >> 1), l));
      if constexpr (SC) eK = *reinterpret_cast<const f32x4*>(p.rows + unit(c) * (4 * CH) + 2 * CH + 16 * w + 4 * q);
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        if constexpr (SC) dv[r] = f32x4{p.rows[unit(c) * (4 * CH) + 3 * CH], 0.f, 0.f, 0.f};
        else dv[r] = *reinterpret_cast<const f32x4*>(p.dvec + unit(c) * KD + 32 * w + 16 * r + 4 * q);
      }
    };
    auto load_k = [&](int c) {
      const ST* kh = (const ST*)p.KeTh + kunit(c) * (CH * KD);
      const ST* kl = (const ST*)p.KeTl + kunit(c) * (CH * KD);
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if constexpr (SC) kt[r][s] = SS::fa(kh + fofs2(2 * w + r, s, l));
          else kt[r][s] = SS::fa3(kh + fofs2(2 * w + r, s, l), kl + fofs2(2 * w + r, s, l));
        }
    };
    // a tile of R or Vn (lane: index r16, tokens 16w + 4q + ii) as half w & 1
    // of slab w >> 1 of the fragment
    const int vo = ((w >> 1) * 64 + l) * 8 + 4 * (w & 1);
    const int fo = (w * 64 + l) * 8;
    load_a(0);
    load_t(0);
    load_k(0);
    lds_barrier();   // the flags and chunk 0's w v
    int is_new = flg[0], same = flg[1];
#pragma unroll 1
    for (int c = 0; c < p.NCb; ++c) {
#pragma unroll
      for (int j = 0; j < NTL; ++j) {
        if (is_new) { S[j][0] = zero4(); S[j][1] = zero4(); }
        // lane (n, q) holds rows 32w + 16r + 4q + ii = element 4r + ii of slab w
        const float x[8] = {S[j][0][0], S[j][0][1], S[j][0][2], S[j][0][3],
                            S[j][1][0], S[j][1][1], S[j][1][2], S[j][1][3]};
        SS::st8s(&Sh_s[j][fo], lo_p(&Sh_s[j][0], &Sl_s[j][0]) + fo, x);
      }
      lds_barrier();   // 1
      F3 sf[2][4];
      ld_s(0, sf[0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NTL; ++j) {
        if (j + 1 < NTL) {
          ld_s(j + 1, sf[(j + 1) & 1]);
          __builtin_amdgcn_sched_barrier(0);
        }
        const f32x4 wv = *reinterpret_cast<const f32x4*>(&wv_s[w][j][4 * l]);
        f32x4 acc = zero4(), acc2 = zero4();
#pragma unroll
        for (int s = 0; s < 4; ++s) mma2<BF>(acc, acc2, s, be[s], sf[j & 1][s]);
        float x[4];
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) {
          const float ks = acc[ii] + acc2[ii];
          x[ii] = SC ? fmaf(-bl[ii], ks, wv[ii]) : wv[ii] - ks;
        }
        SS::st4s(&Rh_s[j][vo], lo_p(&Rh_s[j][0], &Rl_s[j][0]) + vo, x);
      }
      lds_barrier();   // 2
      F3 rf[NTL][2];
      auto ld_rv = [&](ST* hi, ST* lo, F3 (&f)[2]) {
#pragma unroll
        for (int s = 0; s < 2; ++s) f[s] = SS::fa3(hi + (s * 64 + l) * 8, lo_p(hi, lo) + (s * 64 + l) * 8);
      };
#pragma unroll
      for (int j = 0; j < NTL; ++j) ld_rv(Rh_s[j], Rl_s[j], rf[j]);
      __builtin_amdgcn_sched_barrier(0);
      load_a(c + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NTL; ++j) {
        f32x4 acc = zero4(), acc2 = zero4();
        mma2<BF>(acc, acc2, 0, tr[0], rf[j][0]);
        if (w >= 2) mma2<BF>(acc, acc2, 1, tr[1], rf[j][1]);
        float x[4];
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) x[ii] = acc[ii] + acc2[ii];
        SS::st4s(&Vh_s[j][vo], lo_p(&Vh_s[j][0], &Vl_s[j][0]) + vo, x);
        if constexpr (SC) {
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) x[ii] *= eK[ii];
          SS::st4s(&Kh_s[j][vo], &Kl_s[j][vo], x);
        }
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) S[j][r][ii] = same ? dv[r][SC ? 0 : ii] * S[j][r][ii] : 0.f;
      }
      lds_barrier();   // 3
#pragma unroll
      for (int j = 0; j < NTL; ++j) {
        if constexpr (SC) ld_rv(Kh_s[j], Kl_s[j], rf[j]);
        else ld_rv(Vh_s[j], Vl_s[j], rf[j]);
      }
      const int cn = min(c + 1, p.NCb - 1);
      is_new = flg[2 * cn];
      same = flg[2 * cn + 1];
      __builtin_amdgcn_sched_barrier(0);
      load_t(c + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NTL; ++j)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          f32x4 acc2 = zero4();
#pragma unroll
          for (int s = 0; s < 2; ++s) mma2<BF>(S[j][r], acc2, s, kt[r][s], rf[j][s]);
#pragma unroll
          for (int ii = 0; ii < 4; ++ii) S[j][r][ii] += acc2[ii];
        }
      load_k(c + 1);
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) {
        WV x;
#pragma unroll
        for (int j = 0; j < NTL; ++j) {
          if constexpr (NTL == 1) x = S[0][r][ii]; else x[j] = S[j][r][ii];
        }
        *reinterpret_cast<WV*>(p.fin + sbase + (int64_t)(32 * w + 16 * r + 4 * q + ii) * KD) = x;
      }
  } else {
    // ---------------- output: token tile t2, and w v for the recurrence ----------------
    const int t2 = wid - 4;
    // v and w of the chunk whose w v is formed next: lane = token 16 t2 + l / 4,
    // columns 4 NTL (l % 4) .. + 4 NTL - 1 (index n of tile j is column NTL n + j)
    const int hw = vgate_head(p, p.w_h, hv);
    const int vt = 16 * t2 + (l >> 2), vcol = 4 * NTL * (l & 3);
    const TV* vp = (const TV*)p.v + ((int64_t)b * p.L * p.Hv + hv) * KD + vc0;
    const float* wp = (const float*)p.w + ((int64_t)b * p.L * p.w_h + hw) * p.w_c + (WCH ? vc0 : 0);
    const uint32_t vs = (uint32_t)p.Hv * KD, ws = (uint32_t)p.w_h * p.w_c;
    typedef TV V4 __attribute__((ext_vector_type(4)));
    V4 v[NTL];
    f32x4 wg[WCH ? NTL : 1];
    auto load_v = [&](int c) {
      const int t0 = p.t0 + min(c, p.NCb - 1) * CH;
      const uint32_t row = min(vt, t_end - 1 - t0);   // rows past the last token read the last one
#pragma unroll
      for (int j = 0; j < NTL; ++j) v[j] = *reinterpret_cast<const V4*>(vp + t0 * (int64_t)vs + (row * vs + vcol + 4 * j));
      if constexpr (WCH) {
#pragma unroll
        for (int j = 0; j < NTL; ++j) wg[j] = *reinterpret_cast<const f32x4*>(wp + t0 * (int64_t)ws + (row * ws + vcol + 4 * j));
      } else {
        wg[0][0] = (wp + t0 * (int64_t)ws)[row * ws];
      }
    };
    auto put_wv = [&](int c) {
      const bool valid = vt <= t_end - 1 - (p.t0 + min(c, p.NCb - 1) * CH);
      float y[4 * NTL];
#pragma unroll
      for (int e = 0; e < 4 * NTL; ++e) y[e] = WCH ? wg[e / 4][e % 4] : wg[0][0];
      if (!SC && p.fuse) {
#pragma unroll
        for (int e = 0; e < 4 * NTL; ++e) y[e] = sigmoid_fast(y[e]);
      }
      // element (token 16 t2 + 4 q' + ii, index n) of a tile at word (16 q' + n) * 4 + ii
      const int o = (l >> 4) * 64 + 16 * (l & 3) + ((l >> 2) & 3);
#pragma unroll
      for (int e = 0; e < 4 * NTL; ++e) {
        const float x = y[e] * (float)v[e / 4][e % 4];
        wv_s[t2][e % NTL][o + 4 * (e / NTL)] = valid ? x : 0.f;
      }
    };
    // qe (SC: q) and M rows of the token tile, and e^Lambda of its token r16
    // (SC): loaded again for the next chunk as soon as they are used
    std::conditional_t<SC, F1, F3> qe[4];
    F3 m[2];
    float eL = 0.f;
    auto load_q = [&](int c) {
      const ST* qh = (const ST*)p.QeAh + kunit(c) * (CH * KD);
      const ST* ql = (const ST*)p.QeAl + kunit(c) * (CH * KD);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if constexpr (SC) qe[s] = SS::fa(qh + fofs(t2, s, l));
        else qe[s] = SS::fa3(qh + fofs(t2, s, l), ql + fofs(t2, s, l));
      }
      if constexpr (SC) eL = p.rows[unit(c) * (4 * CH) + CH + 16 * t2 + r16];
    };
    auto load_m = [&](int c) {
      const ST* mh = (const ST*)p.MAh + unit(c) * TM;
      const ST* ml = (const ST*)p.MAl + unit(c) * TM;
#pragma unroll
      for (int s = 0; s < 2; ++s) m[s] = SS::fa3(mh + tofs(t2, min(s, t2 >> 1), l), ml + tofs(t2, min(s, t2 >> 1), l));
    };
    // lane (t, q) holds O[token 16 t2 + t][columns NTL (4q + ii) + j]: 4 NTL
    // neighbouring columns
    OutRows<TV> orow(p, b, hv, 16 * t2 + r16, vc0 + 4 * NTL * q);
    load_v(0);
    load_q(0);
    load_m(0);
    put_wv(0);
    load_v(1);
    lds_barrier();   // the flags and chunk 0's w v
#pragma unroll 1
    for (int c = 0; c < p.NCb; ++c) {
      f32x4 res[NTL];
      lds_barrier();   // 1
      F3 sf[2][4];
      ld_s(0, sf[0]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NTL; ++j) {
        if (j + 1 < NTL) {
          ld_s(j + 1, sf[(j + 1) & 1]);
          __builtin_amdgcn_sched_barrier(0);
        }
        f32x4 acc2 = zero4();
        res[j] = zero4();
#pragma unroll
        for (int s = 0; s < 4; ++s) mma2<BF>(res[j], acc2, s, sf[j & 1][s], qe[s]);
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) res[j][ii] = SC ? (res[j][ii] + acc2[ii]) * eL : res[j][ii] + acc2[ii];
      }
      __builtin_amdgcn_sched_barrier(0);
      load_q(c + 1);
      lds_barrier();   // 2
      // (nothing of w v moves up: with one gate per token the compiler took its
      // wait for the gate above the loads of q: 16384 tokens of 17 heads, 634
      // against 555 us of scan; with a gate per channel no difference)
      if constexpr (!WCH) __builtin_amdgcn_sched_barrier(0);
      put_wv(c + 1);   // (the recurrence has read chunk c's)
      load_v(c + 2);
      lds_barrier();   // 3
      F3 vf[NTL][2];
#pragma unroll
      for (int j = 0; j < NTL; ++j)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int fs = (s * 64 + l) * 8;
          vf[j][s] = SS::fa3(&Vh_s[j][fs], lo_p(&Vh_s[j][0], &Vl_s[j][0]) + fs);
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NTL; ++j) {
        f32x4 acc2 = zero4();
        mma2<BF>(res[j], acc2, 0, vf[j][0], m[0]);
        if (t2 >= 2) mma2<BF>(res[j], acc2, 1, vf[j][1], m[1]);
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) res[j][ii] += acc2[ii];
      }
      __builtin_amdgcn_sched_barrier(0);
      load_m(c + 1);
      orow.chunk(p, c);
#pragma unroll
      for (int j4 = 0; j4 < NTL; ++j4) {
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = res[(4 * j4 + e) % NTL][(4 * j4 + e) / NTL];
        orow.st(x, 4 * j4);
      }
    }
  }
}

// ===========================================================================
// k_chain_cols: the scalar-gate scan for 64 columns of one exec head per
// workgroup.  Wave j < 4 owns column tile j with the whole state (128 rows, 32
// VGPRs): a tile's S, R and Vn never leave its registers (an accumulator tile
// pair is the next product's fragment), so a step has no exchange between
// waves and one barrier, where the split by state rows (k_chain) meets three
// times and sends S, R and Vn of every tile through LDS to all eight waves.
// Waves 4-7 copy the operands all four tiles share (k, T, k^T, q, M: 72 KB per
// chunk, fragment-native, 1 KB per instruction and no registers) from the
// workspace into the other half of a double buffer, one chunk ahead.
// Bound by the LDS reads of those operands (84 KB per wave and chunk) beside
// 132 MFMAs per wave.  chunk_gdn, 4 x 8192 tokens, 32 value heads, bf16, timed in
// turn: 434 us with the rows split, 400 us here (3.1 us a chunk against 1 us of
// MFMA issue); with every read waited for in turn, the compiler's order, 435 us.
// (Under the profiler, a dozen calls in a row: 419 to 534 us.)
// ===========================================================================
template <int N> __device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// 64 lanes x 16 bytes from src (each lane's own address) to 1 KB of LDS at dst
__device__ __forceinline__ void copy_to_lds(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

__global__ __launch_bounds__(512) void k_chain_cols(const PF p) {
  using P = Pol<true>;
  using F1 = P::F1;
  using F3 = P::F3;
  using SS = Store<true>;
  constexpr int OK = 0, OT = CH * KD, OKT = OT + 2 * TM, OQ = OKT + CH * KD, OM = OQ + CH * KD, ON = OM + 2 * TM;
  __shared__ __align__(16) bf16 ops[2][ON];
  __shared__ __align__(16) float row_s[2][4 * CH];   // b e^Lambda, e^Lambda, e^{Lend - Lambda}, e^{Lend}
  __shared__ __align__(16) float w_s[2][CH];         // write gate per token
  __shared__ uint8_t flg[kMaxBlockChunks];           // bit 0: is_new_doc, bit 1: all_same_doc
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63, r16 = l & 15, q = l >> 4;
  int ctg, h, b;
  xcd_block(ctg, h, b);
  const int hv = p.gates_at_hv ? h : h * p.G + (64 * ctg) / KD;
  const int hk = p.gates_at_hv ? h / p.G : h;
  const int NCb = p.NCb, t_end = min(p.t0 + p.nt, p.L);
  auto unit = [&](int c) { return ((int64_t)b * p.Hx + h) * NCb + min(c, NCb - 1); };

  if (wid >= 4) {
    // ---------------- loaders: fragment 4 i + w of each operand by wave w ----------------
    const int w = wid - 4;
    const float* wp = (const float*)p.w + (int64_t)b * p.L * p.w_h + vgate_head(p, p.w_h, hv);
    auto copy = [&](const bf16* src, bf16* dst, int n) {
      for (int i = w; i < n; i += 4) copy_to_lds(src + i * 512 + l * 8, dst + i * 512);
    };
    auto load = [&](int c) {
      const int64_t u = unit(c), ku = ((int64_t)b * p.Hk + hk) * NCb + min(c, NCb - 1);
      bf16* o = ops[c & 1];
      copy((const bf16*)p.BeA + ku * (CH * KD), o + OK, 16);
      copy((const bf16*)p.TAh + u * TM, o + OT, 6);
      copy((const bf16*)p.TAl + u * TM, o + OT + TM, 6);
      copy((const bf16*)p.KeTh + ku * (CH * KD), o + OKT, 16);
      copy((const bf16*)p.QeAh + ku * (CH * KD), o + OQ, 16);
      copy((const bf16*)p.MAh + u * TM, o + OM, 6);
      copy((const bf16*)p.MAl + u * TM, o + OM + TM, 6);
      if (w == 3) copy_to_lds(p.rows + u * (4 * CH) + l * 4, row_s[c & 1]);
      // (tokens past the last one read its gate)
      const int t0 = p.t0 + min(c, NCb - 1) * CH;
      if (w == 2)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(wp + min(t0 + l, t_end - 1) * (int64_t)p.w_h),
                                         (__attribute__((address_space(3))) void*)w_s[c & 1], 4, 0, 0);
    };
    load(0);
    if (NCb > 1) load(1);
    for (int i = tid - 256; i < NCb; i += 256) {
      const int32_t* f = p.flags + ((int64_t)b * NCb + i) * 2;
      flg[i] = (f[0] ? 1 : 0) | (f[1] ? 2 : 0);
    }
    wait_vm<0>();
    lds_barrier();   // chunks 0 and 1, the flags
#pragma unroll 1
    for (int c = 0; c < NCb; ++c) {
      wait_vm<0>();   // chunk c + 1 is there
      lds_barrier();  // chunk c is read
      if (c + 2 < NCb) load(c + 2);
    }
  } else {
    // ---------------- column tile j = wid ----------------
    const int vc0 = (64 * ctg) % KD + 16 * wid;   // first column of the tile inside head hv
    const int64_t sbase = ((int64_t)b * p.Hv + hv) * KD * KD + vc0 + r16;
    f32x4 S[8];   // lane (n, q): column n, state rows 16m + 4q + ii
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) S[m][ii] = p.has_init ? p.init[sbase + (int64_t)(16 * m + 4 * q + ii) * KD] : 0.f;
    OutRows<bf16> orow(p, b, hv, r16, vc0 + 4 * q);
    // v of (token 16rt + 4q + ii, this lane's column) of the next chunk, zero
    // past the last token: the resource ends with its row, and the whole row
    // offset is in the lane's own offset (the scalar one takes no part in the
    // bounds check)
    const bf16* vb = (const bf16*)p.v + (((int64_t)b * p.L + p.t0) * p.Hv + hv) * KD;
    const int rowb = p.Hv * KD * 2, vofs = 4 * q * rowb + (vc0 + r16) * 2;
    uint16_t v[4][4];
    auto load_v = [&](int c) {
      const int cc = min(c, NCb - 1), rows = min(CH, t_end - (p.t0 + cc * CH));
      const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(vb) + (int64_t)cc * CH * p.Hv * KD, (short)0,
                                                        (rows - 1) * rowb + KD * 2, 0x00020000);
#pragma unroll
      for (int rt = 0; rt < NB; ++rt)
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) v[rt][ii] = __builtin_amdgcn_raw_buffer_load_b16(rs, vofs + (16 * rt + ii) * rowb, 0, 0);
    };
    load_v(0);
    lds_barrier();   // chunks 0 and 1, the flags
#pragma unroll 1
    for (int c = 0; c < NCb; ++c) {
      const bf16* o = ops[c & 1];
      const float* rw = row_s[c & 1];
      const int f = __builtin_amdgcn_readfirstlane(flg[c]);
      const float* ws = w_s[c & 1];
      if (f & 1) {
#pragma unroll
        for (int m = 0; m < 8; ++m) S[m] = zero4();
      }
      F3 sf[4];   // S^T fragments: slab s = state rows 32s..
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const float x[8] = {S[2 * s][0], S[2 * s][1], S[2 * s][2], S[2 * s][3],
                            S[2 * s + 1][0], S[2 * s + 1][1], S[2 * s + 1][2], S[2 * s + 1][3]};
        sf[s] = P::f3(x);
      }
      // The shared operands go through three buffers of four fragments, each
      // read two groups of products ahead of its use (the compiler's own order
      // waits for every read: 3.4 us a chunk).
      F1 fa[4], fb[4], fc[4];
      auto ld = [&](F1 (&f)[4], int o0, int o1, int o2, int o3) {
        f[0] = SS::fa(o + o0);
        f[1] = SS::fa(o + o1);
        f[2] = SS::fa(o + o2);
        f[3] = SS::fa(o + o3);
        __builtin_amdgcn_sched_barrier(0);
      };
      auto ld_k = [&](F1 (&f)[4], int rt) { ld(f, OK + fofs(rt, 0, l), OK + fofs(rt, 1, l), OK + fofs(rt, 2, l), OK + fofs(rt, 3, l)); };
      auto ld_q = [&](F1 (&f)[4], int rt) { ld(f, OQ + fofs(rt, 0, l), OQ + fofs(rt, 1, l), OQ + fofs(rt, 2, l), OQ + fofs(rt, 3, l)); };
      // rows 0 and 1 of a triangular operand (one slab each), or row rt >= 2 (two slabs): high, low
      auto ld_01 = [&](F1 (&f)[4], int b0) { ld(f, b0 + tofs(0, 0, l), b0 + TM + tofs(0, 0, l), b0 + tofs(1, 0, l), b0 + TM + tofs(1, 0, l)); };
      auto ld_rt = [&](F1 (&f)[4], int b0, int rt) { ld(f, b0 + tofs(rt, 0, l), b0 + TM + tofs(rt, 0, l), b0 + tofs(rt, 1, l), b0 + TM + tofs(rt, 1, l)); };
      auto ld_kt = [&](F1 (&f)[4], int m) { ld(f, OKT + fofs2(m, 0, l), OKT + fofs2(m, 1, l), OKT + fofs2(m + 1, 0, l), OKT + fofs2(m + 1, 1, l)); };
      auto done = [] { __builtin_amdgcn_sched_barrier(0); };

      f32x4 R[4];
      // R[rt] = w v - b e^Lambda (k S)
      auto prod_k = [&](int rt, const F1 (&f)[4]) {
        const f32x4 ww = *reinterpret_cast<const f32x4*>(&ws[16 * rt + 4 * q]);
        const f32x4 bl = *reinterpret_cast<const f32x4*>(&rw[16 * rt + 4 * q]);
        f32x4 a = zero4(), a2 = zero4();
#pragma unroll
        for (int t = 0; t < 4; ++t) mma2<true>(a, a2, t, f[t], sf[t]);
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) R[rt][ii] = fmaf(-bl[ii], a[ii] + a2[ii], ww[ii] * __builtin_bit_cast(float, (uint32_t)v[rt][ii] << 16));
        done();
      };
      auto frag = [&](const f32x4& x0, const f32x4& x1) {
        const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        return P::f3(x);
      };
      F3 rf[2], vf[2], kf[2];
      // Vn = T R, and Vn e^{Lend - Lambda}
      f32x4 Vt[2], Kt[2];
      auto prod_t = [&](int rt, const F1& h0, const F1& l0, const F1& h1, const F1& l1) {
        const f32x4 eK = *reinterpret_cast<const f32x4*>(&rw[2 * CH + 16 * rt + 4 * q]);
        f32x4 a = zero4(), a2 = zero4();
        mma2<true>(a, a2, 0, F3{h0, l0}, rf[0]);
        if (rt >= 2) mma2<true>(a, a2, 1, F3{h1, l1}, rf[1]);
        Vt[rt & 1] = a + a2;
        Kt[rt & 1] = Vt[rt & 1] * eK;
        if (rt & 1) {
          vf[rt >> 1] = frag(Vt[0], Vt[1]);
          kf[rt >> 1] = frag(Kt[0], Kt[1]);
        }
      };
      // S = [same doc] e^{Lend} S + k^T (Vn e^{Lend - Lambda})
      const float dv = (f & 2) ? rw[3 * CH] : 0.f;
      if (!(f & 2)) {
#pragma unroll
        for (int m = 0; m < 8; ++m) S[m] = zero4();   // (sf holds this chunk's; 0 * inf is not 0)
      }
      // (two rows of tiles at a time: their chains interleave)
      auto prod_kt = [&](int m, const F1 (&x)[4]) {
        f32x4 a = dv * S[m], b = dv * S[m + 1];
        mma(a, x[0], kf[0].hi);
        mma(b, x[2], kf[0].hi);
        mma(a, x[0], kf[0].lo);
        mma(b, x[2], kf[0].lo);
        mma(a, x[1], kf[1].hi);
        mma(b, x[3], kf[1].hi);
        mma(a, x[1], kf[1].lo);
        mma(b, x[3], kf[1].lo);
        S[m] = a;
        S[m + 1] = b;
        done();
      };
      // O^T = e^Lambda (S^T q^T) + Vn^T M^T: lane (t, q) holds token 16rt + t,
      // columns 4q + ii of the tile
      f32x4 O[4];
      auto prod_q = [&](int rt, const F1 (&f)[4]) {
        const float eL = rw[CH + 16 * rt + r16];
        f32x4 a = zero4(), a2 = zero4();
#pragma unroll
        for (int t = 0; t < 4; ++t) mma2<true>(a, a2, t, sf[t], f[t]);
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) O[rt][ii] = (a[ii] + a2[ii]) * eL;
        done();
      };
      auto prod_m = [&](int rt, const F1& h0, const F1& l0, const F1& h1, const F1& l1) {
        f32x4 a2 = zero4();
        mma2<true>(O[rt], a2, 0, vf[0], F3{h0, l0});
        if (rt >= 2) mma2<true>(O[rt], a2, 1, vf[1], F3{h1, l1});
        orow.st(O[rt] + a2, 0, 16 * rt);
      };
      orow.chunk(p, c);
      ld_k(fa, 0);
      ld_k(fb, 1);
      ld_k(fc, 2);
      prod_k(0, fa);
      ld_k(fa, 3);
      prod_k(1, fb);
      ld_01(fb, OT);
      rf[0] = frag(R[0], R[1]);
      prod_k(2, fc);
      ld_rt(fc, OT, 2);
      prod_k(3, fa);
      load_v(c + 1);
      ld_rt(fa, OT, 3);
      rf[1] = frag(R[2], R[3]);
      prod_t(0, fb[0], fb[1], fb[0], fb[1]);
      prod_t(1, fb[2], fb[3], fb[2], fb[3]);
      done();
      ld_q(fb, 0);
      prod_t(2, fc[0], fc[1], fc[2], fc[3]);
      done();
      ld_kt(fc, 0);
      prod_t(3, fa[0], fa[1], fa[2], fa[3]);
      done();
      ld_kt(fa, 2);
      prod_q(0, fb);   // (fills the latency of Vn's last tile)
      ld_kt(fb, 4);
      prod_kt(0, fc);
      ld_kt(fc, 6);
      prod_kt(2, fa);
      ld_q(fa, 1);
      prod_kt(4, fb);
      ld_q(fb, 2);
      prod_kt(6, fc);
      ld_q(fc, 3);
      prod_q(1, fa);
      ld_01(fa, OM);
      prod_q(2, fb);
      ld_rt(fb, OM, 2);
      prod_q(3, fc);
      ld_rt(fc, OM, 3);
      prod_m(0, fa[0], fa[1], fa[0], fa[1]);
      prod_m(1, fa[2], fa[3], fa[2], fa[3]);
      prod_m(2, fb[0], fb[1], fb[2], fb[3]);
      prod_m(3, fc[0], fc[1], fc[2], fc[3]);
      lds_barrier();   // chunk c is read
    }
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) p.fin[sbase + (int64_t)(16 * m + 4 * q + ii) * KD] = S[m][ii];
  }
}

// ===========================================================================
// host side
// ===========================================================================
namespace {

struct WsLayout {
  size_t flags, dvec, rows, BeA, QeAh, QeAl, KeTh, KeTl, TAh, TAl, MAh, MAl, lng, carry, total;
};

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// How a call is run: chunks of 64 tokens with their operands applied in the
// scan (kScan, with scalar gates kScalar), or the 128-token affine form of
// dn_prefill_long.hip.
enum Form { kScan, kScalar, kLong };
int chunk_of(Form f) { return f == kLong ? 128 : CH; }

// Split operands have a low-word array in bf16 mode only.  With scalar gates
// the k, q and k^T operands are kept once per key head, as single words.
WsLayout ws_layout(const dn_prefill_args* a, int Hx, int Vp, int NCb, Form form) {
  WsLayout L{};
  const bool bf = a->precision == 0, sc = form == kScalar;
  const size_t es = bf ? 2 : 4;
  const size_t ls = bf ? 2 : 0;
  const size_t units = (size_t)a->B * Hx * NCb;
  const size_t kunits = sc ? (size_t)a->B * a->Hk * NCb : units;
  const size_t sq = (size_t)CH * KD;
  size_t off = 0;
  auto take = [&](size_t bytes) { size_t o = off; off += align256(bytes); return o; };
  L.flags = take((size_t)a->B * NCb * 2 * 4);
  L.dvec = take(units * KD * 4);
  if (form == kLong) {
    L.lng = take(long_workspace(units, Vp, bf));
  } else {
    L.rows = take(sc ? units * 4 * CH * 4 : 0);
    L.BeA = take(kunits * sq * es);
    L.QeAh = take(kunits * sq * es);
    L.QeAl = take(sc ? 0 : kunits * sq * ls);
    L.KeTh = take(kunits * sq * es);
    L.KeTl = take(sc ? 0 : kunits * sq * ls);
    L.TAh = take(units * TM * es);
    L.TAl = take(units * TM * ls);
    L.MAh = take(units * TM * es);
    L.MAl = take(units * TM * ls);
  }
  L.carry = take((size_t)a->B * a->Hv * KD * KD * 4);
  L.total = off;
  return L;
}

// Workspace budget of one call (token blocks beyond it run one after another).
// Larger blocks mean fewer launches and longer chains per launch: chunk_gdn of 4
// sequences of 8192 tokens (32 value heads) runs in one launch pair, and so does
// each 8192-token block of a streamed sequence; with the 128-token form a 160 MiB
// budget cost 10% and 32% there, and smaller budgets cost with this one too.
constexpr size_t kAutoBudget = size_t(4096) << 20;

// 128-token blocks per token block: block_tokens when given, else the most
// that keep the workspace within kAutoBudget.  A hard budget (the
// allocation-free entry point's scratch) also caps a given block_tokens.
int block_128s(const dn_prefill_args* a, int Hx, int Vp, Form form, size_t budget = 0) {
  const int R = 128 / chunk_of(form);
  int n = std::min((a->nt + 127) / 128, kMaxBlockChunks / R);
  if (a->block_tokens > 0) {
    n = std::max(1, std::min(n, a->block_tokens / 128));
    if (budget == 0) return n;
  }
  if (budget == 0) budget = kAutoBudget;
  while (n > 1 && ws_layout(a, Hx, Vp, n * R, form).total > budget) n = (n + 1) / 2;
  return n;
}

int check_args(const dn_prefill_args* a) {
  if (a == nullptr) return set_error(DN_E_INVALID, "null args");
  if (a->abi_version != DN_ABI_VERSION) return set_error(DN_E_ABI, "dn_prefill_args built for another ABI version");
  if (a->K != KD || a->V != KD) return set_error(DN_E_INVALID, "K and V must both be 128");
  if (a->B <= 0 || a->L <= 0 || a->Hk <= 0 || a->Hv <= 0) return set_error(DN_E_INVALID, "non-positive dimension");
  if (a->Hv % a->Hk != 0) return set_error(DN_E_INVALID, "Hv must be a multiple of Hk");
  if (a->t0 < 0 || a->t0 % 128 != 0 || a->nt <= 0 || a->t0 + a->nt > a->L)
    return set_error(DN_E_INVALID, "token range must satisfy 0 <= t0 < t0+nt <= L with t0 % 128 == 0");
  if (!a->q || !a->k || !a->v || !a->g || !a->b || !a->w || !a->out)
    return set_error(DN_E_INVALID, "missing tensor pointer");
  if (a->qk_dtype < DN_F32 || a->qk_dtype > DN_F16)
    return set_error(DN_E_INVALID, "q/k dtype must be f32, bf16 or f16");
  if (a->v_dtype != DN_F32 && a->v_dtype != DN_BF16)
    return set_error(DN_E_INVALID, "v dtype must be f32 or bf16");
  const int G = a->Hv / a->Hk;
  auto gate_ok = [&](int H, int Cc, int dt, int full) {
    return (H == 1 || H == a->Hk || H == a->Hv) && (Cc == 1 || Cc == full) && dt == DN_F32;
  };
  if (!gate_ok(a->g_heads, a->g_chans, a->g_dtype, a->K) || !gate_ok(a->b_heads, a->b_chans, a->b_dtype, a->K) ||
      !gate_ok(a->w_heads, a->w_chans, a->w_dtype, a->V))
    return set_error(DN_E_INVALID, "gates must be float32 with 1, Hk or Hv heads and 1 or 128 channels");
  if (!a->gates_at_hv && G > 1 && (a->g_heads == a->Hv || a->b_heads == a->Hv))
    return set_error(DN_E_INVALID, "g or b has Hv heads: gates_at_hv must be set");
  if (a->seg && a->seg_dtype != DN_I32 && a->seg_dtype != DN_I64) return set_error(DN_E_INVALID, "segment ids must be int32 or int64");
  if (a->precision != 0 && a->precision != 1) return set_error(DN_E_INVALID, "precision must be 0 (bf16) or 1 (fp32)");
  if (a->block_tokens < 0 || a->block_tokens % 128 != 0) return set_error(DN_E_INVALID, "block_tokens must be a multiple of 128");
  return DN_OK;
}

int g_chain_tiles = -1;   // -1: unread; 0: by grid size; 1, 2, 4: forced (DN_CHAIN_TILES, measurements)
int chain_tiles() {
  if (g_chain_tiles < 0) {
    const char* e = getenv("DN_CHAIN_TILES");
    const int v = e ? atoi(e) : 0;
    g_chain_tiles = (v == 1 || v == 2 || v == 4) ? v : 0;
  }
  return g_chain_tiles;
}

int g_prepass_scalar = -1;   // -1: unread; 0: general path forced (DN_PREPASS_SCALAR=0, measurements)
bool prepass_scalar() {
  if (g_prepass_scalar < 0) {
    const char* e = getenv("DN_PREPASS_SCALAR");
    g_prepass_scalar = (e && atoi(e) == 0) ? 0 : 1;
  }
  return g_prepass_scalar == 1;
}

// One decay, one b and one w per (token, head) with bf16 q / k in precision
// "bf16" (the Gated DeltaNet form) runs the scalar-gate kernels.
bool scalar_gates(const dn_prefill_args* a) {
  return prepass_scalar() && a->precision == 0 && a->qk_dtype == DN_BF16 && a->g_chans == 1 && a->b_chans == 1 &&
         a->w_chans == 1 && !a->fuse_prologue;
}

// The long form where its scan, half the steps of 1.4 us against 1.1-1.3 us
// each, outweighs its prepass.  That prepass runs one workgroup per CU, so it
// costs whole rounds of 256 units (head, 128 tokens), 30 us with scalar gates
// and 40-60 with channel-wise ones: at one round the line is a length, at more
// rounds only long sequences of few heads are left.  Both forms measured, long
// form's time / scan's:
//   one round: channel gates, 1 value head per head 2560 tokens 1.00-1.04,
//     3072 0.94-0.99; 2 value heads 3072 0.99-1.04, 4096 0.88-0.93 (8 heads
//     1.04); 4 value heads 4096 1.06-1.13, 6144 0.92-0.97 (4 heads 1.03 at
//     5120); fp32 2560 1.06, 3584 0.92 / 3584 1.02, 5120 0.88 / 5120 1.04,
//     6144 0.97; scalar 4608 1.02, 6144 0.95 (6 heads 1.03 at 5120) / 6144
//     0.95-1.01 / 8192 0.97-1.00
//   more: channel gates 5-8 heads 6144 tokens 1.00-1.16, 8192 0.90-1.13,
//     12288 0.93-1.07; 10-13 heads 8192 1.02-1.26, 12288 0.91-1.01 (4 value
//     heads: 12288 1.00-1.12, 16384 0.93-0.99); 16 heads from 12288 0.98-1.06,
//     17 and more 1.00-1.4.  fp32 6-8 heads 6144 1.01-1.28, 8192 0.91-1.09,
//     16384 0.87-1.00; 11 heads and more 1.03-1.5.
//   scalar gates, more: 1-2 heads 0.74-1.00 throughout; 3-4 heads in the second
//     round 12288 0.99-1.04, 16384 0.92-0.95, 4 heads in the third 1.06 and 5 to
//     12 heads 1.0-1.8; from 1536 units, where the scan's operands no longer fit
//     the 256 MB cache, 3-5 heads 0.88-0.96, 6 heads 0.98-1.02, 7 and more
//     1.00-1.2.
// `width` = heads (5 + 2 G) weighs a head with its G value heads.
Form form_of(const dn_prefill_args* a) {
  const bool sc = scalar_gates(a), bf = a->precision == 0;
  const int64_t G = a->gates_at_hv ? 1 : a->Hv / a->Hk;
  const int64_t heads = (int64_t)a->B * (a->gates_at_hv ? a->Hv : a->Hk);
  const int64_t width = heads * (5 + 2 * G);
  const int64_t units = heads * ((a->nt + 127) / 128), rounds = (units + 255) / 256;
  bool lng;
  if (sc) {
    const bool most = rounds == 1 ? width <= 40
                                  : (rounds == 2 && a->nt >= 16384 && width <= 28 && G <= 2) || (units >= 1536 && width <= 45);
    lng = a->nt >= 4096 + 1024 * G && (width <= 14 || most);
  } else if (rounds == 1) {
    lng = width <= (G <= 2 ? 70 : 40) && a->nt >= 2048 + (bf ? 768 : 1024) * G;
  } else if (width <= 56 && G <= 2) {
    lng = a->nt >= 8192;
  } else {
    lng = width <= (bf ? 112 : 75) && a->nt >= (bf && G <= 2 ? 12288 : 16384);
  }
  if (lng) return kLong;
  return sc ? kScalar : kScan;
}

template <bool BF, bool SC, class TV>
void launch_chain(const PF& p, hipStream_t st) {
  // several column tiles per workgroup once the tiles outnumber the CUs: with
  // scalar gates at four, each wave its own (k_chain_cols)
  const int tiles = (p.Vp / 16) * p.Hx * p.B;
  int ntl = chain_tiles();
  if (ntl == 0) ntl = tiles > 2 * 256 ? 4 : (tiles > 256 ? 2 : 1);
  if (!BF) ntl = 1;
  const dim3 grid(p.Vp / (16 * ntl), p.Hx, p.B), blk(512);
  if constexpr (SC && std::is_same<TV, bf16>::value) {
    if (ntl == 4) {
      hipLaunchKernelGGL(k_chain_cols, grid, blk, 0, st, p);
      return;
    }
  }
  auto go = [&](auto wch) {
    constexpr bool W = decltype(wch)::value;
    if constexpr (BF) {
      if constexpr (!(SC && std::is_same<TV, bf16>::value))
        if (ntl == 4) hipLaunchKernelGGL((k_chain<BF, SC, W, TV, 4>), grid, blk, 0, st, p);
      if (ntl == 2) hipLaunchKernelGGL((k_chain<BF, SC, W, TV, 2>), grid, blk, 0, st, p);
    }
    if (ntl == 1) hipLaunchKernelGGL((k_chain<BF, SC, W, TV, 1>), grid, blk, 0, st, p);
  };
  if constexpr (!SC) {
    if (p.w_c != 1) go(std::true_type{});
    else go(std::false_type{});
  } else {
    go(std::false_type{});
  }
}

template <bool BF, class TIn>
hipError_t launch_all(const PF& p, hipStream_t st, bool v_bf16, bool sc) {
  prof_mark(0, st, false);
  if constexpr (BF && std::is_same<TIn, bf16>::value) {
    if (sc) hipLaunchKernelGGL((k_prepass_sc<TIn>), dim3(p.B * p.Hx * p.NCb), dim3(256), 0, st, p);
  }
  if (!sc) hipLaunchKernelGGL((k_prepass<BF, TIn>), dim3(p.B * p.Hx * p.NCb), dim3(256), 0, st, p);
  prof_mark(0, st, true);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  prof_mark(2, st, false);
  if constexpr (BF && std::is_same<TIn, bf16>::value) {
    if (sc) v_bf16 ? launch_chain<BF, true, bf16>(p, st) : launch_chain<BF, true, float>(p, st);
  }
  if (!sc) v_bf16 ? launch_chain<BF, false, bf16>(p, st) : launch_chain<BF, false, float>(p, st);
  prof_mark(2, st, true);
  return hipGetLastError();
}

template <bool BF>
hipError_t dispatch_qk(const PF& p, hipStream_t st, int qk_dt, bool v_bf16, bool sc) {
  if (qk_dt == DN_BF16) return launch_all<BF, bf16>(p, st, v_bf16, sc);
  if (qk_dt == DN_F16) return launch_all<BF, f16>(p, st, v_bf16, sc);
  return launch_all<BF, float>(p, st, v_bf16, sc);
}

hipError_t dispatch(const PF& p, hipStream_t st, bool bf, int qk_dt, bool v_bf16, bool sc) {
  return bf ? dispatch_qk<true>(p, st, qk_dt, v_bf16, sc) : dispatch_qk<false>(p, st, qk_dt, v_bf16, sc);
}

}  // namespace

}  // namespace dn

using namespace dn;

extern "C" size_t dn_prefill_workspace_size(const dn_prefill_args* a) {
  if (check_args(a) != DN_OK) return 0;
  const int Hx = a->gates_at_hv ? a->Hv : a->Hk;
  const int Vp = a->gates_at_hv ? KD : (a->Hv / a->Hk) * KD;
  const Form form = form_of(a);
  return ws_layout(a, Hx, Vp, block_128s(a, Hx, Vp, form) * (128 / chunk_of(form)), form).total;
}

namespace {

// One dn_prefill_fwd call in token blocks of n 128-token blocks over the workspace ws.
int prefill_run(const dn_prefill_args* a, char* ws, size_t workspace_bytes, int n, Form form, hipStream_t st) {
  const int G = a->Hv / a->Hk;
  const int Hx = a->gates_at_hv ? a->Hv : a->Hk;
  const int Vp = a->gates_at_hv ? KD : G * KD;
  const bool bf = a->precision == 0;
  const int ch = chunk_of(form);
  const WsLayout Lw = ws_layout(a, Hx, Vp, n * (128 / ch), form);
  if (ws == nullptr || workspace_bytes < Lw.total) return set_error(DN_E_WORKSPACE, "workspace too small");

  PF p{};
  p.B = a->B; p.L = a->L; p.Hk = a->Hk; p.Hv = a->Hv; p.G = G; p.Hx = Hx; p.Vp = Vp;
  p.gates_at_hv = a->gates_at_hv;
  p.q = a->q; p.k = a->k; p.v = a->v; p.v_dt = a->v_dtype;
  p.g = a->g; p.g_dt = a->g_dtype; p.g_h = a->g_heads; p.g_c = a->g_chans;
  p.b = a->b; p.b_dt = a->b_dtype; p.b_h = a->b_heads; p.b_c = a->b_chans;
  p.w = a->w; p.w_dt = a->w_dtype; p.w_h = a->w_heads; p.w_c = a->w_chans;
  p.seg = a->seg; p.seg_dt = a->seg_dtype; p.seg_batched = a->seg_batched;
  p.init_seg = a->init_seg;
  p.out = a->out;
  p.scale = a->scale; p.l2norm = a->qk_l2norm; p.fuse = a->fuse_prologue; p.guard = a->stability_guard;
  p.flags = (int32_t*)(ws + Lw.flags);
  p.dvec = (float*)(ws + Lw.dvec);
  p.rows = (float*)(ws + Lw.rows);
  p.BeA = ws + Lw.BeA;
  p.QeAh = ws + Lw.QeAh;
  p.QeAl = bf ? ws + Lw.QeAl : p.QeAh;
  p.KeTh = ws + Lw.KeTh;
  p.KeTl = bf ? ws + Lw.KeTl : p.KeTh;
  p.TAh = ws + Lw.TAh;
  p.TAl = bf ? ws + Lw.TAl : p.TAh;
  p.MAh = ws + Lw.MAh;
  p.MAl = bf ? ws + Lw.MAl : p.MAh;
  float* carry = a->final_state ? a->final_state : (float*)(ws + Lw.carry);

  const int t_stop = a->t0 + a->nt;
  for (int tb = a->t0; tb < t_stop; tb += n * 128) {
    p.t0 = tb;
    p.nt = std::min(n * 128, t_stop - tb);
    p.NCb = (p.nt + ch - 1) / ch;
    const bool first = tb == a->t0;
    p.has_init = first ? (a->init_state != nullptr) : 1;
    p.init = first ? a->init_state : carry;
    p.fin = carry;
    const bool v_bf16 = a->v_dtype == DN_BF16;
    const hipError_t e = form == kLong ? long_prefill(p, ws + Lw.lng, st, bf, a->qk_dtype, v_bf16, prepass_scalar())
                                       : dispatch(p, st, bf, a->qk_dtype, v_bf16, form == kScalar);
    if (e != hipSuccess) return set_error(DN_E_LAUNCH, hipGetErrorString(e));
  }
  return DN_OK;
}

int prefill_shape_ok(const dn_prefill_args* a) {
  const int rc = check_args(a);
  if (rc != DN_OK) return rc;
  const int G = a->Hv / a->Hk;
  const int Vp = a->gates_at_hv ? KD : G * KD;
  if (Vp % 64 != 0 || Vp > 1024) return set_error(DN_E_INVALID, "value width per execution head must be 64..1024");
  return DN_OK;
}

}  // namespace

extern "C" int dn_prefill_fwd(const dn_prefill_args* a, void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = prefill_shape_ok(a);
  if (rc != DN_OK) return rc;
  const int Hx = a->gates_at_hv ? a->Hv : a->Hk;
  const int Vp = a->gates_at_hv ? KD : (a->Hv / a->Hk) * KD;
  const Form form = form_of(a);
  return prefill_run(a, (char*)workspace, workspace_bytes, block_128s(a, Hx, Vp, form), form, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------
// Allocation-free prefill: dn_prefill_fwd over a file-scope device scratch
// array instead of a caller workspace.  Each GPU holds its own copy of
// `scratch` (DN_NOALLOC_SCRATCH_BYTES) from the library's first use on it
// until the process ends.  Host code never passes the array's name to a
// kernel (on the host it is only a stand-in for the symbol): the device
// address comes from hipGetSymbolAddress, taken once per device with that
// device current, and is the only handle used afterwards.
// ---------------------------------------------------------------------------
namespace {

static __device__ __align__(256) char scratch[DN_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
char* g_scratch_ptr[kMaxDevices] = {};

// the current device's address of `scratch` (nullptr and an error set on failure)
char* scratch_address() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error(DN_E_LAUNCH, "no current HIP device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || ptr == nullptr) {
      set_error(DN_E_LAUNCH, e != hipSuccess ? hipGetErrorString(e) : "null scratch address");
      return nullptr;
    }
    g_scratch_ptr[dev] = (char*)ptr;
  }
  return g_scratch_ptr[dev];
}

}  // namespace

extern "C" int dn_prefill_fwd_noalloc(const dn_prefill_args* a, void* stream) {
  const int rc = prefill_shape_ok(a);
  if (rc != DN_OK) return rc;
  const int Hx = a->gates_at_hv ? a->Hv : a->Hk;
  const int Vp = a->gates_at_hv ? KD : (a->Hv / a->Hk) * KD;
  const Form form = form_of(a);
  const int n = block_128s(a, Hx, Vp, form, DN_NOALLOC_SCRATCH_BYTES);
  if (ws_layout(a, Hx, Vp, n * (128 / chunk_of(form)), form).total > DN_NOALLOC_SCRATCH_BYTES)
    return set_error(DN_E_WORKSPACE,
                     "dn_prefill_fwd_noalloc: one 128-token block of every (batch, head) needs more than "
                     "DN_NOALLOC_SCRATCH_BYTES of scratch; use dn_prefill_fwd with a workspace");
  char* ws = scratch_address();
  if (ws == nullptr) return DN_E_LAUNCH;
  return prefill_run(a, ws, DN_NOALLOC_SCRATCH_BYTES, n, form, (hipStream_t)stream);
}
