// Host-side declarations shared by the kernel translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "deltanet_amd.h"

namespace dn {

// Kernel parameter block of one prefill token block (passed by value).
struct PF {
  int B, L, Hk, Hv, G;       // tensor dims, G = Hv / Hk
  int Hx, Vp, gates_at_hv;   // execution heads, value width per execution head
  int t0, nt, NCb;           // token block [t0, t0+nt), chunks in the block
  const void *q, *k, *v;
  int v_dt;
  const void* g; int g_dt, g_h, g_c;
  const void* b; int b_dt, b_h, b_c;
  const void* w; int w_dt, w_h, w_c;
  const void* seg; int seg_dt, seg_batched;
  const float* init; int has_init;
  const int32_t* init_seg;
  void* out;
  float* fin;
  float scale; int l2norm, fuse, guard;
  // workspace arrays (one unit = one (batch, exec head, chunk))
  int32_t* flags;            // [B][NCb][2] : is_new_doc, all_same_doc
  float* dvec;               // [unit][K]    : e^{Lambda_end}
  float* rows;               // [unit][4][64]: b e^Lambda, e^Lambda, e^{Lend - Lambda}, e^{Lend} per token (scalar gates)
  // Workspace, per unit = (batch, exec head, chunk).  Every operand array is
  // fragment-native for its consumer ([tile][slab][lane][8] elements of a
  // 16 x 32 MFMA operand slab).  Split operands have a high and a low array
  // (bf16 mode; in fp32 mode the low pointer aliases the high one).  "ST" =
  // bf16 in bf16 mode, fp32 in fp32 mode.  With scalar gates BeA, QeAh and
  // KeTh hold the normalised k, q and k^T, one unit per key head.
  void* BeA;                 // [4][4] ST : b k e^Lambda, rows = token, first document
  void *QeAh, *QeAl;         // [4][4] ST : q e^Lambda, rows = token, first document
  void *KeTh, *KeTl;         // [8][2] ST : (k e^{Lend - Lambda})^T, rows = key channel, last document
  void *TAh, *TAl;           // [6] ST : T, rows = token (the six slabs that are not all zero)
  void *MAh, *MAl;           // [6] ST : M, rows = token, slabs as T
};

// The 128-token affine form (dn_prefill_long.hip): its workspace for `units`
// (batch, exec head, 128-token chunk) units of value width Vp, and one token
// block over it (p's flags, dvec and 128-token NCb set), one decay and one b per
// token as plain products if `scalar_phases`.
size_t long_workspace(size_t units, int Vp, bool bf);
hipError_t long_prefill(const PF& p, char* ws, hipStream_t st, bool bf, int qk_dt, bool v_bf16, bool scalar_phases);

// Records the message for dn_last_error() and returns `code`.
int set_error(int code, const char* msg);

// Kernel timing (dn_profile_begin / dn_profile_end): returns true when the
// calling thread is profiling; mark() records an event for `kind` on `st`
// (call it once before and once after each launch).
bool profiling();
void prof_mark(int kind, hipStream_t st, bool after);

}  // namespace dn
