// attn_abi.hip -- extern "C" entry points of libmetalllm_attn.so (declared in
// include/metalllm_attn.h). Validation happens on the host before any HIP call, so argument
// errors are reported without touching the device.
#include <cmath>

#include "../../include/metalllm_attn.h"
#include "attn_launch.hpp"
#include "overlap.hpp"

namespace {

int validate(const AttentionParams* p) {
  if (!p) return METALLLM_ATTN_E_NULL;
  if (p->M == 0 || p->M % 64) return METALLLM_ATTN_E_SEQLEN;
  if (p->D != 64 && p->D != 128) return METALLLM_ATTN_E_HEADDIM;
  if (p->NH == 0 || p->B == 0 || (uint64_t)p->N != (uint64_t)p->NH * p->D) return METALLLM_ATTN_E_LAYOUT;
  if ((uint64_t)p->B * p->M * p->N >= (1ull << 31)) return METALLLM_ATTN_E_SIZE;
  return METALLLM_ATTN_OK;
}

bool aligned16(const void* ptr) { return ((uintptr_t)ptr & 15u) == 0; }

float head_scale(uint32_t D) { return 1.0f / std::sqrt((float)D); }  // attention.metal:109,268

// Kernels of a backward entry point (metalllmAttnBackwardRoute's values).
enum Route { kFused = 0, kJoint = 1, kTwo = 2, kStored = 3 };

// acc: flashAttentionBackward, else flashAttentionBackwardWorkspace. An output may lie in the memory of
// an input that the kernels after the one writing it do not read, where that one reads an element
// only in the workgroup that replaces it: dV in v's (and in the fused kernel, which keeps a pair's K in
// LDS, dK in k's); dQ, written from the stored dS and k alone, in those of q, v and dZ. In the joint
// launch dQ's workgroups may read any input after dK's and dV's have ended, so it takes outputs apart
// from the inputs only. The kernels for the others follow from D and T alone, so that a caller can
// plan for them.
Route backward_route(const mla::BwdArgs& a, int D, bool acc) {
  const size_t e = (size_t)a.B * a.T * a.H * D, stat = (size_t)a.B * a.H * a.T;
  const bool apart = !mla::any_overlap({{a.dQ, 4 * e}, {a.dK, 2 * e}, {a.dV, 2 * e}},
                                       {{a.dO, 2 * e}, {a.Dv, 4 * stat}, {a.lse, 4 * stat}, {a.q, 2 * e}, {a.k, 2 * e}, {a.v, 2 * e}});
  const int pairs = a.B * a.H;
  if (!apart) return D == 64 && a.T <= 256 ? kFused : (acc || D == 64) ? kTwo : kStored;
  if (mla::backward_is_short(a.T, D, pairs)) return kFused;
  return acc || mla::workspace_recomputes(a.T, D, pairs) ? kJoint : kStored;
}

// One part of a backward entry point (metalllmAttnBackwardPart), or with `whole` the entry point
// whose first part it is (0: flashAttentionBackward, 2: flashAttentionBackwardWorkspace).
int backward(int part, const uint16_t* dZ, const float* d, const float* l, const uint16_t* q, const uint16_t* k,
             const uint16_t* v, float* dQ, uint16_t* dK, uint16_t* dV, void* workspace, uint64_t workspace_bytes,
             const AttentionParams* p, metalllm_stream_t stream, bool whole) {
  const int rc = validate(p);
  if (rc) return rc;
  if (part < 0 || part > 3) return METALLLM_ATTN_E_LAYOUT;
  if (!dZ || !d || !l || !q || !k || !v || !dQ || !dK || !dV) return METALLLM_ATTN_E_NULL;
  if (!aligned16(dZ) || !aligned16(d) || !aligned16(l) || !aligned16(q) || !aligned16(k) || !aligned16(v) ||
      !aligned16(dQ) || !aligned16(dK) || !aligned16(dV))
    return METALLLM_ATTN_E_ALIGN;
  const int D = (int)p->D;
  const hipStream_t s = (hipStream_t)stream;
  mla::BwdArgs a{dZ, d, l, q, k, v, dQ, dK, dV, (int)p->M, (int)p->NH, (int)p->B, head_scale(p->D)};
  const bool acc = part < 2;  // parts 0 and 1 add into dQ, 2 and 3 write it
  if (!acc) {
    if (!workspace) return METALLLM_ATTN_E_NULL;
    if (!aligned16(workspace)) return METALLLM_ATTN_E_ALIGN;
    if (workspace_bytes < (uint64_t)mla::ds_scratch_bytes(a.B, a.H, a.T)) return METALLLM_ATTN_E_SIZE;
  }
  const bool first = part == 0 || part == 2;
  hipError_t e = hipSuccess;
  switch (backward_route(a, D, acc)) {
    case kFused:  // one kernel computes dK, dV and dQ; the second part has nothing left to do
      if (first) e = mla::launch_backward_short(a, acc, s);
      break;
    case kJoint:
      if (whole) {
        e = mla::launch_backward_both(a, D, acc, s);
        break;
      }
      [[fallthrough]];
    case kTwo:  // dK/dV, then dQ
      if (first) e = mla::launch_backward(a, D, s);
      if (e == hipSuccess && (whole || !first)) e = mla::launch_backward_dq(a, D, acc, s);
      break;
    case kStored:  // dK/dV storing dS into the workspace, then dQ = dS.K
      a.dS = (uint16_t*)workspace;
      if (first) e = mla::launch_backward(a, D, s);
      if (e == hipSuccess && (whole || !first)) e = mla::launch_backward_dqs(a, D, s);
      break;
  }
  return e == hipSuccess ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LAUNCH;
}

}  // namespace

extern "C" {

int flashAttentionForward(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* out, float* l,
                          const AttentionParams* p, metalllm_stream_t stream) {
  const int rc = validate(p);
  if (rc) return rc;
  if (!q || !k || !v || !out || !l) return METALLLM_ATTN_E_NULL;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out) || !aligned16(l))
    return METALLLM_ATTN_E_ALIGN;
  mla::FwdArgs a{q, k, v, out, l, (int)p->M, (int)p->NH, (int)p->B, head_scale(p->D)};
  return mla::launch_forward(a, (int)p->D, (hipStream_t)stream) == hipSuccess ? METALLLM_ATTN_OK
                                                                               : METALLLM_ATTN_E_LAUNCH;
}

int computeD(const uint16_t* dO, const uint16_t* O, float* D, const AttentionParams* p, metalllm_stream_t stream) {
  const int rc = validate(p);
  if (rc) return rc;
  if (!dO || !O || !D) return METALLLM_ATTN_E_NULL;
  if (!aligned16(dO) || !aligned16(O) || !aligned16(D)) return METALLLM_ATTN_E_ALIGN;
  mla::ComputeDArgs a{dO, O, D, (int)p->M, (int)p->NH, (int)p->B};
  return mla::launch_compute_d(a, (int)p->D, (hipStream_t)stream) == hipSuccess ? METALLLM_ATTN_OK
                                                                                : METALLLM_ATTN_E_LAUNCH;
}

int metalllmAttnBackwardWorkspaceSize(const AttentionParams* p, uint64_t* bytes) {
  const int rc = validate(p);
  if (rc) return rc;
  if (!bytes) return METALLLM_ATTN_E_NULL;
  *bytes = (uint64_t)mla::ds_scratch_bytes((int)p->B, (int)p->NH, (int)p->M);
  return METALLLM_ATTN_OK;
}

int metalllmAttnBackwardPart(int part, const uint16_t* dZ, const float* d, const float* l, const uint16_t* q,
                             const uint16_t* k, const uint16_t* v, float* dQ, uint16_t* dK, uint16_t* dV,
                             void* workspace, uint64_t workspace_bytes, const AttentionParams* p,
                             metalllm_stream_t stream) {
  return backward(part, dZ, d, l, q, k, v, dQ, dK, dV, workspace, workspace_bytes, p, stream, false);
}

int flashAttentionBackward(const uint16_t* dZ, const float* d, const float* l, const uint16_t* q,
                           const uint16_t* k, const uint16_t* v, float* dQ, uint16_t* dK, uint16_t* dV,
                           const AttentionParams* p, metalllm_stream_t stream) {
  return backward(0, dZ, d, l, q, k, v, dQ, dK, dV, nullptr, 0, p, stream, true);
}

int flashAttentionBackwardWorkspace(const uint16_t* dZ, const float* d, const float* l, const uint16_t* q,
                                    const uint16_t* k, const uint16_t* v, float* dQ, uint16_t* dK, uint16_t* dV,
                                    void* workspace, uint64_t workspace_bytes, const AttentionParams* p,
                                    metalllm_stream_t stream) {
  return backward(2, dZ, d, l, q, k, v, dQ, dK, dV, workspace, workspace_bytes, p, stream, true);
}

int metalllmAttnBackwardRoute(int workspace, const uint16_t* dZ, const float* d, const float* l, const uint16_t* q,
                              const uint16_t* k, const uint16_t* v, float* dQ, uint16_t* dK, uint16_t* dV,
                              const AttentionParams* p) {
  const int rc = validate(p);
  if (rc) return rc;
  const mla::BwdArgs a{dZ, d, l, q, k, v, dQ, dK, dV, (int)p->M, (int)p->NH, (int)p->B, 0.0f};
  return backward_route(a, (int)p->D, workspace == 0);
}

const char* metalllmAttnErrorString(int code) {
  switch (code) {
    case METALLLM_ATTN_OK: return "ok";
    case METALLLM_ATTN_E_NULL: return "a required pointer is NULL";
    case METALLLM_ATTN_E_SEQLEN: return "sequence length M must be a positive multiple of 64";
    case METALLLM_ATTN_E_HEADDIM: return "head size D must be 64 or 128";
    case METALLLM_ATTN_E_LAYOUT: return "N must equal NH*D with NH >= 1 and B >= 1";
    case METALLLM_ATTN_E_SIZE: return "a tensor exceeds 2^31 elements";
    case METALLLM_ATTN_E_ALIGN: return "tensor pointers must be 16-byte aligned";
    case METALLLM_ATTN_E_LAUNCH: return "kernel launch failed";
    case METALLLM_ATTN_E_LIBRARY: return "platform library call (rocBLAS, device allocation) failed";
    case METALLLM_ATTN_E_CAPTURE: return "scratch would grow during stream capture (call metalllmSublayerReserve first)";
    default: return "unknown error";
  }
}

int metalllmAttnWorkMap(int kind, const AttentionParams* p, int32_t* out, int32_t count) {
  const int rc = validate(p);
  if (rc) return rc;
  if (!out && count > 0) return METALLLM_ATTN_E_NULL;
  if (kind < 0 || kind > 2) return METALLLM_ATTN_E_LAYOUT;
  const int npairs = (int)(p->B * p->NH);
  const int blk = kind == 0 ? mla::kFwdBlockM : kind == 1 ? mla::kBwdBlockN : mla::kDqBlockM;
  const int nblk = ((int)p->M + blk - 1) / blk;
  const int grid = npairs * nblk;
  for (int i = 0; i < count && i < grid; ++i) {
    int pair, b;
    const int round = kind == 0 ? mla::kFwdDispatchRound : mla::bwd_dispatch_round((int)p->D);
    mla::decode_workgroup(i, npairs, nblk, kind != 1, round, pair, b);
    out[2 * i] = pair;
    out[2 * i + 1] = b;
  }
  return grid;
}

int metalllmAttnForwardItems(const AttentionParams* p, int32_t grid, int32_t* out, int32_t count) {
  const int rc = validate(p);
  if (rc) return rc;
  if (grid <= 0) return METALLLM_ATTN_E_LAYOUT;
  if (!out && count > 0) return METALLLM_ATTN_E_NULL;
  const int npairs = (int)(p->B * p->NH);
  const int nblk = ((int)p->M + mla::kFwdBlockM - 1) / mla::kFwdBlockM;
  int n = 0;
  for (int w = 0; w < grid; ++w) {
    int pair, blk;
    for (int k = 0; mla::fwd_item_of(w, grid, k, npairs, nblk, pair, blk); ++k, ++n) {
      if (n < count) {
        out[3 * n] = w;
        out[3 * n + 1] = pair;
        out[3 * n + 2] = blk;
      }
    }
  }
  return n;
}

}  // extern "C"
