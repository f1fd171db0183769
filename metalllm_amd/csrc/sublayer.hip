// sublayer.hip -- the GEMMs of metalLLM's attention sublayer around the attention core, as extern "C"
// entry points with the reference kernels' names and buffer order (declared in
// include/metalllm_attn.h):
//   computeQKV      attention.metal:19-53   Q,K,V = X.Wq, X.Wk, X.Wv                       (bf16)
//   projForward     attention.metal:385-405 out = O.Wp                                    (bf16)
//   projBackwarddW  attention.metal:407-430 dWp += O^T.dZ                       (bf16, accumulated)
//   projBackwarddX  attention.metal:432-455 dO = dZ.Wp^T                                   (bf16)
//   computeGradDx   attention.metal:301-341 dX += dQ.Wq^T + dK.Wk^T + dV.Wv^T   (fp32, accumulated)
//   computeGradDw   attention.metal:343-383 dWq += X^T.dQ (fp32), dWk += X^T.dK, dWv += X^T.dV (bf16)
// Row-major matrices: X, O, dZ, Q, K, V, dK, dV bf16 [R, C] and dQ, dX fp32 [R, C] with R = B*M rows
// and C = N = NH*D features; weights bf16 [C, C] indexed [input feature][output feature].
//
// Small products, and those whose row or feature counts fit no 128-wide tile, run hand-written kernels
// on 64 x 64 tiles (sublayer_tile.hip; the rules below say which). The other bf16 GEMMs run on the
// platform library: rocBLAS gemm_ex with bf16 operands, fp32 accumulation and a bf16 or fp32
// destination (beta = 1 for the reference's multiply_accumulate kernels: the destination is read once
// and the sum rounded once). computeGradDx and computeGradDw read the fp32 dQ, which the library
// cannot take as is: larger ones whose row and feature counts are multiples of 128 run hand-written
// kernels on 128-wide tiles (sublayer_gemm.hip). Both kinds split dQ in registers into two bf16
// terms, dQ = hi + lo + O(2^-16 |dQ|), each product running on both; what is left (feature counts that
// are no multiple of 64) writes the same split to memory (split_dq) and the library runs each product
// twice. Either way the fp32 dQ never makes a bf16 round trip.
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "../../include/metalllm_attn.h"
#include "attn_launch.hpp"
#include "overlap.hpp"
#include "sublayer_tile.hpp"

namespace mla {  // glue.hip
hipError_t launch_block_ln_bwd(const float* dX, const uint16_t* dOut, const uint16_t* xnorm, const uint16_t* gamma,
                               const float* stdev, uint16_t* dStream, float* dgamma, float* dbeta, uint32_t rows,
                               uint32_t cols, hipStream_t s);
}  // namespace mla

namespace mla {  // sublayer_gemm.hip
bool grad_dx_fused_ok(int R, int C);
hipError_t launch_grad_dx(float* dX, const float* dQ, const uint16_t* dK, const uint16_t* dV, const uint16_t* Wq,
                          const uint16_t* Wk, const uint16_t* Wv, int R, int C, bool accumulate, hipStream_t s);
bool grad_dw_fused_ok(int R, int C);
size_t grad_dw_partial_floats(int R, int C);
hipError_t launch_grad_dw(const uint16_t* X, const float* dQ, const uint16_t* dK, const uint16_t* dV, float* dQw,
                          uint16_t* dKw, uint16_t* dVw, float* partial, int R, int C, bool accumulate, hipStream_t s);
size_t grad_dw_one_partial_floats(int R, int C);
hipError_t launch_grad_dw_one(const uint16_t* X, const uint16_t* G, uint16_t* dW, float* partial, int R, int C,
                              bool accumulate, hipStream_t s);
size_t grad_dw4_partial_floats(int R, int C);
hipError_t launch_grad_dxdw4(float* dX, const uint16_t* X, const float* dQ, const uint16_t* dK, const uint16_t* dV,
                             const uint16_t* Wq, const uint16_t* Wk, const uint16_t* Wv, const uint16_t* Xp,
                             const uint16_t* Gp, float* dQw, uint16_t* dKw, uint16_t* dVw, uint16_t* dPw, float* partial,
                             int R, int C, hipStream_t s);
}  // namespace mla

namespace {

int validate_gemm(const AttentionParams* p) {
  if (!p) return METALLLM_ATTN_E_NULL;
  if (p->M == 0) return METALLLM_ATTN_E_SEQLEN;
  if (p->NH == 0 || p->B == 0 || p->D == 0 || (uint64_t)p->N != (uint64_t)p->NH * p->D || p->N % 8)
    return METALLLM_ATTN_E_LAYOUT;  // rows of 16-byte multiples
  if ((uint64_t)p->B * p->M * p->N >= (1ull << 31) || (uint64_t)p->N * p->N >= (1ull << 31)) return METALLLM_ATTN_E_SIZE;
  return METALLLM_ATTN_OK;
}

bool aligned16(const void* ptr) { return ((uintptr_t)ptr & 15u) == 0; }

// Per-device library state: the rocBLAS handle (created on first use with that device current),
// the bf16 split of dQ and the fp32 partials of the weight gradients (grown on demand). A mutex
// per device serialises the host side of a call (stream binding and enqueue); the buffers are
// shared, so computeGradDx, computeGradDw and projBackwarddW calls on different streams of one
// device must not overlap.
struct DeviceState {
  std::mutex mu;
  rocblas_handle handle = nullptr;
  uint16_t* split = nullptr;  // hi [R*C] then lo [R*C]
  size_t split_elems = 0;
  float* partial = nullptr;   // fp32 partial products of the weight gradients [parts][C][C]
  size_t partial_elems = 0;
  uint8_t* attn_ws = nullptr;  // the attention backward's dS tiles (metalllmSublayerEncode)
  size_t attn_ws_bytes = 0;
};

// Grows a per-device buffer (never shrinks). Growing synchronises the device (the old buffer may
// still be in use by work enqueued on any stream) and allocates, so it is refused while `stream`
// is being captured into a graph: metalllmSublayerReserve sizes the buffers ahead of time.
template <typename T>
int ensure(T*& buf, size_t& have, size_t need, hipStream_t stream) {
  if (have >= need) return METALLLM_ATTN_OK;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &cap) != hipSuccess) return METALLLM_ATTN_E_LIBRARY;
  if (cap != hipStreamCaptureStatusNone) return METALLLM_ATTN_E_CAPTURE;
  if (buf) {
    if (hipDeviceSynchronize() != hipSuccess || hipFree(buf) != hipSuccess) return METALLLM_ATTN_E_LIBRARY;
    buf = nullptr;
    have = 0;
  }
  if (hipMalloc((void**)&buf, need * sizeof(T)) != hipSuccess) {
    buf = nullptr;
    return METALLLM_ATTN_E_LIBRARY;
  }
  have = need;
  return METALLLM_ATTN_OK;
}

DeviceState& state(int dev) {
  static std::mutex table_mu;
  static std::vector<DeviceState*> table;
  std::lock_guard<std::mutex> g(table_mu);
  if ((int)table.size() <= dev) table.resize(dev + 1, nullptr);
  if (!table[dev]) table[dev] = new DeviceState();  // lives until the process ends
  return *table[dev];
}

// Locks the current device's state and binds its handle to `stream`; null handle on failure.
struct Session {
  std::unique_lock<std::mutex> lock;
  DeviceState* st = nullptr;
  int rc = METALLLM_ATTN_OK;

  explicit Session(hipStream_t stream) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
      rc = METALLLM_ATTN_E_LIBRARY;
      return;
    }
    st = &state(dev);
    lock = std::unique_lock<std::mutex>(st->mu);
    if (!st->handle && rocblas_create_handle(&st->handle) != rocblas_status_success) {
      st->handle = nullptr;
      rc = METALLLM_ATTN_E_LIBRARY;
      return;
    }
    if (rocblas_set_stream(st->handle, stream) != rocblas_status_success) rc = METALLLM_ATTN_E_LIBRARY;
  }
};

// Where a sequence of GEMMs and helper kernels goes: the rocBLAS handle (already bound to
// `stream`) and the stream. With `query` set, nothing is launched: rocBLAS calls only report the
// device workspace they need (rocblas_start_device_memory_size_query is active on the handle).
struct Ctx {
  rocblas_handle h = nullptr;
  hipStream_t stream = nullptr;
  bool query = false;
};

bool blas_ok(const Ctx& c, rocblas_status s) {
  return s == rocblas_status_success ||
         (c.query && (s == rocblas_status_size_increased || s == rocblas_status_size_unchanged));
}

// Row-major C[M][N] = op(A)[M][K] . op(B)[K][N] + beta * C. op(A) = A stored [M][K] (lda) or, with
// ta, A^T of A stored [K][M]; likewise op(B). rocBLAS is column-major: the row-major product is
// computed as C^T = op(B)^T . op(A)^T on the same memory.
int gemm_rm(const Ctx& c, bool ta, bool tb, int M, int N, int K, const void* A, rocblas_datatype at, int lda,
            const void* B, rocblas_datatype bt, int ldb, float beta, void* C, rocblas_datatype ct, int ldc) {
  const float alpha = 1.0f;
  const rocblas_status s = rocblas_gemm_ex(
      c.h, tb ? rocblas_operation_transpose : rocblas_operation_none, ta ? rocblas_operation_transpose : rocblas_operation_none,
      N, M, K, &alpha, B, bt, ldb, A, at, lda, &beta, C, ct, ldc, C, ct, ldc, rocblas_datatype_f32_r,
      rocblas_gemm_algo_standard, 0, 0);
  return blas_ok(c, s) ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LIBRARY;
}

constexpr rocblas_datatype BF = rocblas_datatype_bf16_r;
constexpr rocblas_datatype F32 = rocblas_datatype_f32_r;

__device__ __forceinline__ uint16_t rne_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);  // finite inputs
}

// hi = bf16(x), lo = bf16(x - hi): four elements per thread (16-byte loads).
__global__ void __launch_bounds__(256) split_kernel(const float4* __restrict__ x, uint2* __restrict__ hi,
                                                    uint2* __restrict__ lo, size_t n4) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n4; i += (size_t)gridDim.x * blockDim.x) {
    const float4 v = x[i];
    const float f[4] = {v.x, v.y, v.z, v.w};
    uint16_t h[4], l[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      h[j] = rne_bf16(f[j]);
      l[j] = rne_bf16(f[j] - __uint_as_float((uint32_t)h[j] << 16));
    }
    hi[i] = uint2{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
    lo[i] = uint2{(uint32_t)l[0] | ((uint32_t)l[1] << 16), (uint32_t)l[2] | ((uint32_t)l[3] << 16)};
  }
}

// Writes hi = bf16(dQ), lo = bf16(dQ - hi) into split[0 .. elems) and split[elems .. 2 elems).
int split_dq(const Ctx& c, const float* dQ, size_t elems, uint16_t* split) {
  if (c.query) return METALLLM_ATTN_OK;
  const size_t n4 = elems / 4;  // C is a multiple of 8 (validate_gemm)
  const unsigned blocks = (unsigned)std::min<size_t>((n4 + 255) / 256, 65536);
  hipLaunchKernelGGL(split_kernel, dim3(blocks), dim3(256), 0, c.stream, (const float4*)dQ, (uint2*)split,
                     (uint2*)(split + elems), n4);
  return hipGetLastError() == hipSuccess ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LAUNCH;
}

// Whether the 64 x 64 tile kernels (sublayer_tile.hip) take a product: up to large sizes where the
// 128-wide kernels (sublayer_gemm.hip) and the library's large tiles do not fit, else small ones, which
// they run in fewer and shorter dependent steps. Device times in us, tile kernel against library or
// 128-wide kernel, launches queued ahead of the host.
//
// Row products, by units of 64 x 64 x 64. A library call also costs 16-21 us of host time, these
// launches about 3, which a program that calls one after another pays: the lines for C in multiples of
// 128 lie where the device loses 1-2 us at most and such a program still gains (C = 768, eager:
// projForward R = 4096 11.4 / 16.3; computeQKV R = 1024 11.7 / 16.5, but R = 2048 17.9 / 16.5).
//   computeQKV, against the library's one batched call 7000 units: C = 768 R = 640 (4320) 8.1 / 9.4, 1024 (6912)
//     12.0 / 10.9, 1536 (10368) 15.0 / 13.2, 2048 (13824) 19.1 / 16.0 (14000 against three calls, which take
//     the time of three projections: 26); C = 384 R = 2432 (4104) 9.3 / 9.2,
//     4096 (6912) 13.5 / 12.5; C = 1024 R = 512 (6144) 13.1 / 11.1, 1024 (12288) 20.2 / 14.6
//   projForward, 10500 units and 1024 tiles (few features: short sums, the copies of x bound): C = 768 R =
//     3840 (8640) 11.9 / 13.5, 4480 (10080) 13.9 / 12.4, 6144 (13824) 17.4 / 13.9; C = 256 R = 7936 (496
//     tiles) 5.5 / 7.2, 16000 (1000) 9.2 / 8.6, 28032 (1752) 15.2 / 11.1. With the encoder's residual add,
//     which saves a pass over the rows, a phase is level at 1152 tiles (C = 384 R = 12288, C = 512 R = 9216)
//   projBackwarddX, 7000 units and 768 tiles: C = 768 R = 2432 (5472) 8.3 / 8.4, 3072 (6912) 11.3 / 9.5,
//     4480 (10080) 13.8 / 11.0; C = 384 R = 3584 (336 tiles) 5.9 / 6.7, 7168 (672) 9.1 / 7.6. With computeD,
//     the phase is level at 768 tiles (C = 768 R = 4096 123.1 / 124.4) and loses 4 us at 960
//   other multiples of 64: computeQKV wins at 320-704 features nearly throughout (C = 448 6976 rows 23 /
//     45, 27008 79 / 92), not far beyond 12000 units from 768 on (C = 960 R = 768 15.0 / 15.9, 1536 24.7 /
//     19.9; C = 1216 R = 448 13.6 / 13.9, 960 24.9 / 19.2), nor 16000 below 256 (C = 192 R = 37952 36.9 /
//     39.6, 56896 51 / 41). The projections: below 256 features 16000 units (C = 192 R = 113792 36.6 / 54,
//     170688 52 / 39); from 768 on 20000 (C = 960 R = 4544 19.4 / 18.9, 12800 44 / 29; C = 1216 R = 4224 24.2 /
//     26.1); between, alone within 10% either way on the mean of the sizes (C = 448 R = 58752 59 / 62, C =
//     576 18944 32 / 21, 25280 39 / 46), and in the encoder, whose results are the entry points' bit for
//     bit, ahead by the pass saved (16384 x 448, 4 bytes an element: about 8 us)
// Gradient products:
//   computeGradDx, the dX + dW launch: C = 768 R = 2048 23 / 52, 2944 34 / 52, 6144 52 / 54, 8192 64 / 57
//     (with the weights break-even at 3072); C = 384 12160 33 / 34, 16384 38 / 35; C = 448 14912 46 / 92. With
//     few features its tiles bound it, 1500 of them: C = 256 R = 23296 (1456) 30.3 / 30.2, 27392 (1712)
//     35.0 / 31.7; C = 128 R = 32896 (1028) 19.0 / 19.7, 54912 (1716) 26.2 / 22.5
//   computeGradDw: C = 768 R = 2944 32 / 36, 4096 44 / 41; C = 512 6784 32.9 / 33.0; up to 384 features,
//     where 192 divides them, C = 384 24320 56 / 66, else C = 256 38400 42.7 / 43.1, 54912 54.5 / 52.1; C =
//     448 R = 14912 48 / 125
//   projBackwarddW: C = 768 R = 5632 23 / 25, 8064 28.6 / 28.0, 16384 41 / 38; C = 384 R = 27648 26 / 28, 32512
//     31 / 29; C = 1024 R = 4480 21 / 28; C = 448 R = 29888 33 / 41
enum Rows { kQkvBatched, kQkv, kProjForward, kProjBackward };
bool tile_rows_ok(int R, int C, Rows what) {
  if (C % 64) return false;
  const int64_t tiles = (int64_t)((R + 63) / 64) * (C / 64) * (what <= kQkv ? 3 : 1), units = tiles * (C / 64);
  const bool wide = C % 128 == 0;
  switch (what) {
    case kQkv: return units <= (wide ? 14000 : 64000);
    case kQkvBatched: return units <= (wide ? 7000 : C < 256 ? 16000 : C < 768 ? 64000 : 12000);
    case kProjForward:
      if (wide) return units <= 10500 && tiles <= 1024;
      break;
    case kProjBackward:
      if (wide) return units <= 7000 && tiles <= 768;
  }
  return units <= (C < 256 ? 16000 : C < 768 ? 64000 : 20000);
}
bool small_product(int R, int C, double limit) { return (double)R * C * C <= limit; }
constexpr double kTileBeforeLibrary = 3e10;
bool tile_dx_ok(int R, int C) {
  if (!mla::grad_dx_fused_ok(R, C)) return C % 64 == 0 && small_product(R, C, kTileBeforeLibrary);
  return small_product(R, C, 1.8e9) && (int64_t)(R / 64) * (C / 64) <= 1500;
}
bool tile_dw_ok(int R, int C) {  // computeGradDw
  const double limit = !mla::grad_dw_fused_ok(R, C) ? kTileBeforeLibrary : C > 384 ? 1.8e9 : C % 192 ? 2.6e9 : 3.6e9;
  return C % 64 == 0 && R % 64 == 0 && small_product(R, C, limit);
}
bool tile_dw_one_ok(int R, int C) {  // projBackwarddW
  return C % 64 == 0 && R % 64 == 0 && small_product(R, C, mla::grad_dw_fused_ok(R, C) ? 4.8e9 : kTileBeforeLibrary);
}
// the phase encoder's launch of computeGradDx and the four weight gradients: where the entry point
// takes them for dX, whose sums are then the same
bool tile_dxdw_ok(int R, int C) { return R % 64 == 0 && tile_dx_ok(R, C); }

// n bf16 or fp32 elements
mla::Span span(const uint16_t* p, size_t n) { return {p, 2 * n}; }
mla::Span span(const float* p, size_t n) { return {p, 4 * n}; }

// Whether the products' destinations are apart from each other and from what any of the products
// reads. The tile kernels need that: their workgroups, of one product or of several in one launch,
// read operands while others store. The calls in turn, which they replace, do not always: the library
// path of the gradient products reads the fp32 dQ once, into its split, before anything is written,
// adds dKw and dVw one after the other, and writes a weight gradient when its sums are complete.
bool qkv_apart(const uint16_t* X, const uint16_t* q, const uint16_t* k, const uint16_t* v, const uint16_t* q_w,
               const uint16_t* k_w, const uint16_t* v_w, int R, int C) {
  const size_t e = (size_t)R * C, w = (size_t)C * C;
  return !mla::any_overlap({span(q, e), span(k, e), span(v, e)}) &&
         !mla::any_overlap({span(q, e), span(k, e), span(v, e)}, {span(X, e), span(q_w, w), span(k_w, w), span(v_w, w)});
}
bool rows_apart(const uint16_t* x, const uint16_t* w, const uint16_t* y, int R, int C) {
  const size_t e = (size_t)R * C;
  return !mla::any_overlap({span(y, e)}, {span(x, e), span(w, (size_t)C * C)});
}
bool proj_dw_apart(const uint16_t* attn_out, const uint16_t* dZ, const uint16_t* dProjw, int R, int C) {
  const size_t e = (size_t)R * C;
  return !mla::any_overlap({span(dProjw, (size_t)C * C)}, {span(attn_out, e), span(dZ, e)});
}
bool grad_dx_apart(const float* dX, const uint16_t* qw, const uint16_t* kw, const uint16_t* vw, const float* dQ,
                   const uint16_t* dK, const uint16_t* dV, int R, int C) {
  const size_t e = (size_t)R * C, w = (size_t)C * C;
  return !mla::any_overlap({span(dX, e)}, {span(dQ, e), span(dK, e), span(dV, e), span(qw, w), span(kw, w), span(vw, w)});
}
bool grad_dw_apart(const uint16_t* x, const float* dQ, const uint16_t* dK, const uint16_t* dV, const float* dQw,
                   const uint16_t* dKw, const uint16_t* dVw, int R, int C) {
  const size_t e = (size_t)R * C, w = (size_t)C * C;
  return !mla::any_overlap({span(dQw, w), span(dKw, w), span(dVw, w)}) &&
         !mla::any_overlap({span(dQw, w), span(dKw, w), span(dVw, w)}, {span(x, e), span(dQ, e), span(dK, e), span(dV, e)});
}

int tile_rows(const Ctx& c, const mla::TileRows& a, bool wt) {
  if (c.query) return METALLLM_ATTN_OK;
  return mla::launch_tile_rows(a, wt, c.stream) == hipSuccess ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LAUNCH;
}

int tile_grad(const Ctx& c, const mla::TileGrad& a, float* partial, bool accumulate) {
  if (c.query) return METALLLM_ATTN_OK;
  return mla::launch_tile_grad(a, partial, accumulate, c.stream) == hipSuccess ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LAUNCH;
}

// Weight gradients W[k][n] += sum_r X[r][k] G[r][n] reduce over all R rows into a small C x C
// output: one GEMM gives the library too few output tiles for the chip. The rows are split into
// `parts` chunks, computed as one strided-batched GEMM into fp32 partials [chunk][C][C], and
// reduce_kernel adds the partials (of one or more such products) and the destination's previous
// value once, then rounds to the destination type.
int row_chunks(int R) {
  for (int s : {16, 8, 4, 2})
    if (R % s == 0 && R / s >= 512) return s;
  return 1;
}

// Elements of the dQ split (hi, then lo) that the library paths of computeGradDx (dx) and
// computeGradDw read: none where the hand-written kernels take the shape (they split in registers).
// `tiles`: the buffers allow the tile kernels (the *_apart conditions).
size_t split_need(int R, int C, bool dx, bool tiles) {
  const bool ok = dx ? (tiles && tile_dx_ok(R, C)) || mla::grad_dx_fused_ok(R, C)
                     : (tiles && tile_dw_ok(R, C)) || mla::grad_dw_fused_ok(R, C);
  return ok ? 0 : 2 * (size_t)R * C;
}

// fp32 partial floats for projBackwarddW, computeGradDw and the encoder's launch: the hand-written
// kernels' chunks, or row_chunks(R) products of C x C (twice that for computeGradDw's dQw) on the
// library path.
size_t partial_need(int R, int C, bool tiles) {
  const size_t tile = C % 64 || R % 64 ? 0
                                       : std::max({mla::tile_grad_partial_floats(R, C, 3, 4, false),
                                                   mla::tile_grad_partial_floats(R, C, 0, 3, false),
                                                   mla::tile_grad_partial_floats(R, C, 0, 4, true)});
  if (tiles && tile_dw_one_ok(R, C) && tile_dw_ok(R, C) && tile_dxdw_ok(R, C)) return tile;
  if (mla::grad_dw_fused_ok(R, C))
    return std::max({tile, mla::grad_dw_one_partial_floats(R, C), mla::grad_dw_partial_floats(R, C),
                     mla::grad_dw4_partial_floats(R, C)});
  return std::max(tile, 2 * (size_t)row_chunks(R) * C * C);
}

// For any buffers, apart or not (partial_need without tiles covers both).
size_t any_split_need(int R, int C) { return std::max(split_need(R, C, true, false), split_need(R, C, false, false)); }

// The most that a call of at most R rows and C features can need of either buffer, whichever kernels
// it runs: a smaller shape may take the 64-wide tiles, whose row chunks grow as C shrinks, the 128-wide
// ones, or the library, where a larger one does not.
size_t split_bound(int R, int C) { return 2 * (size_t)R * C; }
size_t partial_bound(int R, int C) {
  int parts = 1;  // row_chunks of some row count up to R
  while (parts < 16 && R >= 512 * 2 * parts) parts *= 2;
  size_t n = 2 * (size_t)parts * C * C;
  for (int c = 64; c <= C; c += 64) {
    n = std::max({n, mla::tile_grad_partial_bound(R, c, 3, 4, false), mla::tile_grad_partial_bound(R, c, 0, 3, false),
                  mla::tile_grad_partial_bound(R, c, 0, 4, true)});
    if (c % 128 == 0)  // chunks follow the rows up to a limit
      n = std::max({n, mla::grad_dw_one_partial_floats(R, c), mla::grad_dw_partial_floats(R, c), mla::grad_dw4_partial_floats(R, c)});
  }
  return n;
}

// Grows a buffer to `most`, or, where the device has no room for that, to `need`.
template <typename T>
int reserve(T*& buf, size_t& have, size_t most, size_t need) {
  if (have >= most) return METALLLM_ATTN_OK;
  T* grown = nullptr;
  if (hipMalloc((void**)&grown, most * sizeof(T)) != hipSuccess) {
    (void)hipGetLastError();  // not the next launch's error
    return ensure(buf, have, need, nullptr);
  }
  if (buf && (hipDeviceSynchronize() != hipSuccess || hipFree(buf) != hipSuccess)) {
    (void)hipFree(grown);
    return METALLLM_ATTN_E_LIBRARY;
  }
  buf = grown;
  have = most;
  return METALLLM_ATTN_OK;
}

int xt_g_partials(const Ctx& c, const uint16_t* X, const uint16_t* G, int R, int C, int parts, float* out) {
  const float alpha = 1.0f, beta = 0.0f;
  const int Rs = R / parts;
  // row-major out_s[C][C] = X_s^T . G_s; column-major: out_s^T = G_s^T . X_s
  const rocblas_status st = rocblas_gemm_strided_batched_ex(
      c.h, rocblas_operation_none, rocblas_operation_transpose, C, C, Rs, &alpha, G, BF, C, (rocblas_stride)Rs * C, X,
      BF, C, (rocblas_stride)Rs * C, &beta, out, F32, C, (rocblas_stride)C * C, out, F32, C, (rocblas_stride)C * C,
      parts, rocblas_datatype_f32_r, rocblas_gemm_algo_standard, 0, 0);
  return blas_ok(c, st) ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LIBRARY;
}

// dst[i] = round(dst[i] + sum_p part[p * n + i]) with the fp32 sum in p order; dst fp32 or bf16.
// Without acc_dst the destination is written as if it held zeros (bit for bit 0 + sum), unread.
template <bool BF16_DST>
__global__ void __launch_bounds__(256) reduce_kernel(const float* __restrict__ part, int nparts, size_t n, void* dst,
                                                     bool acc_dst) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    float acc = 0.0f;
    for (int p = 0; p < nparts; ++p) acc += part[(size_t)p * n + i];
    if (BF16_DST) {
      uint16_t* d = (uint16_t*)dst;
      d[i] = rne_bf16((acc_dst ? __uint_as_float((uint32_t)d[i] << 16) : 0.0f) + acc);
    } else {
      float* d = (float*)dst;
      d[i] = (acc_dst ? d[i] : 0.0f) + acc;
    }
  }
}

int reduce_into(const Ctx& c, const float* part, int nparts, size_t n, void* dst, bool bf16_dst, bool accumulate = true) {
  if (c.query) return METALLLM_ATTN_OK;
  const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
  if (bf16_dst)
    hipLaunchKernelGGL(reduce_kernel<true>, dim3(blocks), dim3(256), 0, c.stream, part, nparts, n, dst, accumulate);
  else
    hipLaunchKernelGGL(reduce_kernel<false>, dim3(blocks), dim3(256), 0, c.stream, part, nparts, n, dst, accumulate);
  return hipGetLastError() == hipSuccess ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LAUNCH;
}

#define TRY(x)                  \
  do {                          \
    const int rc_ = (x);        \
    if (rc_) return rc_;        \
  } while (0)

#define CHECK_PTRS(...)                                           \
  do {                                                            \
    const void* ps_[] = {__VA_ARGS__};                            \
    for (const void* q_ : ps_) {                                  \
      if (!q_) return METALLLM_ATTN_E_NULL;                       \
      if (!aligned16(q_)) return METALLLM_ATTN_E_ALIGN;           \
    }                                                             \
  } while (0)

// ---- the reference kernels as sequences on a Ctx (R = B*M rows, C = N features) ----

// When q_w, k_w, v_w are equally spaced in memory (a fused [3][C][C] weight, or one weight used
// three times) and q, k, v are equally spaced without overlapping, the three products run as one
// strided-batched library call: 768 workgroups in flight at config 4 instead of three launches of
// 256, 66 against 75 us measured. Otherwise three calls.
int op_qkv(const Ctx& c, const uint16_t* X, uint16_t* q, uint16_t* k, uint16_t* v, const uint16_t* q_w,
           const uint16_t* k_w, const uint16_t* v_w, int R, int C) {
  // distances in bf16 elements, from the integer addresses (the buffers may be separate allocations)
  const auto at = [](const uint16_t* ptr) { return (intptr_t)(uintptr_t)ptr; };
  const intptr_t bw = at(k_w) - at(q_w), by = at(k) - at(q);
  const intptr_t dw = bw / 2, dy = by / 2;
  const bool batched = bw % 2 == 0 && by % 2 == 0 && dw >= 0 && at(v_w) - at(k_w) == bw && dy >= (intptr_t)R * C &&
                       at(v) - at(k) == by;
  if (tile_rows_ok(R, C, batched ? kQkvBatched : kQkv) && qkv_apart(X, q, k, v, q_w, k_w, v_w, R, C))
    return tile_rows(c, mla::TileRows{X, {q_w, k_w, v_w}, {q, k, v}, 3, R, C}, false);
  if (batched) {
    const float alpha = 1.0f, beta = 0.0f;
    // row-major Y_i = X . W_i; column-major Y_i^T = W_i^T . X^T
    const rocblas_status st = rocblas_gemm_strided_batched_ex(
        c.h, rocblas_operation_none, rocblas_operation_none, C, R, C, &alpha, q_w, BF, C, (rocblas_stride)dw, X, BF, C, 0,
        &beta, q, BF, C, (rocblas_stride)dy, q, BF, C, (rocblas_stride)dy, 3, rocblas_datatype_f32_r,
        rocblas_gemm_algo_standard, 0, 0);
    return blas_ok(c, st) ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LIBRARY;
  }
  TRY(gemm_rm(c, false, false, R, C, C, X, BF, C, q_w, BF, C, 0.0f, q, BF, C));
  TRY(gemm_rm(c, false, false, R, C, C, X, BF, C, k_w, BF, C, 0.0f, k, BF, C));
  return gemm_rm(c, false, false, R, C, C, X, BF, C, v_w, BF, C, 0.0f, v, BF, C);
}

int op_proj_fwd(const Ctx& c, const uint16_t* attn_out, const uint16_t* proj_w, uint16_t* out, int R, int C) {
  if (tile_rows_ok(R, C, kProjForward) && rows_apart(attn_out, proj_w, out, R, C))
    return tile_rows(c, mla::TileRows{attn_out, {proj_w}, {out}, 1, R, C}, false);
  return gemm_rm(c, false, false, R, C, C, attn_out, BF, C, proj_w, BF, C, 0.0f, out, BF, C);
}

// partial: at least partial_need(R, C, proj_dw_apart) floats. accumulate = false: dProjw is written as if it
// held zeros (the phase encoder; every op_* below takes the same flag). Larger products in multiples
// of 128 run computeGradDw's 128-wide kernel (sublayer_gemm.hip) on the one bf16 gradient.
int op_proj_dw(const Ctx& c, const uint16_t* attn_out, const uint16_t* dZ, uint16_t* dProjw, int R, int C,
               float* partial, bool accumulate = true) {
  if (tile_dw_one_ok(R, C) && proj_dw_apart(attn_out, dZ, dProjw, R, C)) {
    mla::TileGrad a{};
    a.x[3] = attn_out, a.g[3] = dZ, a.dW[3] = dProjw, a.w0 = 3, a.w1 = 4, a.R = R, a.C = C;
    return tile_grad(c, a, partial, accumulate);
  }
  if (mla::grad_dw_fused_ok(R, C)) {
    if (c.query) return METALLLM_ATTN_OK;
    return mla::launch_grad_dw_one(attn_out, dZ, dProjw, partial, R, C, accumulate, c.stream) == hipSuccess
               ? METALLLM_ATTN_OK
               : METALLLM_ATTN_E_LAUNCH;
  }
  const int parts = row_chunks(R);
  TRY(xt_g_partials(c, attn_out, dZ, R, C, parts, partial));
  return reduce_into(c, partial, parts, (size_t)C * C, dProjw, true, accumulate);
}

int op_proj_dx(const Ctx& c, const uint16_t* dZ, const uint16_t* proj_w, uint16_t* dAttn, int R, int C) {
  if (tile_rows_ok(R, C, kProjBackward) && rows_apart(dZ, proj_w, dAttn, R, C))
    return tile_rows(c, mla::TileRows{dZ, {proj_w}, {dAttn}, 1, R, C}, true);
  return gemm_rm(c, false, true, R, C, C, dZ, BF, C, proj_w, BF, C, 0.0f, dAttn, BF, C);
}

// The hand-written kernels read the fp32 dQ themselves; the library runs on hi, lo, the two-term bf16
// split of dQ (split_dq). tiles: the buffers allow the tile kernel (grad_dx_apart).
int op_grad_dx(const Ctx& c, float* dX, const uint16_t* qw, const uint16_t* kw, const uint16_t* vw, const float* dQ,
               const uint16_t* hi, const uint16_t* lo, const uint16_t* dK, const uint16_t* dV, int R, int C, bool tiles,
               bool accumulate = true) {
  if (tiles && tile_dx_ok(R, C))
    return tile_grad(c, mla::TileGrad{dX, dQ, {qw, kw, vw}, {}, {nullptr, dK, dV}, {}, 0, 0, R, C}, nullptr, accumulate);
  if (mla::grad_dx_fused_ok(R, C)) {
    if (c.query) return METALLLM_ATTN_OK;
    return mla::launch_grad_dx(dX, dQ, dK, dV, qw, kw, vw, R, C, accumulate, c.stream) == hipSuccess
               ? METALLLM_ATTN_OK
               : METALLLM_ATTN_E_LAUNCH;
  }
  TRY(gemm_rm(c, false, true, R, C, C, hi, BF, C, qw, BF, C, accumulate ? 1.0f : 0.0f, dX, F32, C));
  TRY(gemm_rm(c, false, true, R, C, C, lo, BF, C, qw, BF, C, 1.0f, dX, F32, C));
  TRY(gemm_rm(c, false, true, R, C, C, dK, BF, C, kw, BF, C, 1.0f, dX, F32, C));
  return gemm_rm(c, false, true, R, C, C, dV, BF, C, vw, BF, C, 1.0f, dX, F32, C);
}

// partial: at least partial_need(R, C, tiles) floats; hi, lo as in op_grad_dx; tiles: grad_dw_apart.
int op_grad_dw(const Ctx& c, const uint16_t* x, const float* dQ, const uint16_t* hi, const uint16_t* lo,
               const uint16_t* dK, const uint16_t* dV, float* dQw, uint16_t* dKw, uint16_t* dVw, int R, int C,
               float* part, bool tiles, bool accumulate = true) {
  if (tiles && tile_dw_ok(R, C))
    return tile_grad(c, mla::TileGrad{nullptr, dQ, {}, {x, x, x}, {nullptr, dK, dV}, {dQw, dKw, dVw}, 0, 3, R, C}, part,
                     accumulate);
  if (mla::grad_dw_fused_ok(R, C)) {
    if (c.query) return METALLLM_ATTN_OK;
    return mla::launch_grad_dw(x, dQ, dK, dV, dQw, dKw, dVw, part, R, C, accumulate, c.stream) == hipSuccess
               ? METALLLM_ATTN_OK
               : METALLLM_ATTN_E_LAUNCH;
  }
  const int parts = row_chunks(R);
  const size_t cc = (size_t)C * C;
  // dQw: the partials of X^T.hi and X^T.lo together, added into dQw once
  TRY(xt_g_partials(c, x, hi, R, C, parts, part));
  TRY(xt_g_partials(c, x, lo, R, C, parts, part + parts * cc));
  TRY(reduce_into(c, part, 2 * parts, cc, dQw, false, accumulate));
  TRY(xt_g_partials(c, x, dK, R, C, parts, part));
  TRY(reduce_into(c, part, parts, cc, dKw, true, accumulate));
  TRY(xt_g_partials(c, x, dV, R, C, parts, part));
  return reduce_into(c, part, parts, cc, dVw, true, accumulate);
}

// Public entry points: the device's handle and buffers, bound to the caller's stream.
struct Public {
  Session s;
  Ctx c;
  explicit Public(metalllm_stream_t stream) : s((hipStream_t)stream) {
    c.h = s.st ? s.st->handle : nullptr;
    c.stream = (hipStream_t)stream;
  }
};

}  // namespace

extern "C" {

int computeQKV(const uint16_t* X, uint16_t* q, uint16_t* k, uint16_t* v, const uint16_t* q_w, const uint16_t* k_w,
               const uint16_t* v_w, const AttentionParams* p, metalllm_stream_t stream) {
  TRY(validate_gemm(p));
  CHECK_PTRS(X, q, k, v, q_w, k_w, v_w);
  Public u(stream);
  TRY(u.s.rc);
  return op_qkv(u.c, X, q, k, v, q_w, k_w, v_w, (int)(p->B * p->M), (int)p->N);
}

int projForward(const uint16_t* attn_out, const uint16_t* proj_w, uint16_t* out, const AttentionParams* p,
                metalllm_stream_t stream) {
  TRY(validate_gemm(p));
  CHECK_PTRS(attn_out, proj_w, out);
  Public u(stream);
  TRY(u.s.rc);
  return op_proj_fwd(u.c, attn_out, proj_w, out, (int)(p->B * p->M), (int)p->N);
}

int projBackwarddW(const uint16_t* attn_out, const uint16_t* dZ, uint16_t* dProjw, const AttentionParams* p,
                   metalllm_stream_t stream) {
  TRY(validate_gemm(p));
  CHECK_PTRS(attn_out, dZ, dProjw);
  const int R = (int)(p->B * p->M), C = (int)p->N;
  Public u(stream);
  TRY(u.s.rc);
  const size_t partial = partial_need(R, C, proj_dw_apart(attn_out, dZ, dProjw, R, C));
  TRY(ensure(u.s.st->partial, u.s.st->partial_elems, partial, u.c.stream));
  return op_proj_dw(u.c, attn_out, dZ, dProjw, R, C, u.s.st->partial);
}

int projBackwarddX(const uint16_t* dZ, const uint16_t* proj_w, uint16_t* dAttn, const AttentionParams* p,
                   metalllm_stream_t stream) {
  TRY(validate_gemm(p));
  CHECK_PTRS(dZ, proj_w, dAttn);
  Public u(stream);
  TRY(u.s.rc);
  return op_proj_dx(u.c, dZ, proj_w, dAttn, (int)(p->B * p->M), (int)p->N);
}

int computeGradDx(float* dX, const uint16_t* qw, const uint16_t* kw, const uint16_t* vw, const float* dQ,
                  const uint16_t* dK, const uint16_t* dV, const AttentionParams* p, metalllm_stream_t stream) {
  TRY(validate_gemm(p));
  CHECK_PTRS(dX, qw, kw, vw, dQ, dK, dV);
  const int R = (int)(p->B * p->M), C = (int)p->N;
  const size_t e = (size_t)R * C;
  Public u(stream);
  TRY(u.s.rc);
  const bool tiles = grad_dx_apart(dX, qw, kw, vw, dQ, dK, dV, R, C);
  if (!split_need(R, C, true, tiles)) return op_grad_dx(u.c, dX, qw, kw, vw, dQ, nullptr, nullptr, dK, dV, R, C, tiles);
  TRY(ensure(u.s.st->split, u.s.st->split_elems, 2 * e, u.c.stream));
  TRY(split_dq(u.c, dQ, e, u.s.st->split));
  return op_grad_dx(u.c, dX, qw, kw, vw, dQ, u.s.st->split, u.s.st->split + e, dK, dV, R, C, tiles);
}

int computeGradDw(const uint16_t* x, const float* dQ, const uint16_t* dK, const uint16_t* dV, float* dQw,
                  uint16_t* dKw, uint16_t* dVw, const AttentionParams* p, metalllm_stream_t stream) {
  TRY(validate_gemm(p));
  CHECK_PTRS(x, dQ, dK, dV, dQw, dKw, dVw);
  const int R = (int)(p->B * p->M), C = (int)p->N;
  const size_t e = (size_t)R * C;
  Public u(stream);
  TRY(u.s.rc);
  const bool tiles = grad_dw_apart(x, dQ, dK, dV, dQw, dKw, dVw, R, C);
  TRY(ensure(u.s.st->partial, u.s.st->partial_elems, partial_need(R, C, tiles), u.c.stream));
  if (!split_need(R, C, false, tiles))
    return op_grad_dw(u.c, x, dQ, nullptr, nullptr, dK, dV, dQw, dKw, dVw, R, C, u.s.st->partial, tiles);
  TRY(ensure(u.s.st->split, u.s.st->split_elems, 2 * e, u.c.stream));
  TRY(split_dq(u.c, dQ, e, u.s.st->split));
  return op_grad_dw(u.c, x, dQ, u.s.st->split, u.s.st->split + e, dK, dV, dQw, dKw, dVw, R, C, u.s.st->partial,
                    tiles);
}

}  // extern "C"

// ---- Phase encoder ----
// model.h encodes each phase of a training step into one command buffer (forward :441-508,
// backward :587-708) and commits it once (commitWait, :358-366); the buffers are allocated once
// in the constructor (:236-277), so the same dispatches run on the same buffers every step. The
// MI355X form is a HIP graph per phase of the attention sublayer: the launches are recorded once
// on a private stream with the pointers and shapes baked in, and replayed with one launch. Each
// graph owns its rocBLAS handle, that handle's workspace (sized by a rocBLAS size query before
// capture) and its scratch (dQ split, weight-gradient partials, the attention backward's dS
// tiles), so nothing a replay touches is ever reallocated by other calls.
struct metalllmSublayerGraph {
  int phase = 0;
  rocblas_handle h = nullptr;
  void* workspace = nullptr;
  uint16_t* split = nullptr;
  float* partial = nullptr;
  void* attn_ws = nullptr;
  uint64_t attn_ws_bytes = 0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

namespace {

int check_phase(int phase, const metalllmSublayerBuffers* b, const AttentionParams* p) {
  if (!b || !p) return METALLLM_ATTN_E_NULL;
  if (phase != 0 && phase != 1) return METALLLM_ATTN_E_LAYOUT;
  TRY(validate_gemm(p));
  if (p->M % 64) return METALLLM_ATTN_E_SEQLEN;
  if (p->D != 64 && p->D != 128) return METALLLM_ATTN_E_HEADDIM;
  if (phase == 0) {
    CHECK_PTRS(b->X, b->q_w, b->k_w, b->v_w, b->proj_w, b->q, b->k, b->v, b->attn_out, b->l, b->out);
  } else {
    CHECK_PTRS(b->X, b->q_w, b->k_w, b->v_w, b->proj_w, b->q, b->k, b->v, b->attn_out, b->l, b->dOut, b->dAttn,
               b->Dsum, b->dQ, b->dK, b->dV, b->dX, b->dQw, b->dKw, b->dVw, b->dProjw);
    if (b->dX_bf16 && !aligned16(b->dX_bf16)) return METALLLM_ATTN_E_ALIGN;
  }
  if (b->hidden) {  // the block's attention half
    CHECK_PTRS(b->hidden, b->ln_gamma, b->ln_beta, b->ln_xnorm, b->ln_stdev, b->ln_dgamma, b->ln_dbeta, b->residual,
               b->dStream);
    if (p->N > 4096 || !(b->ln_eps >= 0.0f)) return METALLLM_ATTN_E_LAYOUT;
  }
  return METALLLM_ATTN_OK;
}

// Which of a phase's dispatches go into one launch: by shape, and where the buffers that the launch
// would read and write in no order are apart. A buffer may otherwise reuse the memory of one that the
// phase has finished with in the reference's order (dK in attn_out's, Dsum in dOut's, residual in
// attn_out's).
struct Joins {
  bool residual;  // phase 0: residualAdd in projForward's tiles
  bool d;         // phase 1: computeD and the zeroing of the layernorm gradients in projBackwarddX's tiles
  bool dprojw;    // phase 1: dProjw last, with the other weight gradients
  bool tiles;     // phase 1: the gradient products' buffers allow the tile kernels
};
Joins joins(int phase, const metalllmSublayerBuffers* b, const AttentionParams* p) {
  const int R = (int)(p->B * p->M), C = (int)p->N;
  const size_t e = (size_t)R * C, w = (size_t)C * C;
  using mla::any_overlap;
  const mla::Span attn_out = span(b->attn_out, e), proj_w = span(b->proj_w, w);
  Joins j{};
  if (phase == 0) {
    j.residual = b->hidden && tile_rows_ok(R, C, kProjForward) && rows_apart(b->attn_out, b->proj_w, b->out, R, C) &&
                 !any_overlap({span(b->residual, e)}, {attn_out, proj_w});
    return j;
  }
  const mla::Span X = span(b->X, e), dOut = span(b->dOut, e), Dsum = span(b->Dsum, (size_t)R * p->NH), dX = span(b->dX, e);
  const mla::Span dQ = span(b->dQ, e), dK = span(b->dK, e), dV = span(b->dV, e);
  const mla::Span dWq = span(b->dQw, w), dWk = span(b->dKw, w), dWv = span(b->dVw, w), dWp = span(b->dProjw, w);
  j.d = p->D == 64 && tile_rows_ok(R, C, kProjBackward) && rows_apart(b->dOut, b->proj_w, b->dAttn, R, C) &&
        !any_overlap({Dsum}, {dOut, proj_w});
  j.tiles = grad_dx_apart(b->dX, b->q_w, b->k_w, b->v_w, b->dQ, b->dK, b->dV, R, C) &&
            grad_dw_apart(b->X, b->dQ, b->dK, b->dV, b->dQw, b->dKw, b->dVw, R, C) &&
            !any_overlap({dX, dWq, dWk, dWv, dWp}) &&
            !any_overlap({dWq, dWk, dWv, dWp}, {span(b->q_w, w), span(b->k_w, w), span(b->v_w, w), attn_out, dOut}) &&
            !any_overlap({dX}, {X}) && !any_overlap({dWp}, {X, dQ, dK, dV});
  // dProjw reads attn_out and dOut: at the end only where nothing the phase writes before that, nor
  // dX in the same launch, replaces them
  j.dprojw = ((j.tiles && tile_dxdw_ok(R, C)) || (mla::grad_dw_fused_ok(R, C) && mla::grad_dx_fused_ok(R, C))) &&
             !any_overlap({span(b->dAttn, e), Dsum, dQ, dK, dV, dX}, {attn_out, dOut});
  return j;
}

// The launch sequence of one phase (model.h:444-483 forward, :549-555 and :620-693 backward).
int encode(const Ctx& c, int phase, const metalllmSublayerBuffers* b, const AttentionParams* p, uint16_t* split,
           float* partial, void* attn_ws, uint64_t attn_ws_bytes) {
  const int R = (int)(p->B * p->M), C = (int)p->N;
  const size_t e = (size_t)R * C;
  const metalllm_stream_t s = (metalllm_stream_t)c.stream;
  const bool block = b->hidden != nullptr;
  const LayernormParams lp{(uint32_t)R, (uint32_t)C, (uint32_t)std::min(C, 1024), b->ln_eps};
  const Joins j = joins(phase, b, p);
  if (phase == 0) {
    if (block && !c.query)  // model.h:445: X = ln1(hidden)
      TRY(layernormForward(b->hidden, b->ln_xnorm, (uint16_t*)b->X, b->ln_gamma, b->ln_beta, b->ln_stdev, &lp, s));
    TRY(op_qkv(c, b->X, b->q, b->k, b->v, b->q_w, b->k_w, b->v_w, R, C));
    if (!c.query) TRY(flashAttentionForward(b->q, b->k, b->v, b->attn_out, b->l, p, s));
    if (j.residual) {  // the projection's tiles add hidden as they are stored (model.h:483)
      mla::TileRows t{b->attn_out, {b->proj_w}, {b->out}, 1, R, C};
      t.add = b->hidden;
      t.sum = b->residual;
      return tile_rows(c, t, false);
    }
    TRY(op_proj_fwd(c, b->attn_out, b->proj_w, b->out, R, C));
    if (block && !c.query) TRY(residualAdd(b->hidden, b->out, b->residual, (uint32_t)e, s));  // model.h:483
    return METALLLM_ATTN_OK;
  }
  // model.h:549-555 zeroes the accumulated gradients before the pass and the kernels add into
  // them. Each of dX, dQw, dKw, dVw and dProjw has a single producer in this phase, so the phase
  // runs them in write mode instead: the result is bit for bit 0 + the gradient (-0 becomes +0),
  // without the zeroing pass and without reading the destinations. The attention backward writes
  // dQ, dK and dV in full; the block's layernorm gradients (model.h:545-546), which its backward
  // adds into with atomics, are zeroed by the launch that computes D (projBackwarddX's tiles, or
  // computeD's).
  // dProjw (which nothing in this phase reads) joins computeGradDw's launch at the end as a fourth
  // weight: one launch of balanced items instead of projBackwarddW's own short-item launch. Its sum
  // then runs over other row chunks than the entry point's, so it can differ from projBackwarddW's
  // result by the fp32 summation order (one bf16 rounding step at most).
  const bool tile = j.dprojw && j.tiles && tile_dxdw_ok(R, C);
  if (!j.dprojw) TRY(op_proj_dw(c, b->attn_out, b->dOut, b->dProjw, R, C, partial, false));
  // projBackwarddX and computeD: one launch where the tiles of dAttn are whole heads
  float *dgamma = block ? b->ln_dgamma : nullptr, *dbeta = block ? b->ln_dbeta : nullptr;
  if (j.d) {
    mla::TileRows t{b->dOut, {b->proj_w}, {b->dAttn}, 1, R, C};
    t.O = b->attn_out;
    t.Dv = b->Dsum;
    t.T = (int)p->M;
    t.H = (int)p->NH;
    t.zero0 = dgamma;
    t.zero1 = dbeta;
    TRY(tile_rows(c, t, true));
  } else {
    TRY(op_proj_dx(c, b->dOut, b->proj_w, b->dAttn, R, C));
    if (!c.query && mla::launch_compute_d(mla::ComputeDArgs{b->dAttn, b->attn_out, b->Dsum, (int)p->M, (int)p->NH,
                                                            (int)p->B, dgamma, dbeta, block ? (uint32_t)C : 0u},
                                          (int)p->D, c.stream) != hipSuccess)
      return METALLLM_ATTN_E_LAUNCH;
  }
  if (!c.query) {
    TRY(flashAttentionBackwardWorkspace(b->dAttn, b->Dsum, b->l, b->q, b->k, b->v, b->dQ, b->dK, b->dV, attn_ws,
                                        attn_ws_bytes, p, s));
  }
  uint16_t* lo = nullptr;  // no split when hand-written kernels take both products
  if (!j.dprojw && std::max(split_need(R, C, true, j.tiles), split_need(R, C, false, j.tiles))) {
    TRY(split_dq(c, b->dQ, e, split));  // one split serves both consumers
    lo = split + e;
  } else {
    split = nullptr;
  }
  if (tile) {
    TRY(tile_grad(c, mla::TileGrad{b->dX, b->dQ, {b->q_w, b->k_w, b->v_w}, {b->X, b->X, b->X, b->attn_out},
                                   {nullptr, b->dK, b->dV, b->dOut}, {b->dQw, b->dKw, b->dVw, b->dProjw}, 0, 4, R, C}, partial, false));
  } else if (j.dprojw) {
    // computeGradDx and the four weight gradients in one launch (dX tiles first, then the
    // weight-gradient items, which start as the dX tiles finish), then the reduction
    if (!c.query && mla::launch_grad_dxdw4(b->dX, b->X, b->dQ, b->dK, b->dV, b->q_w, b->k_w, b->v_w, b->attn_out,
                                           b->dOut, b->dQw, b->dKw, b->dVw, b->dProjw, partial, R, C,
                                           c.stream) != hipSuccess)
      return METALLLM_ATTN_E_LAUNCH;
  } else {
    TRY(op_grad_dx(c, b->dX, b->q_w, b->k_w, b->v_w, b->dQ, split, lo, b->dK, b->dV, R, C, j.tiles, false));
    TRY(op_grad_dw(c, b->X, b->dQ, split, lo, b->dK, b->dV, b->dQw, b->dKw, b->dVw, R, C, partial, j.tiles, false));
  }
  if (c.query) return METALLLM_ATTN_OK;
  if (block)  // model.h:692-695: cast of dX, ln1 backward and the skip add
    return mla::launch_block_ln_bwd(b->dX, b->dOut, b->ln_xnorm, b->ln_gamma, b->ln_stdev, b->dStream, b->ln_dgamma,
                                    b->ln_dbeta, (uint32_t)R, (uint32_t)C, c.stream) == hipSuccess
               ? METALLLM_ATTN_OK
               : METALLLM_ATTN_E_LAUNCH;
  if (b->dX_bf16) TRY(castFloatToBfloat(b->dX, b->dX_bf16, (uint32_t)e, s));
  return METALLLM_ATTN_OK;
}

// bf16 elements of the dQ split and floats of weight-gradient partials that phase 1 may use.
void phase_scratch(const metalllmSublayerBuffers* b, const AttentionParams* p, size_t& split, size_t& partial) {
  const int R = (int)(p->B * p->M), C = (int)p->N;
  const Joins j = joins(1, b, p);
  split = j.dprojw ? 0 : std::max(split_need(R, C, true, j.tiles), split_need(R, C, false, j.tiles));
  partial = partial_need(R, C, j.tiles && (j.dprojw || proj_dw_apart(b->attn_out, b->dOut, b->dProjw, R, C)));
}

int build_graph(metalllmSublayerGraph* g, const metalllmSublayerBuffers* b, const AttentionParams* p) {
  const int R = (int)(p->B * p->M), C = (int)p->N;
  if (rocblas_create_handle(&g->h) != rocblas_status_success) {
    g->h = nullptr;
    return METALLLM_ATTN_E_LIBRARY;
  }
  if (g->phase == 1) {
    size_t split = 0, partial = 0;
    phase_scratch(b, p, split, partial);
    if (split && hipMalloc((void**)&g->split, split * sizeof(uint16_t)) != hipSuccess) g->split = nullptr;
    if (partial && hipMalloc((void**)&g->partial, partial * sizeof(float)) != hipSuccess) g->partial = nullptr;
    TRY(metalllmAttnBackwardWorkspaceSize(p, &g->attn_ws_bytes));
    if (hipMalloc(&g->attn_ws, g->attn_ws_bytes) != hipSuccess) g->attn_ws = nullptr;
    if ((split && !g->split) || (partial && !g->partial) || !g->attn_ws) return METALLLM_ATTN_E_LIBRARY;
  }
  // the workspace the phase's rocBLAS calls need, owned by the graph
  size_t ws = 0;
  if (rocblas_start_device_memory_size_query(g->h) != rocblas_status_success) return METALLLM_ATTN_E_LIBRARY;
  Ctx q;
  q.h = g->h;
  q.query = true;
  const int qrc = encode(q, g->phase, b, p, g->split, g->partial, g->attn_ws, g->attn_ws_bytes);
  if (rocblas_stop_device_memory_size_query(g->h, &ws) != rocblas_status_success || qrc) return METALLLM_ATTN_E_LIBRARY;
  if (ws && hipMalloc(&g->workspace, ws) != hipSuccess) {
    g->workspace = nullptr;
    return METALLLM_ATTN_E_LIBRARY;
  }
  if (rocblas_set_workspace(g->h, g->workspace, ws) != rocblas_status_success) return METALLLM_ATTN_E_LIBRARY;
  mla::forward_prepare();  // the forward's device queries, before the capture
  hipStream_t cap = nullptr;
  if (hipStreamCreateWithFlags(&cap, hipStreamNonBlocking) != hipSuccess) return METALLLM_ATTN_E_LIBRARY;
  int rc = rocblas_set_stream(g->h, cap) == rocblas_status_success ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LIBRARY;
  if (!rc && hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal) != hipSuccess) rc = METALLLM_ATTN_E_LIBRARY;
  else if (!rc) {
    Ctx c;
    c.h = g->h;
    c.stream = cap;
    rc = encode(c, g->phase, b, p, g->split, g->partial, g->attn_ws, g->attn_ws_bytes);
    const hipError_t e = hipStreamEndCapture(cap, &g->graph);  // always ends the capture
    if (!rc && e != hipSuccess) rc = METALLLM_ATTN_E_LIBRARY;
  }
  if (!rc && hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0) != hipSuccess) rc = METALLLM_ATTN_E_LIBRARY;
  (void)hipStreamDestroy(cap);
  return rc;
}

}  // namespace

extern "C" {

int metalllmSublayerEncode(int phase, const metalllmSublayerBuffers* b, const AttentionParams* p,
                           metalllm_stream_t stream) {
  TRY(check_phase(phase, b, p));
  const int R = (int)(p->B * p->M), C = (int)p->N;
  Public u(stream);
  TRY(u.s.rc);
  uint64_t ws = 0;
  if (phase == 1) {
    size_t split = 0, partial = 0;
    phase_scratch(b, p, split, partial);
    TRY(ensure(u.s.st->split, u.s.st->split_elems, split, u.c.stream));
    TRY(ensure(u.s.st->partial, u.s.st->partial_elems, partial, u.c.stream));
    TRY(metalllmAttnBackwardWorkspaceSize(p, &ws));
    TRY(ensure(u.s.st->attn_ws, u.s.st->attn_ws_bytes, (size_t)ws, u.c.stream));
  }
  return encode(u.c, phase, b, p, u.s.st->split, u.s.st->partial, u.s.st->attn_ws, ws);
}

int metalllmSublayerRoute(int phase, const metalllmSublayerBuffers* b, const AttentionParams* p) {
  TRY(check_phase(phase, b, p));
  const Joins j = joins(phase, b, p);
  return phase == 0 ? (j.residual ? 1 : 0) : (j.d ? 1 : 0) | (j.dprojw ? 2 : 0) | (j.tiles ? 4 : 0);
}

int metalllmSublayerScratch(const AttentionParams* p, uint64_t need[2], uint64_t reserved[2]) {
  TRY(validate_gemm(p));
  if (!need || !reserved) return METALLLM_ATTN_E_NULL;
  const int R = (int)(p->B * p->M), C = (int)p->N;
  need[0] = any_split_need(R, C);
  need[1] = partial_need(R, C, false);
  reserved[0] = split_bound(R, C);
  reserved[1] = partial_bound(R, C);
  return METALLLM_ATTN_OK;
}

int metalllmSublayerReserve(const AttentionParams* p) {
  TRY(validate_gemm(p));
  if (p->D != 64 && p->D != 128) return METALLLM_ATTN_E_HEADDIM;
  if (p->M % 64) return METALLLM_ATTN_E_SEQLEN;
  const int R = (int)(p->B * p->M), C = (int)p->N;
  uint64_t ws = 0;
  TRY(metalllmAttnBackwardWorkspaceSize(p, &ws));
  Public u(nullptr);
  TRY(u.s.rc);
  TRY(reserve(u.s.st->split, u.s.st->split_elems, split_bound(R, C), any_split_need(R, C)));
  TRY(reserve(u.s.st->partial, u.s.st->partial_elems, partial_bound(R, C), partial_need(R, C, false)));
  TRY(ensure(u.s.st->attn_ws, u.s.st->attn_ws_bytes, (size_t)ws, nullptr));
  return METALLLM_ATTN_OK;
}

int metalllmSublayerGraphCreate(int phase, const metalllmSublayerBuffers* b, const AttentionParams* p,
                                metalllmSublayerGraph** out) {
  if (!out) return METALLLM_ATTN_E_NULL;
  *out = nullptr;
  TRY(check_phase(phase, b, p));
  metalllmSublayerGraph* g = new metalllmSublayerGraph();
  g->phase = phase;
  const int rc = build_graph(g, b, p);
  if (rc) {
    metalllmSublayerGraphDestroy(g);
    return rc;
  }
  *out = g;
  return METALLLM_ATTN_OK;
}

int metalllmSublayerGraphLaunch(metalllmSublayerGraph* g, metalllm_stream_t stream) {
  if (!g || !g->exec) return METALLLM_ATTN_E_NULL;
  return hipGraphLaunch(g->exec, (hipStream_t)stream) == hipSuccess ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LAUNCH;
}

int metalllmSublayerGraphDestroy(metalllmSublayerGraph* g) {
  if (!g) return METALLLM_ATTN_OK;
  if (g->exec) (void)hipGraphExecDestroy(g->exec);
  if (g->graph) (void)hipGraphDestroy(g->graph);
  if (g->h) (void)rocblas_destroy_handle(g->h);
  if (g->workspace) (void)hipFree(g->workspace);
  if (g->split) (void)hipFree(g->split);
  if (g->partial) (void)hipFree(g->partial);
  if (g->attn_ws) (void)hipFree(g->attn_ws);
  delete g;
  return METALLLM_ATTN_OK;
}

}  // extern "C"
