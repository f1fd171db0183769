// glue.hip -- the kernels of metalLLM's pre-LN block that sit around the attention sublayer
// (declared in include/metalllm_attn.h):
//   castFloatToBfloat  elementwise.metal:19-28  out[i] = bf16(in[i])  (model.h:692: the fp32 dX of
//                      computeGradDx handed to the layernorm backward as bf16)
//   residualAdd        elementwise.metal:7-17   out[i] = bf16(a[i] + b[i])  (model.h:483,618,695)
//   layernormForward   layernorm.metal:10-70    per row: mean, variance, stdev = sqrt(var + eps),
//                      x_norm = bf16((x - mean)/stdev), out = bf16(gamma*xn + beta)  (model.h:385-396)
//   layernormBackward  layernorm.metal:73-127   dgamma += bf16(xn*dZ), dbeta += dZ (fp32, per column),
//                      dx_norm = bf16(dZ*gamma), dZ <- bf16(rstd*(dxn - mean(dxn) - xn*mean(bf16(dxn*xn))))
//                      (model.h:398-410, in place on dZ)
// All are HBM-bound. The elementwise kernels stream with 16-byte accesses in grid-stride loops.
// The layernorm kernels give each row to one wave: the row stays in registers as packed bf16
// (cols/512 16-byte chunks per lane), its sums are wave reductions, and it is read once and written
// once. The backward's column sums (dgamma, dbeta) are accumulated per workgroup over many rows in
// registers and LDS, then added with one fp32 atomic per column per workgroup. The reference adds
// one atomic per element from every row.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../../include/metalllm_attn.h"

namespace {

// float -> bf16, round to nearest even (Metal's float -> bfloat conversion); NaN stays a quiet
// NaN of the same sign, infinities and overflow to infinity as in IEEE rounding.
__device__ __forceinline__ uint32_t to_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

__global__ void __launch_bounds__(256) cast_kernel(const float* __restrict__ in, uint16_t* __restrict__ out,
                                                   uint32_t count) {
  const size_t n4 = count / 4;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n4; i += stride) {
    const float4 v = ((const float4*)in)[i];
    ((uint2*)out)[i] = uint2{to_bf16(v.x) | (to_bf16(v.y) << 16), to_bf16(v.z) | (to_bf16(v.w) << 16)};
  }
  // the count % 4 tail
  const size_t t = 4 * n4 + blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (t < count) out[t] = (uint16_t)to_bf16(in[t]);
}

unsigned grid_for(size_t items) { return (unsigned)std::max<size_t>(1, std::min<size_t>((items + 255) / 256, 8192)); }

__device__ __forceinline__ float bf_f(uint32_t h) { return __uint_as_float(h << 16); }
// Two floats -> packed bf16 pair by v_cvt_pk_bf16_f32: to_bf16's result for every float, NaNs
// included (compared over all 2^32 of them).
__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{lo, hi}, b2));
}

// out = bf16(a + b), eight elements per thread and step
__global__ void __launch_bounds__(256) residual_kernel(const uint4* __restrict__ a, const uint4* __restrict__ b,
                                                       uint4* __restrict__ out, uint32_t count) {
  const size_t n8 = count / 8;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n8; i += stride) {
    const uint4 x = a[i], y = b[i];
    const uint32_t xs[4] = {x.x, x.y, x.z, x.w}, ys[4] = {y.x, y.y, y.z, y.w};
    uint32_t r[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      r[j] = to_bf16(bf_f(xs[j] & 0xffffu) + bf_f(ys[j] & 0xffffu)) |
             (to_bf16(bf_f(xs[j] >> 16) + bf_f(ys[j] >> 16)) << 16);
    out[i] = uint4{r[0], r[1], r[2], r[3]};
  }
  const size_t t = 8 * n8 + blockIdx.x * (size_t)blockDim.x + threadIdx.x;  // the count % 8 tail
  if (t < count) {
    const uint16_t* a16 = (const uint16_t*)a;
    const uint16_t* b16 = (const uint16_t*)b;
    ((uint16_t*)out)[t] = (uint16_t)to_bf16(bf_f(a16[t]) + bf_f(b16[t]));
  }
}

// Sum over the 64 lanes of a wave, the same result in every lane: the butterfly over partners at
// distance 32, 16, 8, 4, 2, 1 in register moves (no LDS permutes, whose latency a row's two sums
// would wait for six times). After the first three levels the lanes i and i ^ 8 hold the same
// value, so a rotation by 4 within the row of 16 reaches the partner i ^ 4.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float wave_sum(float v) {
  const uint32_t u = __float_as_uint(v);
  auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const uint32_t w = __float_as_uint(v);
  auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
  v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  v += dpp<0x128>(v);  // row_ror:8
  v += dpp<0x124>(v);  // row_ror:4
  v += dpp<0x4e>(v);   // quad_perm 2,3,0,1
  v += dpp<0xb1>(v);   // quad_perm 1,0,3,2
  return v;
}

// Row layout in a wave: lane l holds the 16-byte chunks c = l + 64 j (j < NCH) of the row, i.e.
// columns 8c .. 8c + 7; chunks past cols/8 are absent (their lanes hold zeros and skip stores).
template <int NCH>
struct RowChunks {
  uint4 v[NCH];
};

template <int NCH>
__device__ __forceinline__ void load_row(const uint4* row, int nchunk, int lane, RowChunks<NCH>& r) {
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int c = lane + 64 * j;
    r.v[j] = c < nchunk ? row[c] : uint4{0u, 0u, 0u, 0u};
  }
}

__device__ __forceinline__ void unpack8(const uint4& u, float (&f)[8]) {
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    f[2 * k] = __uint_as_float(w[k] << 16);
    f[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
  }
}
__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) w[k] = pk_bf16(f[2 * k], f[2 * k + 1]);
  return uint4{w[0], w[1], w[2], w[3]};
}
// rounds eight floats in place to bf16 values
__device__ __forceinline__ void round8(float (&f)[8]) {
  unpack8(pack8(f), f);
}

// layernorm.metal:10-70, one row per wave, four waves per workgroup.
template <int NCH>
__global__ void __launch_bounds__(256) ln_fwd_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ xnorm,
                                                     uint16_t* __restrict__ out, const uint16_t* __restrict__ gamma,
                                                     const uint16_t* __restrict__ beta, float* __restrict__ stdev,
                                                     uint32_t rows, uint32_t cols, float eps) {
  const int lane = threadIdx.x & 63;
  const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int nchunk = (int)(cols / 8);
  const size_t base = (size_t)row * cols;
  RowChunks<NCH> r;
  load_row<NCH>((const uint4*)(x + base), nchunk, lane, r);
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    float f[8];
    unpack8(r.v[j], f);
#pragma unroll
    for (int k = 0; k < 8; ++k) s += f[k];
  }
  const float mean = wave_sum(s) / (float)cols;
  float q = 0.0f;
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    if (lane + 64 * j >= nchunk) continue;
    float f[8];
    unpack8(r.v[j], f);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float d = f[k] - mean;
      q += d * d;
    }
  }
  const float var = wave_sum(q) / (float)cols;
  const float sd = sqrtf(var + eps);
  const float rstd = 1.0f / sd;
  if (lane == 0) stdev[row] = sd;
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int c = lane + 64 * j;
    if (c >= nchunk) continue;
    float f[8], g[8], b[8], xn[8], o[8];
    unpack8(r.v[j], f);
    unpack8(((const uint4*)gamma)[c], g);
    unpack8(((const uint4*)beta)[c], b);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      xn[k] = (f[k] - mean) * rstd;
      o[k] = g[k] * xn[k] + b[k];  // two roundings (no contraction: built with -ffp-contract=off)
    }
    ((uint4*)(xnorm + base))[c] = pack8(xn);
    ((uint4*)(out + base))[c] = pack8(o);
  }
}

// How ln_bwd_kernel's steps (16/S rows each) are dealt to its workgroups. q = 0: step k of workgroup
// b is k*gridDim.x + b. Else contiguous ranges of about q steps, the first `more` workgroups one more,
// and of each three workgroups one has a step less and one a step more (ln_bwd_deal says when).
struct LnDeal {
  uint32_t q, more;
};
__device__ __forceinline__ uint32_t ln_first_step(const LnDeal& d, uint32_t b) {
  return b * d.q + min(b, d.more) - (b % 3 ? 1u : 0u);
}

// layernorm.metal:73-127. A workgroup of 16 waves takes 16/S rows at a time, each by S waves (S > 1
// for rows of more than 1024 columns, so that a lane holds at most two 16-byte chunks of a row: with
// whole wide rows per lane the sums and the row leave room for one wave per SIMD), in the steps
// that LnDeal says. Each lane keeps the dgamma/dbeta
// partial sums of its own columns across its rows; the waves' partials meet in LDS and one fp32
// atomic per column adds the workgroup's sum. All workgroups add into the same 2*cols addresses and
// atomics on one address run one after another (about 34 ns each), so the grid is a compromise
// (ln_bwd_grid). Four waves a workgroup, up to 1024 workgroups, rounding in integer arithmetic and
// row sums through LDS permutes took 48 us at 16384 x 768, 71 us at 32768 x 1024 and 85 us at 4096 x
// 4096; this took 24, 35 (5.8 TB/s) and 24 us, and LnDeal's ranges take the first and last another 13
// and 8% down (back to back 22.3 -> 19.4 and 29.9 -> 27.5 us).
// BLOCK (the phase encoder's form): the gradient comes in as the fp32 dX and is rounded to bf16
// first (castFloatToBfloat), and `add` is added to the result, rounded again (residualAdd): the
// three kernels' results bit for bit, with one read of dX and one write of dZ instead of three and
// two passes over the rows.
template <int NC, int S, bool BLOCK>
__global__ void __launch_bounds__(1024) ln_bwd_kernel(uint16_t* __restrict__ dZ, const float* __restrict__ dX,
                                                      const uint16_t* __restrict__ add,
                                                      const uint16_t* __restrict__ xnorm,
                                                      const uint16_t* __restrict__ gamma,
                                                      const float* __restrict__ stdev, uint16_t* __restrict__ dxnorm,
                                                      float* __restrict__ dgamma, float* __restrict__ dbeta,
                                                      uint32_t rows, uint32_t cols, LnDeal deal) {
  constexpr int W = 16, RW = W / S;  // waves, rows per step
  __shared__ float red[2][W][512];
  __shared__ float2 rsum[2][W];  // S > 1: the waves' parts of a row's two sums, by step parity
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rg = wave / S, sub = wave % S;
  const int nchunk = (int)(cols / 8);
  const int c0 = lane + 64 * NC * sub;  // this lane's first 16-byte chunk of a row
  float pg[NC][8], pb[NC][8];
  uint4 gam[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
#pragma unroll
    for (int k = 0; k < 8; ++k) pg[j][k] = pb[j][k] = 0.0f;
    const int c = c0 + 64 * j;
    gam[j] = c < nchunk ? ((const uint4*)gamma)[c] : uint4{0u, 0u, 0u, 0u};
  }
  const uint4 none = uint4{0u, 0u, 0u, 0u};
  const uint32_t first = deal.q ? ln_first_step(deal, blockIdx.x) : blockIdx.x, stride = deal.q ? 1 : gridDim.x;
  const uint32_t end = deal.q && blockIdx.x + 1 < gridDim.x ? ln_first_step(deal, blockIdx.x + 1) : (rows + RW - 1) / RW;
  for (uint32_t at = first, it = 0; at < end; at += stride, ++it) {
    const uint32_t r0 = at * RW;
    const uint32_t row = r0 + rg;
    const bool live = row < rows;  // false only past the last row: the wave adds zeros and stores nothing
    const size_t base = (size_t)min(row, rows - 1) * cols;
    uint4 dz[NC], xn[NC], ad[BLOCK ? NC : 1], dxn[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      // chunks past the row are read in bounds and taken as zeros: loads behind a per-lane branch
      // are waited for one by one (32768 x 1024: 43 us, 35 us without the branch)
      const bool in = live && c0 + 64 * j < nchunk;
      const int c = min(c0 + 64 * j, nchunk - 1);
      const uint4 x = ((const uint4*)(xnorm + base))[c];
      xn[j] = in ? x : none;
      if constexpr (BLOCK) {
        const uint4 a = ((const uint4*)(dX + base))[2 * c], b = ((const uint4*)(dX + base))[2 * c + 1];
        ad[j] = ((const uint4*)(add + base))[c];
        dz[j] = uint4{pk_bf16(__uint_as_float(a.x), __uint_as_float(a.y)), pk_bf16(__uint_as_float(a.z), __uint_as_float(a.w)),
                      pk_bf16(__uint_as_float(b.x), __uint_as_float(b.y)), pk_bf16(__uint_as_float(b.z), __uint_as_float(b.w))};
      } else {
        dz[j] = ((const uint4*)(dZ + base))[c];
      }
      if (!in) dz[j] = none;
    }
    const float rdev = 1.0f / stdev[min(row, rows - 1)];
    float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      float z[8], x[8], g[8], a[8], d[8], t[8];
      unpack8(dz[j], z);
      unpack8(xn[j], x);
      // opaque: gamma stays packed across rows (hoisted, its floats take the registers of a row)
      asm volatile("" : "+v"(gam[j].x), "+v"(gam[j].y), "+v"(gam[j].z), "+v"(gam[j].w));
      unpack8(gam[j], g);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        a[k] = x[k] * z[k];
        d[k] = z[k] * g[k];
      }
      round8(a);  // bfloat * bfloat is a bfloat
      dxn[j] = pack8(d);
      unpack8(dxn[j], d);
#pragma unroll
      for (int k = 0; k < 8; ++k) t[k] = d[k] * x[k];
      round8(t);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        pg[j][k] += a[k];
        pb[j][k] += z[k];
        s1 += d[k];
        s2 += t[k];
      }
      const int c = c0 + 64 * j;
      if (!BLOCK && dxnorm && live && c < nchunk) ((uint4*)(dxnorm + base))[c] = dxn[j];
    }
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    if constexpr (S > 1) {
      if (lane == 0) rsum[it & 1][wave] = float2{s1, s2};
      __syncthreads();  // the other parity's slots were read before the previous step's barrier
      s1 = s2 = 0.0f;
#pragma unroll
      for (int u = 0; u < S; ++u) {
        const float2 v = rsum[it & 1][rg * S + u];
        s1 += v.x;
        s2 += v.y;
      }
    }
    const float rs1 = s1 / (float)cols, rs2 = s2 / (float)cols;
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int c = c0 + 64 * j;
      if (!live || c >= nchunk) continue;
      float x[8], d[8], o[8];
      unpack8(xn[j], x);
      unpack8(dxn[j], d);
#pragma unroll
      for (int k = 0; k < 8; ++k) o[k] = rdev * ((d[k] - rs1) - x[k] * rs2);
      if constexpr (BLOCK) {
        float r[8];
        unpack8(ad[j], r);
        round8(o);
#pragma unroll
        for (int k = 0; k < 8; ++k) o[k] += r[k];
      }
      ((uint4*)(dZ + base))[c] = pack8(o);
    }
  }
  // column partials of the waves that share columns -> one atomic per column
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    if (j) __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; k += 4) {
      *(float4*)&red[0][wave][8 * lane + k] = float4{pg[j][k], pg[j][k + 1], pg[j][k + 2], pg[j][k + 3]};
      *(float4*)&red[1][wave][8 * lane + k] = float4{pb[j][k], pb[j][k + 1], pb[j][k + 2], pb[j][k + 3]};
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < 1024 * S; i += 1024) {
      const uint32_t which = (i >> 9) & 1, u = i >> 10, c = i & 511, col = 512 * (NC * u + j) + c;
      if (col >= cols) continue;
      float sum = red[which][u][c];
#pragma unroll
      for (int w = 1; w < RW; ++w) sum += red[which][w * S + u][c];
      atomicAdd((which ? dbeta : dgamma) + col, sum);
    }
  }
}

// Workgroups of ln_bwd_kernel: the rows' traffic (6 bytes an element, about 20 GB/s a workgroup)
// takes t = 6 rows cols / (20e9 n) seconds on n of them and the atomics 34e-9 n; the sum is least at
// n = 0.094 sqrt(rows cols), and there is one workgroup per CU. A step of short rows takes the time of
// its dependent loads and sums, 1.2 us, which 256 columns' traffic takes too: 12500 x 8 42.0 -> 10.3
// us, 131072 x 8 122 -> 48.5, 4000 x 32 13.9 -> 7.1, 40000 x 64 28.3 -> 20.9, 4000 x 128 9.0 -> 7.8.
uint32_t ln_bwd_grid(uint32_t rows, uint32_t cols, int rows_per_step) {
  const uint32_t n = (uint32_t)(0.094 * std::sqrt((double)rows * std::max(cols, 256u)));
  const uint32_t steps = (rows + rows_per_step - 1) / rows_per_step;
  return std::max<uint32_t>(1, std::min<uint32_t>(steps, std::min<uint32_t>(256, std::max<uint32_t>(n, 16))));
}

// Equally long workgroups all end, and add into the same columns, at the same time. With ends a step
// apart one third's atomics run while the others still stream rows: 16384 x 768 22.3 -> 19.4 us, 12288
// x 768 19.3 -> 16.8, 8192 x 1536 23.6 -> 20.1, 32768 x 384 21.8 -> 20.6. Not with fewer than three
// steps each; nor where a step is long against the atomics and the ends drift apart by themselves
// (98304 elements a workgroup, 24576 x 1024, 28.8 -> 28.4; 131072, 32768 x 1024, 34.5 -> 35.6); nor
// where the steps do not divide and are few, so that ends differ already (13000 x 520, three and a
// third steps, 17.1 -> 17.0, the encoder's form 21.1 -> 22.1; 32768 x 200, eight and a half, 20.4 -> 19.6).
LnDeal ln_bwd_deal(uint32_t rows, uint32_t cols, int rows_per_step, uint32_t n) {
  const uint32_t steps = (rows + rows_per_step - 1) / rows_per_step, q = steps / n, more = steps - q * n;
  const bool apart = q >= 3 && (uint64_t)rows * cols < 100000ull * n && (q >= 8 || more * 8 < n);
  return apart ? LnDeal{q, more} : LnDeal{0, 0};
}

template <bool BLOCK>
hipError_t launch_ln_bwd(uint16_t* dZ, const float* dX, const uint16_t* add, const uint16_t* xnorm, const uint16_t* gamma,
                         const float* stdev, uint16_t* dxnorm, float* dgamma, float* dbeta, uint32_t rows, uint32_t cols,
                         hipStream_t s) {
  const int nch = (int)((cols / 8 + 63) / 64);
  const int S = nch <= 2 ? 1 : (nch <= 4 ? 2 : 4);
  const dim3 grid(ln_bwd_grid(rows, cols, 16 / S));
  const LnDeal deal = ln_bwd_deal(rows, cols, 16 / S, grid.x);
#define LNB(NC, S_) \
  hipLaunchKernelGGL((ln_bwd_kernel<NC, S_, BLOCK>), grid, dim3(1024), 0, s, dZ, dX, add, xnorm, gamma, stdev, dxnorm, \
                     dgamma, dbeta, rows, cols, deal)
  if (nch == 1) LNB(1, 1);
  else if (S == 1) LNB(2, 1);
  else if (S == 2) LNB(2, 2);
  else LNB(2, 4);
#undef LNB
  return hipGetLastError();
}

int validate_ln(const LayernormParams* p) {
  if (!p) return METALLLM_ATTN_E_NULL;
  if (p->rows == 0 || p->cols == 0 || p->cols % 8 || p->cols > 4096) return METALLLM_ATTN_E_LAYOUT;
  if ((uint64_t)p->rows * p->cols >= (1ull << 31)) return METALLLM_ATTN_E_SIZE;
  if (!(p->eps >= 0.0f)) return METALLLM_ATTN_E_LAYOUT;
  return METALLLM_ATTN_OK;
}

bool al16(const void* q) { return ((uintptr_t)q & 15u) == 0; }

}  // namespace

namespace mla {
// The phase encoder's end of the backward (model.h:692-695) in one launch: dStream =
// bf16(ln backward(bf16(dX)) + dOut), dgamma and dbeta added into.
hipError_t launch_block_ln_bwd(const float* dX, const uint16_t* dOut, const uint16_t* xnorm, const uint16_t* gamma,
                               const float* stdev, uint16_t* dStream, float* dgamma, float* dbeta, uint32_t rows,
                               uint32_t cols, hipStream_t s) {
  return launch_ln_bwd<true>(dStream, dX, dOut, xnorm, gamma, stdev, nullptr, dgamma, dbeta, rows, cols, s);
}
}  // namespace mla

extern "C" {

int residualAdd(const uint16_t* a, const uint16_t* b, uint16_t* out, uint32_t count, metalllm_stream_t stream) {
  if (count == 0) return METALLLM_ATTN_OK;
  if (!a || !b || !out) return METALLLM_ATTN_E_NULL;
  if (!al16(a) || !al16(b) || !al16(out)) return METALLLM_ATTN_E_ALIGN;
  hipLaunchKernelGGL(residual_kernel, dim3(grid_for(count / 8 + 1)), dim3(256), 0, (hipStream_t)stream,
                     (const uint4*)a, (const uint4*)b, (uint4*)out, count);
  return hipGetLastError() == hipSuccess ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LAUNCH;
}

int layernormForward(const uint16_t* x, uint16_t* x_norm, uint16_t* out, const uint16_t* gamma, const uint16_t* beta,
                     float* stdev, const LayernormParams* p, metalllm_stream_t stream) {
  const int rc = validate_ln(p);
  if (rc) return rc;
  if (!x || !x_norm || !out || !gamma || !beta || !stdev) return METALLLM_ATTN_E_NULL;
  if (!al16(x) || !al16(x_norm) || !al16(out) || !al16(gamma) || !al16(beta) || !al16(stdev))
    return METALLLM_ATTN_E_ALIGN;
  const dim3 grid((p->rows + 3) / 4);
  const hipStream_t s = (hipStream_t)stream;
  const int nch = (int)((p->cols / 8 + 63) / 64);
#define LNF(N) hipLaunchKernelGGL(ln_fwd_kernel<N>, grid, dim3(256), 0, s, x, x_norm, out, gamma, beta, stdev, p->rows, p->cols, p->eps)
  switch (nch) {
    case 1: LNF(1); break;
    case 2: LNF(2); break;
    case 3: LNF(3); break;
    case 4: LNF(4); break;
    case 5: LNF(5); break;
    case 6: LNF(6); break;
    case 7: LNF(7); break;
    default: LNF(8); break;
  }
#undef LNF
  return hipGetLastError() == hipSuccess ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LAUNCH;
}

int layernormBackward(uint16_t* dZ, const uint16_t* x_norm_cache, const uint16_t* gamma, const float* stdev,
                      uint16_t* dx_norm, float* dgamma, float* dbeta, const LayernormParams* p,
                      metalllm_stream_t stream) {
  const int rc = validate_ln(p);
  if (rc) return rc;
  if (!dZ || !x_norm_cache || !gamma || !stdev || !dgamma || !dbeta) return METALLLM_ATTN_E_NULL;
  if (!al16(dZ) || !al16(x_norm_cache) || !al16(gamma) || !al16(stdev) || !al16(dgamma) || !al16(dbeta) ||
      (dx_norm && !al16(dx_norm)))
    return METALLLM_ATTN_E_ALIGN;
  return launch_ln_bwd<false>(dZ, nullptr, nullptr, x_norm_cache, gamma, stdev, dx_norm, dgamma, dbeta, p->rows, p->cols,
                              (hipStream_t)stream) == hipSuccess
             ? METALLLM_ATTN_OK
             : METALLLM_ATTN_E_LAUNCH;
}

int castFloatToBfloat(const float* in, uint16_t* out, uint32_t count, metalllm_stream_t stream) {
  if (count == 0) return METALLLM_ATTN_OK;
  if (!in || !out) return METALLLM_ATTN_E_NULL;
  if (((uintptr_t)in & 15u) || ((uintptr_t)out & 15u)) return METALLLM_ATTN_E_ALIGN;
  hipLaunchKernelGGL(cast_kernel, dim3(grid_for(count / 4 + 1)), dim3(256), 0, (hipStream_t)stream, in, out, count);
  return hipGetLastError() == hipSuccess ? METALLLM_ATTN_OK : METALLLM_ATTN_E_LAUNCH;
}

}  // extern "C"
