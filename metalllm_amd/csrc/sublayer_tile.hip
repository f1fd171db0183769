// sublayer_tile.hip -- the attention sublayer's matrix products on 64 x 64 output tiles, for sizes
// that leave the chip short of work or of whole 128-wide tiles:
//   computeQKV      attention.metal:19-53     projForward     attention.metal:385-405
//   projBackwarddW  attention.metal:407-430   projBackwarddX  attention.metal:432-455
//   computeGradDx   attention.metal:301-341   computeGradDw   attention.metal:343-383
// Any row count for the row products, a multiple of 64 for the weight gradients (their sums run over
// the rows); feature counts that are multiples of 64.
//
// What bounds such a product is the chain of dependent steps (load a slab of both operands, multiply,
// next slab), not the matrix cores: one sequence of the reference's training shape (256 rows, 384
// features) has 24 tiles of 6 steps. So a workgroup owns one 64 x 64 tile and its waves split the
// sum over k: every wave takes every unit of its own contiguous range of k, with its own 16 KB of
// LDS and no barrier, and the partial tiles meet in LDS once at the end, added in wave order (the
// result does not depend on timing). The destination is read and written once, by whole rows.
//
// A unit is 16 products of v_mfma_f32_32x32x16_bf16 (64 x 64 x 64, or 64 x 64 x 32 for the fp32 dQ,
// which is split into two bf16 terms hi = bf16(x), lo = bf16(x - hi) as in sublayer_gemm.hip, and
// runs twice). Its operands are copied global -> LDS by the hardware (global_load_lds_dwordx4, 1 KB
// an instruction), read into registers at once, and the next unit's copies are issued before the
// products. out[p][c] = sum_k A[c][k] B[p][k]; the operand tiles in LDS are
//   by rows  [64 idx][64 k], 128-byte rows: 16-byte reads of 8 k of one row
//   by k     [64 k][64 idx], 128-byte rows: ds_read_b64_tr_b16, 8 k of one column by two reads
// both XOR-swizzled in 16-byte chunks so that the reads are free of bank conflicts (counted: none, reads
// and writes; the matrix cores are busy 12-22% at 3840 x 448, 6-14% at 960 x 320).
#include <algorithm>

#include "attn_common.hpp"
#include "sublayer_tile.hpp"

namespace mla {

// sublayer_gemm.hip
hipError_t launch_grad_dw_reduce(const float* part, float* dQw, uint16_t* dKw, uint16_t* dVw, uint16_t* dPw, int C, int nq,
                                 int nkv, int w0, int nw, bool accumulate, hipStream_t s);

namespace {

constexpr int kWaveLds = 16384;

__device__ __forceinline__ u32x4 ld16(uint32_t a) { return *(const __attribute__((address_space(3))) u32x4*)(uintptr_t)a; }
__device__ __forceinline__ void st16(uint32_t a, u32x4 v) { *(__attribute__((address_space(3))) u32x4*)(uintptr_t)a = v; }
__device__ __forceinline__ u32x2 ldtr(uint32_t a) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(uintptr_t)a));
}

// LDS chunk of global chunk c in row r of a tile read by rows (16 lanes read 16 rows: distinct banks)
__device__ __forceinline__ int row_sw(int r) { return (r >> 1) & 7; }
// the same for a tile read by k (32 lanes read 64 bytes of 4 rows) and for 64-byte rows
__device__ __forceinline__ int col_sw(int r) { return 4 * ((r >> 1) & 1); }
__device__ __forceinline__ int half_sw(int r) { return (r >> 2) & 3; }

struct Lane {
  int lane, h, l32, g16, s16;
};

// A pointer that is the same in every lane, in scalar registers (the copies' base operand).
__device__ __forceinline__ const void* uniform_ptr(const void* p) {
  const uint64_t u = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return (const void*)(((uint64_t)hi << 32) | lo);
}

// dma16 (attn_common.hpp) with the wait states that the compiler does not insert before inline asm:
// one after a scalar write of m0, five after a vector write of the base registers.
__device__ __forceinline__ void copy16(uint32_t voff, const void* sbase, uint32_t m0) {
  asm volatile("s_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "{m0}"(m0) : "memory");
}

// ---- copies of a unit's operand tiles to LDS address `dst` ----
// 64 rows of 128 bytes: row r of the tile is src + min(r, last) * pitch (bytes)
template <bool BYK>
__device__ __forceinline__ void copy64(const Lane& L, const void* src, uint32_t pitch, int last, uint32_t dst) {
  src = uniform_ptr(src);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int r = 8 * i + (L.lane >> 3), p = L.lane & 7;
    copy16((uint32_t)min(r, last) * pitch + 16 * (p ^ (BYK ? col_sw(r) : row_sw(r))), src, dst + 1024 * i);
  }
}
// 64 rows of 64 bytes
__device__ __forceinline__ void copy_half(const Lane& L, const void* src, uint32_t pitch, uint32_t dst) {
  src = uniform_ptr(src);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 16 * i + (L.lane >> 2), p = L.lane & 3;
    copy16((uint32_t)r * pitch + 16 * (p ^ half_sw(r)), src, dst + 1024 * i);
  }
}
// 32 rows (k) of 128 bytes
__device__ __forceinline__ void copy32k(const Lane& L, const void* src, uint32_t pitch, uint32_t dst) {
  src = uniform_ptr(src);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 8 * i + (L.lane >> 3), p = L.lane & 7;
    copy16((uint32_t)r * pitch + 16 * (p ^ col_sw(r)), src, dst + 1024 * i);
  }
}

// ---- operand reads: idx 32t .. 32t+31 (lane l32), k 16ks + 8h .. +7 ----
__device__ __forceinline__ u32x4 read_row(const Lane& L, uint32_t a, int t, int ks) {
  const int r = 32 * t + L.l32;
  return ld16(a + r * 128 + 16 * ((2 * ks + L.h) ^ row_sw(r)));
}
__device__ __forceinline__ u32x4 read_half(const Lane& L, uint32_t a, int t, int ks) {
  const int r = 32 * t + L.l32;
  return ld16(a + r * 64 + 16 * ((2 * ks + L.h) ^ half_sw(r)));
}
__device__ __forceinline__ u32x4 read_k(const Lane& L, uint32_t a, int t, int ks) {
  const int r = 16 * ks + 8 * L.h + (L.s16 >> 2);  // + 4 for the second read: the same swizzle
  const int c = 4 * t + 2 * (L.g16 & 1) + ((L.s16 & 3) >> 1);
  const uint32_t ad = a + r * 128 + 16 * (c ^ col_sw(r)) + 8 * (L.s16 & 1);
  const u32x2 lo = ldtr(ad), hi = ldtr(ad + 4 * 128);
  return u32x4{lo[0], lo[1], hi[0], hi[1]};
}

// x = hi + lo in bf16 (|x - hi - lo| <= 2^-17 |x|)
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  hi = pack_bf16(a, b);
  lo = pack_bf16(a - bf_lo(hi), b - bf_hi(hi));
}

// This wave's copies have landed (no other wave reads them: no barrier).
__device__ __forceinline__ void wait_copies() {
  wait_vm<0>();
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void wait_lds() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0) only
  asm volatile("" ::: "memory");
}

template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}

// acc[tc][tp]: c 32tc + 8g + 4h + i (register 4g + i), p 32tp + l32
struct Acc {
  f32x16 v[2][2];
};

__device__ __forceinline__ void products(Acc& acc, const u32x4 (&A)[2], const u32x4 (&B)[2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc.v[i][j] = mfma(A[i], B[j], acc.v[i][j]);
}

// Adds the NW waves' tiles in wave order; put(row, column, four consecutive values) for each.
template <int NW, class Put>
__device__ __forceinline__ void reduce_tiles(const Lane& L, int tid, int wave, uint32_t smem, const Acc& acc, Put put) {
  // row p of a partial tile: 16 chunks of 4 floats, chunk c at c ^ (p & 15)
  const uint32_t mine = smem + wave * kWaveLds;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int p = 32 * j + L.l32, c = 8 * i + 2 * g + L.h;
        const f32x4 v = {acc.v[i][j][4 * g], acc.v[i][j][4 * g + 1], acc.v[i][j][4 * g + 2], acc.v[i][j][4 * g + 3]};
        st16(mine + p * 256 + 16 * (c ^ (p & 15)), __builtin_bit_cast(u32x4, v));
      }
  __syncthreads();
#pragma unroll
  for (int n = 0; n < 16 / NW; ++n) {
    const int e = tid + 64 * NW * n, p = e >> 4, c = e & 15;
    const uint32_t a = smem + p * 256 + 16 * (c ^ (p & 15));
    f32x4 s = __builtin_bit_cast(f32x4, ld16(a));
#pragma unroll
    for (int w = 1; w < NW; ++w) s += __builtin_bit_cast(f32x4, ld16(a + w * kWaveLds));
    put(p, 4 * c, s);
  }
}

__device__ __forceinline__ Lane lane_of(int tid) {
  Lane L;
  L.lane = tid & 63;
  L.h = L.lane >> 5;
  L.l32 = L.lane & 31;
  L.g16 = L.lane >> 4;
  L.s16 = L.lane & 15;
  return L;
}

// Item of workgroup bid: consecutive items on one XCD (workgroups are dealt to the 8 XCDs in turn),
// so that tiles which share rows share an L2. The grid is padded to a multiple of 8.
__device__ __forceinline__ int item_of(int bid, int grid) { return (bid & 7) * (grid >> 3) + (bid >> 3); }

__device__ __forceinline__ uint32_t lds_base(unsigned char* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) unsigned char*)p;
}

// ---- bf16 row products: Y[r][n] = sum_k X[r][k] W (WT: W[n][k], else W[k][n]), one to three weights ----
template <int NW, bool WT>
__global__ void __launch_bounds__(64 * NW, 2) tile_rows_kernel(TileRows a) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[NW * kWaveLds];
  const int item = item_of((int)blockIdx.x, (int)gridDim.x);
  const int nc = a.C / 64, nr = (a.R + 63) / 64;
  if (item >= nr * nc * a.n) return;
  const int rt = item / (nc * a.n), rest = item - rt * nc * a.n, y = rest / nc, ct = rest - y * nc;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Lane L = lane_of(tid);
  const uint32_t smem = lds_base(smem_raw), sx = smem + wave * kWaveLds, sw = sx + 8192;
  const uint32_t pitch = 2u * a.C;
  const int r0 = 64 * rt, c0 = 64 * ct;
  const char* X = (const char*)(a.x + (size_t)r0 * a.C);
  const char* W = (const char*)(a.w[y] + (WT ? (size_t)c0 * a.C : (size_t)c0));
  const int u0 = nc * wave / NW, u1 = nc * (wave + 1) / NW;
  auto issue = [&](int u) __attribute__((always_inline)) {
    copy64<false>(L, X + 128 * u, pitch, a.R - 1 - r0, sx);
    copy64<!WT>(L, WT ? W + 128 * u : W + (size_t)64 * u * pitch, pitch, 63, sw);
  };
  Acc acc;
#pragma unroll
  for (int i = 0; i < 4; ++i) acc.v[i >> 1][i & 1] = zero16();
  if (u0 < u1) issue(u0);
  for (int u = u0; u < u1; ++u) {
    wait_copies();
    u32x4 A[4][2], B[4][2];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        A[ks][t] = WT ? read_row(L, sw, t, ks) : read_k(L, sw, t, ks);
        B[ks][t] = read_row(L, sx, t, ks);
      }
    wait_lds();
    if (u + 1 < u1) issue(u + 1);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) products(acc, A[ks], B[ks]);
  }
  if (a.zero0 && item == 0)
    for (int i = tid; i < a.C; i += 64 * NW) a.zero0[i] = a.zero1[i] = 0.0f;
  uint16_t* out = a.y[y];
  reduce_tiles<NW>(L, tid, wave, smem, acc, [&](int p, int c, f32x4 s) {
    const bool live = r0 + p < a.R;
    const size_t o = (size_t)(live ? r0 + p : a.R - 1) * a.C + c0 + c;  // past the end: read in bounds, not stored
    const u32x2 v = {pack_bf16(s[0], s[1]), pack_bf16(s[2], s[3])};
    if (live) *(u32x2*)(out + o) = v;
    if (a.sum) {
      const u32x2 x = *(const u32x2*)(a.add + o);
      if (live)
        *(u32x2*)(a.sum + o) = u32x2{pack_bf16(bf_lo(x[0]) + bf_lo(v[0]), bf_hi(x[0]) + bf_hi(v[0])),
                                     pack_bf16(bf_lo(x[1]) + bf_lo(v[1]), bf_hi(x[1]) + bf_hi(v[1]))};
    }
    if (a.Dv) {
      // computeD's sum (attn_computed.hip) bit for bit: columns l and l + 32 first, from 0, then the
      // butterfly over the 32 sums. The 16 lanes of a row hold columns 4 k .. 4 k + 3 (k = lane % 16):
      // l + 32 is lane k + 8, distances 16, 8, 4 are lanes k ^ 4, k ^ 2, k ^ 1, and 2, 1 in-lane. The
      // rotations reach the partners because lanes k and k ^ 8 hold the same sums by then.
      const u32x2 y = *(const u32x2*)(a.O + o);
      const uint32_t p0 = pack_bf16(bf_lo(v[0]) * bf_lo(y[0]), bf_hi(v[0]) * bf_hi(y[0]));
      const uint32_t p1 = pack_bf16(bf_lo(v[1]) * bf_lo(y[1]), bf_hi(v[1]) * bf_hi(y[1]));
      float d[4] = {bf_lo(p0), bf_hi(p0), bf_lo(p1), bf_hi(p1)};
      const float zero = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (c < 32) d[i] = zero + d[i];
        d[i] += dpp_move<0x128>(d[i]);  // row_ror:8
        d[i] += dpp_move<0x124>(d[i]);  // row_ror:4
        d[i] += dpp_move<0x4e>(d[i]);   // quad_perm 2,3,0,1
        d[i] += dpp_move<0xb1>(d[i]);   // quad_perm 1,0,3,2
      }
      const float total = (d[0] + d[2]) + (d[1] + d[3]);
      if (live && c == 0) {
        const int r = r0 + p, b = r / a.T;
        a.Dv[((size_t)b * a.H + ct) * a.T + (r - b * a.T)] = bf_lo(pack_bf16(total, total));
      }
    }
  });
}

// ---- computeGradDx: dX[r][i] (+)= sum_j dQ[r][j] Wq[i][j] + dK[r][j] Wk[i][j] + dV[r][j] Wv[i][j] ----
template <int NW, bool ACC>
__device__ __forceinline__ void grad_dx_tile(unsigned char* smem_raw, const TileGrad& a, int item) {
  const int nb = a.C / 64, rt = item / nb, ct = item - rt * nb;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Lane L = lane_of(tid);
  const uint32_t smem = lds_base(smem_raw), sg = smem + wave * kWaveLds, sw = sg + 8192;
  const uint32_t pitch = 2u * a.C;
  const int r0 = 64 * rt, i0 = 64 * ct, last = a.R - 1 - r0;
  const size_t go = (size_t)r0 * a.C, wo = (size_t)i0 * a.C;
  // units: 2 nb of dQ (32 j each), nb of dK, nb of dV
  const int U = 4 * nb, u0 = U * wave / NW, u1 = U * (wave + 1) / NW;
  auto issue = [&](int u) __attribute__((always_inline)) {
    if (u < 2 * nb) {
      copy64<false>(L, (const char*)(a.dQ + go) + 128 * u, 2 * pitch, last, sg);
      copy_half(L, (const char*)(a.W[0] + wo) + 64 * u, pitch, sw);
    } else {
      const int s = u >= 3 * nb ? 2 : 1, b = u - (s + 1) * nb;
      copy64<false>(L, (const char*)(a.g[s] + go) + 128 * b, pitch, last, sg);
      copy64<false>(L, (const char*)(a.W[s] + wo) + 128 * b, pitch, 63, sw);
    }
  };
  Acc acc;
#pragma unroll
  for (int i = 0; i < 4; ++i) acc.v[i >> 1][i & 1] = zero16();
  if (u0 < u1) issue(u0);
  for (int u = u0; u < u1; ++u) {
    wait_copies();
    if (u < 2 * nb) {
      u32x4 A[2][2], F[2][2][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          A[ks][t] = read_half(L, sw, t, ks);
          const int r = 32 * t + L.l32, c = 4 * ks + 2 * L.h;  // 8 floats: chunks c, c + 1
          F[ks][t][0] = ld16(sg + r * 128 + 16 * (c ^ row_sw(r)));
          F[ks][t][1] = ld16(sg + r * 128 + 16 * ((c + 1) ^ row_sw(r)));
        }
      wait_lds();
      if (u + 1 < u1) issue(u + 1);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        u32x4 H[2], Lo[2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const u32x4& f = F[ks][t][q >> 1];
            uint32_t hi, lo;
            split2(__uint_as_float(f[2 * (q & 1)]), __uint_as_float(f[2 * (q & 1) + 1]), hi, lo);
            H[t][q] = hi;
            Lo[t][q] = lo;
          }
        products(acc, A[ks], H);
        products(acc, A[ks], Lo);
      }
    } else {
      u32x4 A[4][2], B[4][2];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          A[ks][t] = read_row(L, sw, t, ks);
          B[ks][t] = read_row(L, sg, t, ks);
        }
      wait_lds();
      if (u + 1 < u1) issue(u + 1);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) products(acc, A[ks], B[ks]);
    }
  }
  reduce_tiles<NW>(L, tid, wave, smem, acc, [&](int p, int c, f32x4 s) {
    if (p > last) return;
    f32x4* d = (f32x4*)(a.dX + (size_t)(r0 + p) * a.C + i0 + c);
    *d = (ACC ? *d : f32x4{0.0f, 0.0f, 0.0f, 0.0f}) + s;
  });
}

// ---- weight gradients: dW[w][i][j] (+)= sum_r x[w][r][i] G[r][j]; FP32: dQw, G the fp32 dQ ----
// over the rows of chunk `chunk` of nch.
template <int NW, bool ACC, bool FP32>
__device__ __forceinline__ void grad_dw_tile(unsigned char* smem_raw, const TileGrad& a, int w, int chunk, int nch,
                                             int tile) {
  const int nb = a.C / 64, it = tile / nb, jt = tile - it * nb;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Lane L = lane_of(tid);
  const uint32_t smem = lds_base(smem_raw), sx = smem + wave * kWaveLds, sg = sx + 8192;
  const uint32_t pitch = 2u * a.C;
  const int i0 = 64 * it, j0 = 64 * jt;
  const char* X = (const char*)(a.x[w] + i0);
  Acc acc;
#pragma unroll
  for (int i = 0; i < 4; ++i) acc.v[i >> 1][i & 1] = zero16();
  // the rows in units of 32 (FP32) or 64, this wave's share of the chunk's
  const int U = a.R / (FP32 ? 32 : 64), parts = nch * NW, part = chunk * NW + wave, each = U / parts, more = U - each * parts;
  const int u0 = each * part + min(part, more), u1 = u0 + each + (part < more ? 1 : 0);
  if constexpr (FP32) {
    // dQ: 32 rows of 64 floats through registers (each lane 8 words of 4 floats: row 4q + lane/16),
    // split and written as hi and lo tiles by k (32 rows of 128 bytes each)
    const float* G = a.dQ + j0;
    f32x4 f[8];
    auto fetch = [&](int u) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < 8; ++q)
        f[q] = *(const f32x4*)(G + (size_t)(32 * u + 4 * q + (L.lane >> 4)) * a.C + 4 * (L.lane & 15));
    };
    auto issue = [&](int u) __attribute__((always_inline)) { copy32k(L, X + (size_t)32 * u * pitch, pitch, sx); };
    if (u0 < u1) {
      fetch(u0);
      issue(u0);
    }
    for (int u = u0; u < u1; ++u) {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        uint32_t h0, l0, h1, l1;
        split2(f[q][0], f[q][1], h0, l0);
        split2(f[q][2], f[q][3], h1, l1);
        const int r = 4 * q + (L.lane >> 4), c = (L.lane & 15) >> 1;
        const uint32_t ad = sg + r * 128 + 16 * (c ^ col_sw(r)) + 8 * (L.lane & 1);
        *(__attribute__((address_space(3))) u32x2*)(uintptr_t)ad = u32x2{h0, h1};
        *(__attribute__((address_space(3))) u32x2*)(uintptr_t)(ad + 4096) = u32x2{l0, l1};
      }
      wait_copies();
      u32x4 A[2][2], Al[2][2], B[2][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          A[ks][t] = read_k(L, sg, t, ks);
          Al[ks][t] = read_k(L, sg + 4096, t, ks);
          B[ks][t] = read_k(L, sx, t, ks);
        }
      wait_lds();
      if (u + 1 < u1) {
        fetch(u + 1);
        issue(u + 1);
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        products(acc, A[ks], B[ks]);
        products(acc, Al[ks], B[ks]);
      }
    }
  } else {
    const char* G = (const char*)(a.g[w] + j0);
    auto issue = [&](int u) __attribute__((always_inline)) {
      copy64<true>(L, X + (size_t)64 * u * pitch, pitch, 63, sx);
      copy64<true>(L, G + (size_t)64 * u * pitch, pitch, 63, sg);
    };
    if (u0 < u1) issue(u0);
    for (int u = u0; u < u1; ++u) {
      wait_copies();
      u32x4 A[4][2], B[4][2];
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          A[ks][t] = read_k(L, sg, t, ks);
          B[ks][t] = read_k(L, sx, t, ks);
        }
      wait_lds();
      if (u + 1 < u1) issue(u + 1);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) products(acc, A[ks], B[ks]);
    }
  }
  reduce_tiles<NW>(L, tid, wave, smem, acc, [&](int p, int c, f32x4 s) {
    const size_t o = (size_t)(i0 + p) * a.C + j0 + c;
    if (a.part) {
      const int first = w == 0 ? 0 : (a.w0 == 0 ? a.nq + (w - 1) * a.nkv : 0);
      *(f32x4*)(a.part + (size_t)(first + chunk) * a.C * a.C + o) = s;
    } else if constexpr (FP32) {
      f32x4* d = (f32x4*)((float*)a.dW[0] + o);
      *d = (ACC ? *d : f32x4{0.0f, 0.0f, 0.0f, 0.0f}) + s;
    } else {
      u32x2* d = (u32x2*)((uint16_t*)a.dW[w] + o);
      const u32x2 old = ACC ? *d : u32x2{0u, 0u};
      *d = u32x2{pack_bf16(bf_lo(old[0]) + s[0], bf_hi(old[0]) + s[1]), pack_bf16(bf_lo(old[1]) + s[2], bf_hi(old[1]) + s[3])};
    }
  });
}

// Items of one launch: dQw's (tile by tile, chunk by chunk), the other weights', computeGradDx's tiles
// where dX is set. Workgroups are dealt to the 8 XCDs in turn; an XCD takes a contiguous eighth of each
// kind (rounded up: the last ones may be empty), the weight gradients' longer sums first. (A contiguous
// eighth of the whole list gave some XCDs only the long sums and others only computeGradDx's tiles.)
struct GradItems {
  int tiles, nq, nkv, nx;    // tiles of a weight; items of each kind (one list: all weights' in nq + nkv)
  int per_q, per_kv, per_x;  // an XCD's share
};
__host__ __device__ inline GradItems grad_items(const TileGrad& a) {
  GradItems g;
  const int nb = a.C / 64;
  g.tiles = nb * nb;
  g.nq = a.w0 == 0 && a.w1 > 0 ? g.tiles * a.nq : 0;
  g.nkv = g.tiles * a.nkv * (a.w1 - (a.w0 == 0 && a.w1 > 0 ? 1 : a.w0));
  g.nx = a.dX ? (a.R + 63) / 64 * nb : 0;
  const bool one_list = a.part && !a.dX;
  g.per_q = (g.nq + (one_list ? g.nkv : 0) + 7) / 8;
  g.per_kv = one_list ? 0 : (g.nkv + 7) / 8;
  g.per_x = (g.nx + 7) / 8;
  return g;
}

template <int NW, bool ACC>
__global__ void __launch_bounds__(64 * NW, 2) tile_grad_kernel(TileGrad a) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem_raw[NW * kWaveLds];
  const GradItems n = grad_items(a);
  const int x = blockIdx.x & 7;
  const int k = blockIdx.x >> 3;
  if (k < n.per_q + n.per_kv) {
    int item = k < n.per_q ? x * n.per_q + k : x * n.per_kv + k - n.per_q;
    if (k < n.per_q && item < n.nq) {
      const int chunk = item / n.tiles;
      grad_dw_tile<NW, ACC, true>(smem_raw, a, 0, chunk, a.nq, item - chunk * n.tiles);
      return;
    }
    if (k < n.per_q) {
      if (n.per_kv) return;  // past the end of dQw's own share
      item -= n.nq;
    }
    const int i = item / n.tiles, w = i / a.nkv;
    if (item < n.nkv)
      grad_dw_tile<NW, ACC, false>(smem_raw, a, w + max(a.w0, 1), i - w * a.nkv, a.nkv, item - i * n.tiles);
    return;
  }
  const int item = x * n.per_x + k - n.per_q - n.per_kv;
  if (item < n.nx) grad_dx_tile<NW, ACC>(smem_raw, a, item);
}

// Tiles up to which a workgroup has 8 waves (one workgroup per CU); beyond it 4, two workgroups per
// CU, whose first loads and last stores run beside the other's products.
constexpr unsigned kDeepItems = 256;

unsigned padded(int items) { return (unsigned)((items + 7) / 8 * 8); }

}  // namespace

hipError_t launch_tile_rows(const TileRows& a, bool wt, hipStream_t s) {
  const unsigned grid = padded((a.R + 63) / 64 * (a.C / 64) * a.n);
  const bool deep = grid <= kDeepItems;
  auto kern = wt ? (deep ? tile_rows_kernel<8, true> : tile_rows_kernel<4, true>)
                 : (deep ? tile_rows_kernel<8, false> : tile_rows_kernel<4, false>);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(deep ? 512 : 256), 0, s, a);
  return hipGetLastError();
}

namespace {

struct Chunks {
  int nq, nkv;
};

// Row chunks of the weight gradients: as many as bring a wave's chain of units (R / 64 / 4 for a
// bf16 weight, twice that for dQw) down to about half of what every wave of the chip has to do, when
// the undivided chain is longer than all of it (which `divide` takes for granted: the number of chunks
// then only grows with R).
Chunks grad_chunks(int R, int C, int w0, int w1, bool dx, bool divide = false) {
  if (w1 <= w0) return {1, 1};
  const double tiles = (double)(C / 64) * (C / 64), rows = R / 64.0;
  const double mean = tiles * rows * ((dx ? 4 : 0) + (w1 - w0) + (w0 == 0 ? 1 : 0)) / (256 * 8);
  const double chain = rows / 4 * (w0 == 0 ? 2 : 1);
  if (!divide && chain <= 1.25 * mean + 8) return {1, 1};
  const int n = (int)(rows / 4 / std::max(4.0, mean / 2) + 0.999);
  return {w0 == 0 ? std::max(1, 2 * n) : 0, std::max(1, n)};
}

size_t partial_floats(const Chunks& k, int C, int w0, int w1) {
  if (k.nkv == 1 && k.nq <= 1) return 0;
  return (size_t)(k.nq + (w1 - std::max(w0, 1)) * k.nkv) * C * C;
}

}  // namespace

size_t tile_grad_partial_floats(int R, int C, int w0, int w1, bool dx) {
  return partial_floats(grad_chunks(R, C, w0, w1, dx), C, w0, w1);
}

size_t tile_grad_partial_bound(int R, int C, int w0, int w1, bool dx) {
  return partial_floats(grad_chunks(R, C, w0, w1, dx, true), C, w0, w1);
}

hipError_t launch_tile_grad(TileGrad a, float* partial, bool accumulate, hipStream_t s) {
  const Chunks k = grad_chunks(a.R, a.C, a.w0, a.w1, a.dX != nullptr);
  a.nq = k.nq;
  a.nkv = k.nkv;
  a.part = k.nkv == 1 && k.nq <= 1 ? nullptr : partial;
  const GradItems n = grad_items(a);
  const unsigned grid = 8u * (unsigned)(n.per_q + n.per_kv + n.per_x);
  // computeGradDx's waves follow its own tile count alone: its sums are the same bit for bit with and
  // without weight gradients in the launch
  const bool deep = a.dX ? (unsigned)n.nx <= kDeepItems / 2 : grid <= kDeepItems;
  auto kern = accumulate ? (deep ? tile_grad_kernel<8, true> : tile_grad_kernel<4, true>)
                         : (deep ? tile_grad_kernel<8, false> : tile_grad_kernel<4, false>);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(deep ? 512 : 256), 0, s, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || !a.part) return e;
  if (a.w0 == 0)
    return launch_grad_dw_reduce(a.part, (float*)a.dW[0], (uint16_t*)a.dW[1], (uint16_t*)a.dW[2], (uint16_t*)a.dW[3], a.C,
                                 k.nq, k.nkv, 0, a.w1, accumulate, s);
  return launch_grad_dw_reduce(a.part, nullptr, (uint16_t*)a.dW[a.w0], nullptr, nullptr, a.C, 0, k.nkv, 1, 1, accumulate, s);
}

}  // namespace mla
