// attn_bwd.hip -- the kernels of flashAttentionBackward's dK/dV half (attn_bwd_dkdv.hpp holds a
// workgroup's body) and the fused backward of short sequences.
#include <algorithm>

#include "attn_bwd_dkdv.hpp"

namespace mla {

// D = 64 without the dS store: three workgroups per CU (168 VGPRs, a few spilled outside the
// product loop), 6-8% faster than two. D = 128 needs its 244-253 VGPRs and runs two. Without the dS
// store these run where outputs are in inputs' memory (the joint launch needs them apart), and as parts.
template <int D, bool DS>
__global__ void __launch_bounds__(256, D == 64 ? 3 : 2) bwd_kernel(BwdArgs a) {
  static_assert(D == 128 || !DS, "no dS is stored at D = 64");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[BwdCfg<D>::SMEM];
  bwd_body<D, DS>(smem, (int)blockIdx.x, a);
}

// Short sequences (D = 64, T <= 256, the reference's own length, where the pairs nearly fill their
// rounds: backward_is_short; and outputs in inputs' memory): one persistent workgroup of 8 waves per
// CU takes (b,h) pairs in turn and does each pair's whole backward, in one launch and without a
// workspace. LDS holds all query tiles of the pair (bwd_kernel's stage layout, one stage per tile),
// the pair's K rows and the dS tiles of one query tile.
//   * Step qt (all waves in step): wave w owns one 32-key group and, when the group lies at or
//     below query tile qt, runs the DkdvWave step on it and leaves its dS tile in LDS (the
//     workspace's layout, swizzled as the dQ-from-dS kernel's copies are). Waves w and w + 4
//     share a SIMD and own key groups g and nkg - 1 - g.
//   * Then waves 0-3, one per SIMD, compute dQ of query tile qt = dS.K over its key tiles (a
//     32 d x 32 query block each), in the order of attn_bwd_dqs.hip.
//   * The next pair's tile qt - 1 is copied into the stage step qt - 1 freed, and its K and V rows
//     are loaded after the last step, so every copy has the rest of the pair to land.
// dK and dV are bit-identical to bwd_kernel's, dQ to the dQ-from-dS kernel's; with ACC the result
// is added into dQ (flashAttentionBackward's contract), else written.
constexpr int kShortT = 256;
constexpr int kShortQT = kShortT / 64;

template <bool ACC>
__global__ void __launch_bounds__(512, 1) bwd_short_kernel(BwdArgs a) {
  constexpr int D = 64;
  using C = BwdCfg<D>;
  constexpr int KREG = kShortQT * C::STAGE;   // K rows of the pair: key * 2D bytes, 32 KB
  constexpr int DSB = KREG + kShortT * 2 * D;  // dS tiles (qt, kt) of the current query tile at DSB + kt * 8 KB
  static_assert(C::STAGE % 1024 == 0 && C::TBYTES % 1024 == 0 && KREG % 1024 == 0 && DSB % 1024 == 0, "1 KB granules");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[DSB + kShortQT * 8192];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5, l32 = lane & 31, g16 = lane >> 4, s16 = lane & 15;
  const int npairs = a.B * a.H;
  const int rs = a.H * D;
  const size_t tile_bytes = (size_t)C::BM * rs * 2;
  const int nqt = a.T / 64, nkg = a.T / 32;
  const uint32_t smem_a = lds_addr_b(smem);
  auto base_of = [&](int pair) -> size_t {
    const int b = pair / a.H, hd = pair - b * a.H;
    return ((size_t)b * a.T * a.H + hd) * D;
  };

  // Stage copies: 2*PER row instructions (Q then dO, bwd_kernel's padded slot order) spread over
  // the 8 waves, instruction n by wave n % 8; lse and D by wave 2 (lanes 0-15 and 16-31; 32-63
  // repeat them).
  constexpr int PER = C::TBYTES / 1024;
  constexpr int NCP = (2 * PER + 7) / 8;
  uint32_t off[NCP];
#pragma unroll
  for (int j = 0; j < NCP; ++j) {
    const int n = wave + 8 * j, i = n >= PER ? n - PER : n;
    const int sl = 64 * i + lane, row = sl / C::SLOTS, c = min(sl % C::SLOTS, D / 8 - 1);
    off[j] = (uint32_t)(row * rs * 2 + c * 16);
  }
  auto issue_tile = [&](int pair, int qt) {  // tile qt of `pair` into stage qt
    const size_t bq = base_of(pair) * 2 + (size_t)qt * tile_bytes;
    const uint32_t dst = smem_a + qt * C::STAGE;
#pragma unroll
    for (int j = 0; j < NCP; ++j) {
      const int n = wave + 8 * j;
      if (n < 2 * PER) {
        const bool go = n >= PER;
        const int i = go ? n - PER : n;
        dma16(off[j], (const char*)(go ? a.dO : a.q) + bq, dst + (go ? C::TBYTES : 0) + 1024 * i);
      }
    }
    if (wave == 2) {
      const float* src = (l32 < 16 ? a.lse : a.Dv) + (size_t)pair * a.T + qt * C::BM + 4 * (l32 & 15);
      dma16_v(src, dst + C::STAT);
    }
  };

  // key group of this wave: g and nkg - 1 - g share a SIMD (waves w and w + 4)
  const int g = wave < 4 ? (wave < nkg ? wave : -1) : (nkg - 1 - (wave - 4) >= 4 ? nkg - 1 - (wave - 4) : -1);
  const int kt = g >> 1, hw = g & 1;
  const int key = 32 * (g < 0 ? 0 : g) + l32;
  // dQ block of waves 0-3: d half wd, query half nq (32 d x 32 queries of the query tile)
  const int wd = wave & 1, nq = (wave >> 1) & 1;
  // operand lanes as in attn_bwd_dqs.hip; K row r holds chunk p at LDS chunk p ^ kx(r)
  auto kx = [](int r) { return 4 * ((r >> 1) & 1); };
  const int ra = 8 * (g16 >> 1) + (s16 >> 2);
  const int ca = (wd * 32) / 8 + 2 * (g16 & 1) + ((s16 & 3) >> 1);
  const uint32_t a_lane = (uint32_t)(ra * 2 * D + 16 * (ca ^ kx(ra)) + 8 * (s16 & 1));
  const int cr = 2 * (g16 & 1) + ((s16 & 3) >> 1), slq = 8 * (g16 >> 1) + (s16 >> 2);
  uint32_t b_lane[2];
#pragma unroll
  for (int hi = 0; hi < 2; ++hi)
    b_lane[hi] = (uint32_t)(cr * 1024 + 16 * ((slq + 4 * hi) ^ (4 * cr)) + 8 * (s16 & 1) + (32 * nq) * 16);
  const int qin = 32 * (l32 >> 4) + 8 * ((l32 >> 2) & 3) + 4 * nq + (l32 & 3);  // this lane's query row

  int pair = blockIdx.x;
  if (pair >= npairs) return;
  DkdvWave<D, true> wv;
  wv.init(lane, key, a.scale);
  for (int t = 0; t < nqt; ++t) issue_tile(pair, t);
  if (g >= 0) wv.load_rows(a.k + base_of(pair), a.v + base_of(pair), key, rs);
  for (;;) {
    const size_t base = base_of(pair);
    const int next = pair + (int)gridDim.x;
    const bool more = next < npairs;
    __builtin_amdgcn_s_waitcnt(0);  // this pair's tiles and rows (copied during the previous pair)
    if (wave == 2) {                // lse -> lse*log2(e), by the wave that copied it: exponents are base 2
      for (int t = 0; t < nqt; ++t) {
        float* l2 = (float*)(smem + t * C::STAGE + C::STAT);
        l2[lane] = l2[lane] * kLog2e;
      }
    }
    if (g >= 0) {
#pragma unroll
      for (int c = 0; c < C::KC; ++c)
        *(__attribute__((address_space(3))) u32x4*)(uintptr_t)(smem_a + KREG + key * 2 * D + 16 * ((2 * c + h) ^ kx(key))) =
            wv.Kr[c];
    }
    __syncthreads();

    for (int qt = 0; qt < nqt; ++qt) {
      if (qt >= 1 && more) issue_tile(next, qt - 1);  // stage qt - 1 was last read in step qt - 1
      // dK/dV step of the wave's key group; its dS tile (qt, kt) into LDS
      if (g >= 0 && kt <= qt) {
        if (qt == kt)
          wv.template qtile<true>(qt, smem_a + qt * C::STAGE, NoDsSink{});
        else
          wv.template qtile<false>(qt, smem_a + qt * C::STAGE, NoDsSink{});
        const LdsDsSink sink{smem_a + DSB + (uint32_t)(kt * 8192 + hw * 4096), 16u * lane, true};
#pragma unroll
        for (int s = 0; s < 4; ++s) sink.store(s, wv.dS);
      }
      __syncthreads();  // every dS tile of query tile qt is in LDS
      if (wave < 4) {
        float* dQg = a.dQ + base + (size_t)qt * 64 * rs + wd * 32 + 4 * h + (size_t)qin * rs;
        f32x4 old[4];
        if (ACC) {  // loads in flight during the products
#pragma unroll
          for (int gg = 0; gg < 4; ++gg) old[gg] = *(const f32x4*)(dQg + 8 * gg);
        }
        // products i = 4 k2 + ks in order, each one's operands read one product ahead
        auto operands = [&](int i, u32x4& A, u32x4& Bv) {
          const int k2 = i >> 2, ks = i & 3;
          const uint32_t da = smem_a + DSB + k2 * 8192 + b_lane[0] + 4 * (ks >> 1) * 1024 + (16 * (ks & 1)) * 16;
          const uint32_t ad = smem_a + KREG + k2 * 8192 + a_lane + 16 * ks * 2 * D;
          const u32x2 blo = lds_tr_b(da), bhi = lds_tr_b(da - b_lane[0] + b_lane[1]);
          const u32x2 alo = lds_tr_b(ad), ahi = lds_tr_b(ad + 4 * 2 * D);
          A = u32x4{alo[0], alo[1], ahi[0], ahi[1]};
          Bv = u32x4{blo[0], blo[1], bhi[0], bhi[1]};
        };
        f32x16 acc = zero16();
        const int np = 4 * (qt + 1);
        u32x4 A0, B0, A1, B1;
        operands(0, A0, B0);
        for (int i = 0; i < np; i += 2) {  // np is a multiple of 4
          operands(i + 1, A1, B1);
          acc = mfma(A0, B0, acc);
          if (i + 2 < np) operands(i + 2, A0, B0);
          acc = mfma(A1, B1, acc);
        }
        // the stored dS are 8 dS (power-of-two scale folded): dQ = acc / 8 exactly
#pragma unroll
        for (int gg = 0; gg < 4; ++gg) {
          f32x4 v = f32x4{acc[4 * gg], acc[4 * gg + 1], acc[4 * gg + 2], acc[4 * gg + 3]} * 0.125f;
          if (ACC) v = old[gg] + v;
          *(f32x4*)(dQg + 8 * gg) = v;
        }
      }
      __syncthreads();  // the dS tiles are free for the next step
    }
    if (g >= 0) {
      wv.finish();
      wv.store_rows(a.dK + base + (size_t)key * rs, a.dV + base + (size_t)key * rs);
    }
    if (!more) break;
    issue_tile(next, nqt - 1);
    wv.init(lane, key, a.scale);
    if (g >= 0) wv.load_rows(a.k + base_of(next), a.v + base_of(next), key, rs);
    pair = next;
  }
}

hipError_t launch_backward_short(const BwdArgs& a, bool accumulate, hipStream_t s) {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
      cus <= 0)
    return hipErrorInvalidDevice;
  const dim3 grid((unsigned)std::min(a.B * a.H, cus));  // one persistent workgroup per CU
  if (accumulate)
    hipLaunchKernelGGL((bwd_short_kernel<true>), grid, dim3(512), 0, s, a);
  else
    hipLaunchKernelGGL((bwd_short_kernel<false>), grid, dim3(512), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_backward(const BwdArgs& a, int D, hipStream_t s) {
  const int nkb = (a.T + kBwdBlockN - 1) / kBwdBlockN;
  const dim3 grid((unsigned)(a.B * a.H * nkb));
  if (a.dS) {
    if (D == 64) return hipErrorInvalidValue;
    hipLaunchKernelGGL((bwd_kernel<128, true>), grid, dim3(256), 0, s, a);
  } else {
    if (D == 64)
      hipLaunchKernelGGL((bwd_kernel<64, false>), grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((bwd_kernel<128, false>), grid, dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

}  // namespace mla
