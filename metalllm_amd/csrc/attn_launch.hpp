// attn_launch.hpp -- host-side launch interface between the C ABI (attn_abi.hip) and the
// kernels (attn_fwd.hip, attn_bwd.hip, attn_computed.hip). Shapes arrive validated.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mla {

// Q/K/V/O/dO/dQ/dK/dV are [B,T,H,D] (row of one token = H*D elements); LSE and D are [B,H,T].
struct FwdArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* out;
  float* lse;
  int T, H, B;
  float scale;  // 1/sqrt(D) in fp32, as the reference computes it (attention.metal:109)
};

struct ComputeDArgs {
  const uint16_t* dO;
  const uint16_t* O;
  float* Dv;
  int T, H, B;
  // optional: n_zero floats each set to 0 by the same launch (the phase encoder's layernorm gradients)
  float* zero0 = nullptr;
  float* zero1 = nullptr;
  uint32_t n_zero = 0;
};

struct BwdArgs {
  const uint16_t* dO;
  const float* Dv;
  const float* lse;
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  float* dQ;
  uint16_t* dK;
  uint16_t* dV;
  int T, H, B;
  float scale;
  // Optional: the dS tiles of the causal lower triangle, bf16, written by launch_backward and
  // read by launch_backward_dqs (ds_scratch_bytes(); layout in attn_bwd_dqs.hip). NULL: not stored.
  uint16_t* dS = nullptr;
};

// Bytes of the dS tile store for B*H pairs of T rows: one 64x64 bf16 tile per (query tile,
// key tile <= query tile) of every pair.
inline size_t ds_scratch_bytes(int B, int H, int T) {
  const size_t nqt = (size_t)T / 64;
  return (size_t)B * H * (nqt * (nqt + 1) / 2) * 8192;
}

hipError_t launch_forward(const FwdArgs& a, int D, hipStream_t s);
void forward_prepare();  // device queries of launch_forward, done ahead of a stream capture
hipError_t launch_compute_d(const ComputeDArgs& a, int D, hipStream_t s);
hipError_t launch_backward(const BwdArgs& a, int D, hipStream_t s);     // dK, dV (key-owner)
// dQ (query-owner, recomputing dS): added into dQ (accumulate) or written
hipError_t launch_backward_dq(const BwdArgs& a, int D, bool accumulate, hipStream_t s);
hipError_t launch_backward_dqs(const BwdArgs& a, int D, hipStream_t s); // dQ from the stored dS
// launch_backward (without the dS store) and launch_backward_dq in one launch, the same results
hipError_t launch_backward_both(const BwdArgs& a, int D, bool accumulate, hipStream_t s);
// Short sequences (D = 64, T <= 256): dK, dV and dQ of a (b,h) pair by one workgroup per CU, one
// launch, no workspace; dQ added into (accumulate) or written. It takes the same time for each round of
// kCus pairs, full or not (T = 128, 192, 256: 10.3, 15.7, 21.5 us), and a little for the first;
// bwd_both_kernel takes a time per pair, which grows by a fifth where a call's tensors exceed what the
// caches hold (from 350000 rows on), as it reads the inputs twice. So this kernel is the faster one
// where its rounds are nearly full, by more the larger the call. us, this kernel against the other,
// dQ written / added into:
//   T = 256: 240 pairs 24.9 / 25.6 against 26.3 / 26.5, 320 42.0 / 43.1 against 31.9 / 33.5, 768 65.2 /
//     66.6 against 66.2 / 72.0, 1536 142 / 150 against 158 / 169, 3072 273 / 287 against 325 / 354
//   T = 192: 448 33.0 / 33.9 against 32.9 / 34.5, 512 34.4 / 35.1 against 36.6 / 39.1, 640 46.6 / 48.0 against
//     44.9 / 47.5, 1280 76 / 78 against 84 / 90, 3072 201 / 215 against 246 / 267
//   T = 128: 768 33.2 / 33.9 against 31.9 / 34.7, 1024 41.7 / 42.7 against 43.4 / 45.1, 2048 79.7 / 82.9 against
//     79.2 / 85.4, 4096 173 / 184 against 199 / 220
//   T = 64: 1024 23.9 / 25.0 against 23.3 / 24.5, 6144 176 / 187 against 146 / 169
// Defined below, at kCus.
__host__ __device__ inline bool backward_is_short(int T, int D, int pairs);
// Whether the workspace entry point runs the recomputing kernels (dK/dV without the dS store and dQ
// written, in one launch) instead of the dS round trip. Yes at D = 64: the dK/dV kernel without the
// store runs three workgroups per CU and the pair is faster (config 2 step 0.436 -> 0.41 ms, config
// 4's 0.733 -> 0.716 ms). At D = 128 the round trip saves two of the seven products but needs its two
// kernels in sequence: it loses while the grid's longest chains, not its products, set the time,
// which is the case up to two blocks of 128 rows per CU (1 x 8 x 1024: 39.9 against 58.8 us; 1 x 8 x
// 8192, 512 blocks: 466 against 528; 640 blocks of T = 2048: 190 against 184; 1024: 489 against 428),
// and up to one and a half where T < 512 (384 blocks of T = 128, 256, 384: 34.4, 38.3, 41.2 against
// 33.6, 38.5, 44.4 us; 512 blocks: 43.2, 53.1, 55.3 against 38.8, 45.3, 52.6).
inline bool workspace_recomputes(int T, int D, int pairs);
hipError_t launch_backward_short(const BwdArgs& a, bool accumulate, hipStream_t s);

// Dispatch chunk sizes, in workgroups per XCD group. The backward's is one round of resident
// workgroups: two per CU on the 32 CUs of an MI355X XCD (the three-per-CU D = 64 kernels use the
// same figure). The forward's is two rounds: measured at T = 4096, D = 128 with one round per
// chunk, two and four, the forward took 1.345, 1.275 and 1.29 ms and the dK/dV kernel 2.31,
// 2.39 and 2.37 ms.
constexpr int kFwdDispatchRound = 128;
constexpr int kBwdDispatchRound = 64;
// At D = 64 the backward's kernels (dK/dV without the dS store, the recomputing dQ kernel) run
// three workgroups per CU, 96 per XCD, and their chunks span two such rounds. Measured on one box
// (the workspace backward at config 2 and at config 4's attention shape): chunks of 64, 96, 192
// workgroups and all of an XCD's pairs in one chunk gave 0.317, 0.325, 0.306, 0.303 ms and 0.263,
// 0.272, 0.240, 0.239 ms; with 64 the last chunk's long blocks started late and ran alone.
constexpr int kBwdDispatchRound64 = 192;
__host__ __device__ inline int bwd_dispatch_round(int D) { return D == 64 ? kBwdDispatchRound64 : kBwdDispatchRound; }

// Pairs per dispatch chunk: enough that one chunk's blocks fill a round of resident workgroups.
__host__ __device__ inline int dispatch_chunk(int nblk, int group_slots) {
  const int c = (group_slots + nblk - 1) / nblk;
  return c > 1 ? c : 1;
}

// Workgroup -> (pair = b*H + h, block) decode shared by host tests and kernels. Pairs are
// spread so that every block of one pair lands on the same XCD (workgroups are handed to the
// 8 XCDs round-robin by id). A group's pairs are taken in chunks of dispatch_chunk(nblk, round)
// pairs (round: workgroups per XCD group, kFwdDispatchRound or bwd_dispatch_round(D)); inside
// a chunk the blocks go out block-major, the largest causal work first, across the chunk's pairs:
//   forward : block = query block, longest (last) first
//   backward: block = key block, longest (first) first
// The hardware starts workgroups in id order as slots free up, so the long blocks of the last
// pairs no longer start late and run alone at the end (pair by pair, the tail was up to one long
// block), while the workgroups running at once still share a few pairs' tiles in L2.
__host__ __device__ inline void decode_workgroup(int bid, int npairs, int nblk, bool last_first, int round,
                                                 int& pair, int& blk) {
  const bool grouped = (npairs & 7) == 0;  // 8 groups, one per XCD
  const int g = grouped ? 8 : 1;
  const int x = grouped ? (bid & 7) : 0, slot = grouped ? (bid >> 3) : bid;
  const int npx = npairs / g;  // pairs of this group
  const int C = dispatch_chunk(nblk, grouped ? round : 8 * round);
  const int chunk = slot / (C * nblk);
  const int r = slot - chunk * C * nblk;
  const int cc = C < npx - chunk * C ? C : npx - chunk * C;  // pairs in this chunk (the last may be short)
  const int local = r / cc;
  pair = (chunk * C + (r - local * cc)) * g + x;
  blk = last_first ? (nblk - 1 - local) : local;
}

// Workgroups are dealt to the XCDs in turn and, inside an XCD, to its CUs in turn while they are
// free: ids that differ by a multiple of kCus start on the same CU.
constexpr int kCus = 256;
static_assert((kCus & (kCus - 1)) == 0, "rows of kCus ids by masks (fwd_item_of)");

__host__ __device__ inline bool backward_is_short(int T, int D, int pairs) {
  const int rounds = (pairs + kCus - 1) / kCus;
  const bool large = (int64_t)pairs * T >= 350000;
  const int fill = T == 256 ? (large ? 88 : 93) : T == 192 ? (large ? 85 : 90) : (large ? 90 : 95);  // percent
  return D == 64 && T >= 128 && T <= 256 && rounds >= (T == 256 ? 1 : T == 192 ? 2 : 4) &&
         (int64_t)pairs * 100 >= (int64_t)fill * kCus * rounds;
}

// Item k of workgroup `bid` of a persistent grid of `grid` workgroups over npairs x nblk
// (pair, block) items; false when the workgroup has fewer than k + 1 items. When both the pair
// count and the grid are multiples of 8, the workgroups on XCD x (bid % 8 == x) serve the pairs
// p = x (mod 8), so all blocks of a pair share one L2; otherwise all workgroups form one group.
// With two items or more per workgroup a group's items are listed pair by pair, each pair's last
// (largest causal) block first, and dealt in snake order over its workgroups: every workgroup gets
// about the same work, and the workgroups running at once share a few pairs' tiles in L2. With fewer
// the list goes block by block, longest first, and its first W items snake over rows of one
// workgroup per CU, so that the workgroups that share a CU have about the same work together. (Pair
// by pair, the workgroups w, w + 256 and w + 512 of 12 pairs of T = 8192 all had blocks of the same
// length and the CUs with the longest three took twice the mean: 204 us.) Shifts for the groups of 8 and
// the rows: the smallest calls wait for this arithmetic (one division is left).
__host__ __device__ inline bool fwd_item_of(int bid, int grid, int k, int npairs, int nblk, int& pair, int& blk) {
  const int sh = ((npairs | grid) & 7) == 0 ? 3 : 0;  // 8 groups or one
  const int x = bid & ((1 << sh) - 1), W = grid >> sh, n = (npairs >> sh) * nblk;
  int w = bid >> sh;
  const bool few = n < 2 * W;
  if (few) {
    const int row = kCus >> sh, at = w & ~(row - 1);  // the row's first id
    if (w & row) {                                    // every second row's ids in reverse
      const int end = at + row < W ? at + row : W;
      w = at + (end - 1 - w);
    }
  }
  const int m = k * W + ((k & 1) ? W - 1 - w : w);
  if (m >= n) return false;
  const int per = few ? npairs >> sh : nblk;
  const int i = m / per, j = m - i * per;
  pair = ((few ? j : i) << sh) + x;
  blk = nblk - 1 - (few ? i : j);
  return true;
}

// Index in the dQ grid of workgroup `bid` >= n1 of a grid of `grid` workgroups whose first n1 own
// key blocks (bwd_both_kernel). Both grids go longest first. When all workgroups start at once (at
// most `slots` per CU), the dQ blocks of every second row of kCus ids go shortest first instead, so
// that a CU which starts a long block gets a short one beside it; eight ids at a time where the
// grids are dealt by XCD (decode_workgroup), so that an id keeps its XCD.
__host__ __device__ inline int both_dq_index(int bid, int n1, int grid, int slots) {
  const int row = bid / kCus, i = bid - n1;
  if ((row & 1) == 0 || grid > slots * kCus) return i;
  const int lo = (row * kCus > n1 ? row * kCus : n1) - n1;
  const int hi = ((row + 1) * kCus < grid ? (row + 1) * kCus : grid) - n1;
  if (((n1 | grid) & 7) != 0) return lo + (hi - 1 - i);
  return lo + (hi - 8 - (i & ~7)) + (i & 7);
}

constexpr int kFwdBlockM = 128;  // query rows per forward workgroup
// The forward runs persistent (each resident workgroup takes items in turn, the next item's first
// tiles loaded during the current item's last step) when there are at most this many (pair, query
// block) items per resident workgroup; with more, one workgroup per item in the chunked dispatch
// order balances better. Measured: persistent faster at two items per slot (config 1, and config
// 4's attention, 0.0855 against 0.090 ms), one workgroup per item faster at four (config 2,
// 0.110 against 0.1155 ms) and at sixteen (T = 4096, D = 128).
constexpr int kFwdPersistItems = 2;
constexpr int kBwdBlockN = 128;  // keys owned by one dK/dV workgroup

inline bool workspace_recomputes(int T, int D, int pairs) {
  return D == 64 || (int64_t)pairs * ((T + kBwdBlockN - 1) / kBwdBlockN) <= (T >= 512 ? 2 * kCus : kCus * 3 / 2);
}

constexpr int kDqBlockM = 128;   // query rows owned by one dQ workgroup
constexpr int kTile = 64;        // the reference's TILE_M = TILE_N (attention.metal:14-15)

}  // namespace mla
