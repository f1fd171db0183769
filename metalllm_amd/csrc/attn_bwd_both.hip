// attn_bwd_both.hip -- both halves of flashAttentionBackward in one launch: workgroups [0, n1) own
// key blocks (dK/dV, attn_bwd_dkdv.hpp), the rest own query blocks (dQ recomputing the softmax,
// attn_bwd_dq.hpp). Neither half reads what the other writes.
//
// Few pairs leave most CUs idle and each half takes its longest chain of causal tiles; in one launch
// the two chains run side by side. Many pairs fill the chip with either half, and the launch saves
// the first grid's tail. Against the two launches: B=1, T=3008, H=5, D=128 with computeD 170 -> 104 us;
// B=1, T=2048, H=12, D=64 84 -> 53 us; B=8, T=2048, H=12, D=64, all CUs busy in both halves, takes 212
// us, bound by vector instruction issue like each half alone.
#include "attn_bwd_dkdv.hpp"
#include "attn_bwd_dq.hpp"

namespace mla {

// Occupancy of the two halves' own kernels: three workgroups per CU at D = 64, two at D = 128.
template <int D, bool ACC>
__global__ void __launch_bounds__(256, D == 64 ? 3 : 2) bwd_both_kernel(BwdArgs a, int n1) {
  constexpr int SM = BwdCfg<D>::SMEM > DqCfg<D>::SMEM ? BwdCfg<D>::SMEM : DqCfg<D>::SMEM;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[SM];
  const int bid = (int)blockIdx.x;
  if (bid < n1)
    bwd_body<D, false>(smem, bid, a);
  else
    bwd_dq_body<D, ACC>(smem, both_dq_index(bid, n1, (int)gridDim.x, D == 64 ? 3 : 2), a);
}

hipError_t launch_backward_both(const BwdArgs& a, int D, bool accumulate, hipStream_t s) {
  const int pairs = a.B * a.H;
  const int n1 = pairs * ((a.T + kBwdBlockN - 1) / kBwdBlockN), n2 = pairs * ((a.T + kDqBlockM - 1) / kDqBlockM);
  auto kern = D == 64 ? (accumulate ? bwd_both_kernel<64, true> : bwd_both_kernel<64, false>)
                      : (accumulate ? bwd_both_kernel<128, true> : bwd_both_kernel<128, false>);
  hipLaunchKernelGGL(kern, dim3((unsigned)(n1 + n2)), dim3(256), 0, s, a, n1);
  return hipGetLastError();
}

}  // namespace mla
