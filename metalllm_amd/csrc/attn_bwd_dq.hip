// attn_bwd_dq.hip -- the kernel of flashAttentionBackward's dQ half by itself (attn_bwd_dq.hpp holds a
// workgroup's body): the second of two launches where outputs are in inputs' memory, and a part.
#include "attn_bwd_dq.hpp"

namespace mla {

template <int D, bool ACC>
__global__ void __launch_bounds__(256, 2) bwd_dq_kernel(BwdArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[DqCfg<D>::SMEM];
  bwd_dq_body<D, ACC>(smem, (int)blockIdx.x, a);
}

hipError_t launch_backward_dq(const BwdArgs& a, int D, bool accumulate, hipStream_t s) {
  const int nqb = (a.T + kDqBlockM - 1) / kDqBlockM;
  const dim3 grid((unsigned)(a.B * a.H * nqb));
  if (D == 64) {
    if (accumulate)
      hipLaunchKernelGGL((bwd_dq_kernel<64, true>), grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((bwd_dq_kernel<64, false>), grid, dim3(256), 0, s, a);
  } else {
    if (accumulate)
      hipLaunchKernelGGL((bwd_dq_kernel<128, true>), grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((bwd_dq_kernel<128, false>), grid, dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

}  // namespace mla
