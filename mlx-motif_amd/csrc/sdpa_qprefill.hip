// Prompt-chunk kernels over the packed cache (sdpa_qprefill.hpp).
#include "sdpa_dispatch.hpp"
#include "sdpa_qprefill.hpp"

namespace motif {

template <int BITS, typename E>
static int launch_qprefill(const SdpaArgs& a, int waves, int ncb, int nblocks, hipStream_t st) {
  if (waves == 8 && ncb == 2)
    hipLaunchKernelGGL((sdpa_qprefill_kernel<BITS, E, 8, 2>), dim3(nblocks), dim3(512), 0, st, a);
  else if (waves == 8)
    hipLaunchKernelGGL((sdpa_qprefill_kernel<BITS, E, 8, 1>), dim3(nblocks), dim3(512), 0, st, a);
  else
    hipLaunchKernelGGL((sdpa_qprefill_kernel<BITS, E, 4, 1>), dim3(nblocks), dim3(256), 0, st, a);
  return check_launch("sdpa_dual_v_q (prompt chunk)");
}

int launch_sdpa_qprefill(const SdpaArgs& a, bool bf16, int bits, int waves, int ncb, int nblocks,
                         hipStream_t st) {
  if (bits == 4)
    return bf16 ? launch_qprefill<4, bf16_t>(a, waves, ncb, nblocks, st)
                : launch_qprefill<4, half_t>(a, waves, ncb, nblocks, st);
  return bf16 ? launch_qprefill<8, bf16_t>(a, waves, ncb, nblocks, st)
              : launch_qprefill<8, half_t>(a, waves, ncb, nblocks, st);
}

}  // namespace motif
