// Near-field kernels of the Helmholtz double layer (and adjoint double layer) potential on
// surfaces whose triangles are very short against the wave length (FP64).
#include "nf_device.h"

namespace h2hip {
namespace nf {

int launch_helmholtz_dlp_tp(int rb, int cb, uint32_t q, const KArgs &a,
                            uint32_t ntiles, const SPair *sp,
                            const uint32_t *ncls, hipStream_t stream) {
  return launch_family<K_HELM_DLP_TP>(rb, cb, q, a, ntiles, sp, ncls, stream);
}

}  // namespace nf
}  // namespace h2hip
