// Near-field kernels of the Helmholtz single layer potential.
#include "nf_device.h"

namespace h2hip {
namespace nf {

int launch_helmholtz_slp(int rb, int cb, uint32_t q, const KArgs &a,
                         uint32_t ntiles, const SPair *sp,
                         const uint32_t *ncls, hipStream_t stream) {
  return launch_family<K_HELM_SLP>(rb, cb, q, a, ntiles, sp, ncls, stream);
}

}  // namespace nf
}  // namespace h2hip
