// The producer / consumer kernel (mid_kernel.h), fp16, gate/up.
#include "mid_kernel.h"

namespace fsw {

hipError_t launch_mid_fp16_gateup(const MidPlan& p, const GemmArgs& a, int ph, hipStream_t stream) {
  return launch_mid_typed<Fp16, true>(p, a, ph, stream);
}

}  // namespace fsw
