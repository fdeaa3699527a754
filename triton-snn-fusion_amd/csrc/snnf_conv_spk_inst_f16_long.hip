// Instantiates the blocked-layout conv+LIF kernel for f16_t activations, five and six timesteps in one window.
#include "snnf_conv_spk_kernel.h"

namespace snnf {
int launch_conv_spk_f16_long(const SpkLaunch& L) {
    return L.g.in_layout == SNNF_LAYOUT_BITS ? launch_conv_spk_long<f16_t, 6, SNNF_LAYOUT_BITS>(L) : launch_conv_spk_long<f16_t, 6, SNNF_LAYOUT_C8>(L);
}
}  // namespace snnf
