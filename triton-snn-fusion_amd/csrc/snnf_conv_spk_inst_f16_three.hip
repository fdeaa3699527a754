// Instantiates the blocked-layout conv+LIF kernel for f16_t activations, three timesteps side by side.
#include "snnf_conv_spk_kernel.h"

namespace snnf {
int launch_conv_spk_f16_three(const SpkLaunch& L) {
    return L.g.in_layout == SNNF_LAYOUT_BITS ? launch_conv_spk_variant<f16_t, 3, SNNF_LAYOUT_BITS>(L) : launch_conv_spk_variant<f16_t, 3, SNNF_LAYOUT_C8>(L);
}
int launch_conv_spk_f16_three_shortcut(const SpkLaunch& L) { return launch_conv_spk_shortcut<f16_t, 3>(L); }
}  // namespace snnf
