// Instantiates the blocked-layout conv+LIF kernel for bf16_t activations, three timesteps side by side.
#include "snnf_conv_spk_kernel.h"

namespace snnf {
int launch_conv_spk_bf16_three(const SpkLaunch& L) {
    return L.g.in_layout == SNNF_LAYOUT_BITS ? launch_conv_spk_variant<bf16_t, 3, SNNF_LAYOUT_BITS>(L) : launch_conv_spk_variant<bf16_t, 3, SNNF_LAYOUT_C8>(L);
}
int launch_conv_spk_bf16_three_shortcut(const SpkLaunch& L) { return launch_conv_spk_shortcut<bf16_t, 3>(L); }
}  // namespace snnf
