// Instantiates the blocked-layout conv+LIF kernel for bf16_t activations and dense frames, one per timestep.
#include "snnf_conv_spk_kernel.h"

namespace snnf {
int launch_conv_spk_bf16_steps(const SpkLaunch& L, int tt) {
    switch (tt) {
        case 6: return launch_conv_spk_steps<bf16_t, 6>(L);
        case 4: return launch_conv_spk_steps<bf16_t, 4>(L);
        case 3: return launch_conv_spk_steps<bf16_t, 3>(L);
        case 2: return launch_conv_spk_steps<bf16_t, 2>(L);
        default: return launch_conv_spk_steps<bf16_t, 1>(L);
    }
}
}  // namespace snnf
