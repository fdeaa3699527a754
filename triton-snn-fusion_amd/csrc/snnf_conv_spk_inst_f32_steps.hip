// Instantiates the blocked-layout conv+LIF kernel for fp32 tensors (two bf16 terms) and dense frames, one per timestep.
#include "snnf_conv_spk_kernel.h"

namespace snnf {
int launch_conv_spk_f32_steps(const SpkLaunch& L, int tt) {
    switch (tt) {
        case 4: return launch_conv_spk_steps<float, 4>(L);
        case 3: return launch_conv_spk_steps<float, 3>(L);
        case 2: return launch_conv_spk_steps<float, 2>(L);
        default: return launch_conv_spk_steps<float, 1>(L);
    }
}
}  // namespace snnf
