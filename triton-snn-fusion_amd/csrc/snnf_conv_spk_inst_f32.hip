// conv_spk_kernel, fp32 tensors as two bf16 terms.
#include "snnf_conv_spk_kernel.h"

namespace snnf {
int launch_conv_spk_f32(const SpkLaunch& L, int tt) {
    if (tt == 3) return launch_conv_spk_split<3>(L);
    return tt == 4 ? launch_conv_spk_split<4>(L) : (tt == 2 ? launch_conv_spk_split<2>(L) : launch_conv_spk_split<1>(L));
}
}  // namespace snnf
