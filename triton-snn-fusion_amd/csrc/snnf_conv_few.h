// The kernel for convolutions of few output pixels on the internal layouts (snnf_conv_few.hip): its geometry and launcher.
#pragma once

#include "snnf_conv_spk_kernel.h"

namespace snnf {

struct FewGeom {
    int N, C8in, H, W, Cout, C8out, KH, KW, sh, sw, ph, pw, Ho, Wo, T;
    int Cin;
    int taps, kw_mul;            // tap / KW == (tap * kw_mul) >> 16
    int res_layout, out_layout;  // snnf_layout codes; res_layout < 0: no residual
    int pool;                    // 2x2 averages of the spikes leave, in C8
    int v16, v_in_place;         // the membrane holds the activation dtype; the initial one lies where the final one goes
    int64_t out_step_stride;     // bytes
    // planned
    int PI, PR, PC, RR, RC, region;          // pixels of a workgroup (rows x columns of PI images), their halo per image, halo items per channel group
    int patches_x, patches_img, px_log2, frags;
    int64_t patches;
    int C8e, Gs;                 // channel groups rounded up to pairs; those staged
    int oc_tiles, grid;
    int npairs, gph_log2, frag_bytes;        // packed weight: pairs of k-slots per chunk, log2 of the pairs per tap, bytes between 32-row fragments
    uint32_t weight_bytes;
    SpkDiv d_oc_tiles, d_patches_img, d_patches_x, d_ppx, d_PC, d_region, d_rrrc, d_RC, d_taps;
};

struct FewLaunch {
    StepPtrs xs, residuals;
    FewGeom g;
    const void* wpacked;
    const float* bias;
    const void* v_start;
    void* out;
    void* v_store;
    LifParams lif;
    size_t lds_bytes;
    hipStream_t stream;
};

// Plans a layer whose extents, layouts and options stand in `g`; false where the kernel does not take it.
bool plan_few(FewGeom& g, const PackGeom& pg, size_t& lds_bytes);
int launch_conv_few(const FewLaunch& L, bool f16, int in_layout);

}  // namespace snnf
