// 1x1 convolutions without a neuron on dense 16-bit tensors, any stride (snnf_conv_columns.hip): geometry and launcher.
#pragma once

#include "snnf_conv_common.h"

namespace snnf {

struct ColumnsGeom {
    int Cin, Cout, plane, W, P, Wo, sh, sw;   // plane: input pixels of an image; P: output pixels
    int columns, tiles;                       // output pixels of a timestep's images, and tiles of 32 of them
    int groups, pairs;                        // channel groups of 8, and pairs of them (packed weight fragments of 32 channels)
    int oc_tiles, items;
    int64_t out_step_stride;                  // elements
    int64_t frag_stride;                      // 16-bit elements between 32-channel fragments of the packed weight
    FastDiv d_oc_tiles, d_tiles, d_P, d_Wo;
};

struct ColumnsLaunch {
    StepPtrs xs;
    int T;
    ColumnsGeom g;
    const uint16_t* wpacked;
    const float* bias;
    void* out;
    hipStream_t stream;
};

// Whether the kernel takes a 1x1 layer without padding, residual and neuron, and is the faster one there.
bool takes_columns(int T, int N, int Cin, int H, int W, int Cout, int sh, int sw);
int launch_conv_columns(ColumnsLaunch L, int N, int Cin, int H, int W, int Cout, int sh, int sw, const PackGeom& pg, bool f16);

}  // namespace snnf
