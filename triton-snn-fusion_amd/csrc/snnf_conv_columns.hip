// 1x1 convolution + bias without a neuron on dense 16-bit tensors (the projection shortcuts of residual networks): any stride, no padding, no residual.
//
// A wave owns 32 output pixels of a timestep (of any images: columns of the matrix product, so that no lane is idle but in a step's last tile) x up to 128 output channels.
// A lane's operand is eight channels of its pixel, which it loads itself (eight loads of one element, the half-wave's pixels side by side), up to four pairs of channel groups
// ahead: no halo in LDS, and one barrier, where the four waves of a workgroup share an item's K. What bounds a launch of a small batch is one trip to memory and the launch
// itself (5 to 8 us; the matrix kernel, which stages halo tiles, takes 13 to 34); larger ones the issue of the elementwise loads and stores.
#include <algorithm>
#include <type_traits>

#include "snnf_conv_columns.h"

namespace snnf {
namespace {

constexpr int kColWaves = 4;
constexpr int kColAhead = 4;       // pairs of channel groups in flight

typedef __bf16 col_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 col_f16x8 __attribute__((ext_vector_type(8)));
typedef float col_f32x16 __attribute__((ext_vector_type(16)));
typedef float col_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t col_u32x4 __attribute__((ext_vector_type(4)));

template <bool F16>
__device__ __forceinline__ col_f32x16 col_mfma(col_u32x4 a, col_u32x4 b, col_f32x16 c) {
    if constexpr (F16) return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(col_f16x8, a), __builtin_bit_cast(col_f16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(col_bf16x8, a), __builtin_bit_cast(col_bf16x8, b), c, 0, 0, 0);
}

// Entry i of the pointer table that is the kernel's first argument.
typedef const void* col_cvp;
__device__ __forceinline__ const uint16_t* col_step(int i) {
    typedef const __attribute__((address_space(4))) col_cvp* entry;
    return static_cast<const uint16_t*>(((entry)__builtin_amdgcn_kernarg_segment_ptr())[i]);
}

// NF: fragments of 32 channels of a wave. SHARE: the four waves of a workgroup have one item, a quarter of its K each.
template <typename XT, int NF, bool SHARE>
__global__ __launch_bounds__(kColWaves * 64, 2) void conv_columns_kernel(const StepPtrs xs, const ColumnsGeom g, const uint16_t* __restrict__ wpacked,
                                                                         const float* __restrict__ bias, XT* __restrict__ out) {
    constexpr bool F16 = dtype_of<XT>::value == SNNF_F16;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int lane = threadIdx.x & 63, half = lane >> 5;
    const int item = SHARE ? static_cast<int>(blockIdx.x) : static_cast<int>(blockIdx.x) * kColWaves + wave;   // the channel tiles of a column tile follow each other: they share its lines
    if (!SHARE && item >= g.items) return;
    const int tile_t = fast_div(item, g.d_oc_tiles);
    const int oc0 = (item - tile_t * g.oc_tiles) * (32 * NF);
    const int t = fast_div(tile_t, g.d_tiles);
    const int column = (tile_t - t * g.tiles) * 32 + (lane & 31);
    const bool live = column < g.columns;
    const int n = fast_div(live ? column : 0, g.d_P);
    const int pixel = (live ? column : 0) - n * g.P;
    const int oh = fast_div(pixel, g.d_Wo);
    const uint32_t x_at = static_cast<uint32_t>(n * g.Cin * g.plane + oh * g.sh * g.W + (pixel - oh * g.Wo) * g.sw);
    const uint32_t o_at = static_cast<uint32_t>((n * g.Cout + 4 * half) * g.P + pixel);
    const uint16_t* __restrict__ const src = col_step(t);
    const int last_f = (g.Cout - 1) >> 5;
    const uint16_t* __restrict__ w_at[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) w_at[f] = wpacked + static_cast<int64_t>(min((oc0 >> 5) + f, last_f)) * g.frag_stride;      // (channels beyond the last are never stored)

    // This wave's pairs of channel groups.
    const int per_wave = SHARE ? (g.pairs + kColWaves - 1) / kColWaves : g.pairs;
    const int q0 = SHARE ? wave * per_wave : 0;
    const int np = min(per_wave, g.pairs - q0);

    col_u32x4 w[kColAhead][NF];
    uint32_t x[kColAhead][8];
    // Pair q of channel groups: the lower half of the wave has group 2 q, the upper half the next one.
    auto load = [&](int q, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int f = 0; f < NF; ++f) w[s][f] = *reinterpret_cast<const col_u32x4*>(w_at[f] + static_cast<uint32_t>(q * (kFragBytes / 2) + lane * 8));
        uint32_t at = x_at + static_cast<uint32_t>(min(2 * q + half, g.groups - 1) * 8 * g.plane);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            x[s][j] = src[at];
            at += static_cast<uint32_t>(g.plane);
        }
    };
    col_f32x16 acc[NF];
    auto start = [&]() __attribute__((always_inline)) {      // from the bias (its zeros behind the last channel where K is shared, but for the first wave)
        const float* __restrict__ const from = bias + (SHARE && wave > 0 ? (last_f + 2) / 2 * 64 : oc0) + 4 * half;
        const int step = SHARE && wave > 0 ? 0 : 8;
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const Pack<float, 4> b = *reinterpret_cast<const Pack<float, 4>*>(from + (4 * f + k) * step);
#pragma unroll
                for (int c = 0; c < 4; ++c) acc[f][4 * k + c] = b.v[c];
            }
    };
    auto multiply = [&](int q, int s) __attribute__((always_inline)) {
        const bool there = 2 * q + half < g.groups;      // an odd number of groups: the upper half's last one is not there
        col_u32x4 b;
#pragma unroll
        for (int k = 0; k < 4; ++k) b[k] = there ? __builtin_amdgcn_perm(x[s][2 * k + 1], x[s][2 * k], 0x05040100u) : 0u;
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[f] = col_mfma<F16>(w[s][f], b, acc[f]);
    };
    if (np <= 0) {
        start();
    } else {
        int q = 0;
#pragma unroll
        for (int s = 0; s < kColAhead; ++s)
            if (s < np) load(q0 + s, s);
        start();
        for (; q + 2 * kColAhead <= np; q += kColAhead) {
#pragma unroll
            for (int s = 0; s < kColAhead; ++s) {
                multiply(q0 + q + s, s);
                load(q0 + q + kColAhead + s, s);
            }
        }
#pragma unroll
        for (int s = 0; s < kColAhead; ++s) {
            if (q + s < np) multiply(q0 + q + s, s);
            if (q + kColAhead + s < np) load(q0 + q + kColAhead + s, s);
        }
#pragma unroll
        for (int s = 0; s < kColAhead; ++s)
            if (q + kColAhead + s < np) multiply(q0 + q + kColAhead + s, s);
    }

    // Accumulator register r of fragment f: channel 32 f + 8 (r / 4) + 4 half + r % 4. Four channels at a time, their places worked out where they stand.
    auto store = [&](int f, int k, const col_f32x4& sum) __attribute__((always_inline)) {
        int oc = oc0 + 32 * f + 8 * k;
        asm volatile("" : "+s"(oc));
        if (!live) return;
        XT* const to = out + static_cast<int64_t>(t) * g.out_step_stride + static_cast<int64_t>(oc) * g.P;
        const int left = g.Cout - oc - 4 * half;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (c < left) (to + c * g.P)[o_at] = from_float<XT>(sum[c]);
    };
    if constexpr (SHARE) {
        // [wave][fragment][quad][lane] sums; wave w finishes quad w of every fragment, adding the four parts in the order of K.
        __shared__ __align__(16) float parts[kColWaves * NF * 4 * 64 * 4];
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                *reinterpret_cast<col_f32x4*>(parts + (((wave * NF + f) * 4 + k) * 64 + lane) * 4) = col_f32x4{acc[f][4 * k], acc[f][4 * k + 1], acc[f][4 * k + 2], acc[f][4 * k + 3]};
        __syncthreads();
#pragma unroll
        for (int e = 0; e < NF; ++e) {      // quads wave, wave + 4, ... of the 4 NF
            const int at = wave + e * kColWaves;
            col_f32x4 sum = *reinterpret_cast<const col_f32x4*>(parts + (at * 64 + lane) * 4);
#pragma unroll
            for (int p = 1; p < kColWaves; ++p) sum += *reinterpret_cast<const col_f32x4*>(parts + ((p * NF * 4 + at) * 64 + lane) * 4);
            store(at >> 2, at & 3, sum);
        }
    } else {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int k = 0; k < 4; ++k) store(f, k, col_f32x4{acc[f][4 * k], acc[f][4 * k + 1], acc[f][4 * k + 2], acc[f][4 * k + 3]});
    }
}

}  // namespace

// us, matrix kernel / here, T = 4 and bf16 unless said. Shortcuts of ResNet-18: 64 -> 128 at 56^2 stride 2, one image 13.1 / 5.0, 4 images 13.1 / 7.2, 16 17.8 / 17.9, 64 65 / 60, 128 -> 256 at 28^2
// 15.8 / 5.2, 16.1 / 6.4, 17.9 / 14.8, 36.2 / 39.1, 256 -> 512 at 14^2 33 / 5.9, 34 / 7.2, 27.2 / 12.8, 37.7 / 31.9; 72 -> 200 at 21 x 17, T = 8 52 / 6.6, 24 -> 40 at 45^2 stride 3 x 64
// 24.4 / 8.8, 32 -> 64 at 112^2 stride 2 x 32 61 / 35, 256 -> 256 at 14^2 stride 1 x 16 17.5 / 15.3. It loses where many outputs have a long K, whose activations every tile of 128 channels reads
// again in single elements (256 -> 512 at 14^2 stride 2 x 80 39.6 / 38.1, x 120 43 / 54, at 28^2 x 32 31 / 57, 128 -> 256 at 28^2 x 256 135 / 151), and of stride 1, which the matrix
// kernel reads in pairs of pixels, by its outputs alone (64 -> 128 at 56^2 x 4, 6 M outputs, 16.2 / 16.0, x 8 18.0 / 25.9, 128 -> 128 at 28^2 x 16 19.3 / 18.2, x 32 22.1 / 31.3).
bool takes_columns(int T, int N, int Cin, int H, int W, int Cout, int sh, int sw) {
    if (Cin % 8 != 0) return false;
    const int64_t P = static_cast<int64_t>((H - 1) / sh + 1) * ((W - 1) / sw + 1), outputs = T * N * P * Cout;
    if (outputs > (1LL << 23) && !((sh > 1 || sw > 1) && Cin <= 64)) return false;
    return static_cast<int64_t>(N) * Cin * H * W < (1LL << 30) && outputs < (1LL << 30);      // (32-bit offsets)
}

int launch_conv_columns(ColumnsLaunch L, int N, int Cin, int H, int W, int Cout, int sh, int sw, const PackGeom& pg, bool f16) {
    ColumnsGeom& g = L.g;
    g.Cin = Cin; g.Cout = Cout; g.plane = H * W; g.W = W; g.sh = sh; g.sw = sw;
    g.Wo = (W - 1) / sw + 1;
    g.P = ((H - 1) / sh + 1) * g.Wo;
    g.columns = N * g.P;
    g.groups = Cin / 8;
    g.pairs = (g.groups + 1) / 2;
    g.frag_stride = static_cast<int64_t>(pg.nchunks) * pg.npairs * (kFragBytes / 2);
    g.tiles = (g.columns + 31) / 32;
    const int nf = Cout > 64 ? 4 : (Cout > 32 ? 2 : 1);
    g.oc_tiles = (Cout + 32 * nf - 1) / (32 * nf);
    g.items = L.T * g.tiles * g.oc_tiles;
    g.d_oc_tiles = make_fast_div(g.oc_tiles);
    g.d_tiles = make_fast_div(g.tiles);
    g.d_P = make_fast_div(g.P);
    g.d_Wo = make_fast_div(g.Wo);
    // Four waves on an item are faster at any number of items: the stores of a wave are a quarter, too (64 -> 128 at 56^2 stride 2, one image 13.3 -> 5.0 us, 64 images 68 -> 61).
    const bool share = g.pairs >= kColWaves;
    const dim3 grid(share ? g.items : (g.items + kColWaves - 1) / kColWaves);
    auto run = [&](auto* xt, auto nf_tag) -> int {
        using XT = std::remove_pointer_t<decltype(xt)>;
        constexpr int NF = decltype(nf_tag)::value;
        if (share) conv_columns_kernel<XT, NF, true><<<grid, kColWaves * 64, 0, L.stream>>>(L.xs, L.g, L.wpacked, L.bias, static_cast<XT*>(L.out));
        else conv_columns_kernel<XT, NF, false><<<grid, kColWaves * 64, 0, L.stream>>>(L.xs, L.g, L.wpacked, L.bias, static_cast<XT*>(L.out));
        return check_launch("snnf_conv_bias");
    };
    auto form = [&](auto* xt) -> int {
        if (nf == 4) return run(xt, std::integral_constant<int, 4>{});
        if (nf == 2) return run(xt, std::integral_constant<int, 2>{});
        return run(xt, std::integral_constant<int, 1>{});
    };
    return f16 ? form(static_cast<f16_t*>(nullptr)) : form(static_cast<bf16_t*>(nullptr));
}

}  // namespace snnf
