// Host side of the convolution + LIF operator on the internal activation layouts (channel-blocked C8, bit-packed BITS):
// argument validation, patch planning and launch of conv_spk_kernel.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>

#include "snnf_conv_few.h"
#include "snnf_conv_spk_kernel.h"

namespace snnf {
namespace {

constexpr int kWaveLds = (static_cast<int>(kMaxLds) - static_cast<int>(kSpkHeaderBytes)) / kSpkWaves / 16 * 16;   // private staging bytes of a wave

struct SpkPlan {
    int PR, PC, PI, RR, RC, region, G, patches_x, patches_y, img_groups;
    double score;
};

// Patch of a wave (PR x PC output pixels of one image, or PI whole planes when a plane has at most 32 pixels) and the
// channel groups per LDS stage G: the patch with the most useful matrix lanes and the smallest halo whose stage fits the
// wave's LDS region and its staging slots; the largest such G (fewer, longer stages).
bool plan_spk(const SpkGeom& g0, int tt, SpkPlan& best, int only_pc = 0, int only_g = 0, bool even = false) {
    best.score = -1.0;
    const int cus = compute_units();
    for (int pc = 1; pc <= 32 && pc <= g0.Wo; ++pc) {
        if (only_pc > 0 && pc != only_pc) continue;
        const int pr = std::min(32 / pc, g0.Ho);
        if (even && ((pc & 1) || (pr & 1))) continue;   // 2x2 windows of the output must lie inside a patch
        const bool whole = pr == g0.Ho && pc == g0.Wo;
        int pi = whole ? std::max(1, std::min(g0.N, 32 / (pr * pc))) : 1;
        // Whole planes of several images per patch: half as many images (idle matrix lanes) when the layer would otherwise have
        // fewer tiles than half the compute units; a tile's K is shared by the eight waves of a workgroup at that size, so tiles
        // are workgroups (512 -> 512 on 2 x 2 planes at batch 64: 64 workgroups of 8 images 24.1 us, 128 of 4 images 21.3 us,
        // 256 of 2 images 22.6 us, single images 34.7 us).
        const int oc_tiles = g0.narrow ? (g0.Cout + 31) / 32 : (g0.Cout + 63) / 64;
        if (pi > 1 && ((g0.N + pi - 1) / pi) * oc_tiles * 2 < cus) pi >>= 1;
        const int rr = (pr - 1) * g0.sh + g0.KH;
        const int pair = g0.in_layout == kSpkSteps ? 2 : 1;    // items that a lane stages at a time
        const int rc = ((pc - 1) * g0.sw + g0.KW + pair - 1) / pair * pair;
        if (rr > 255 || rc > 255) continue;
        // Where the halos of so many planes don't fit (5x5 on 2x2 planes, strided 3x3 onto 2x2 and 4x4) half as many, and again, before a part
        // of one plane: 512 -> 512 stride 2 from 4x4 x 155 in tiles of 2 x 1 pixels 170 us, of four planes 48, 256 -> 512, 5x5 on 2x2 x 122,
        // T = 8 252 / 55. Up to 256 pixels times tiles of channels parts are faster, as more workgroups (384 -> 64, 5x5 stride 2 from 4x4 x 15
        // 21.0 / 24.1; the quotient passes 1 there over 770 layers).
        const bool fewer = static_cast<int64_t>(g0.N) * pr * pc * oc_tiles > cus;
        int region, G = 0;
        for (;; pi >>= 1) {
            region = pi * rr * rc;
            if (g0.tap_pairs) {
                if (region <= 64 * kSpkSlots && tt * (region + pair) * 16 <= kWaveLds) G = 1;
            } else {
                for (int cand = g0.gpc; cand >= 2; cand >>= 1) {
                    if (only_g > 0 && cand > only_g) continue;
                    if (cand * region <= 64 * kSpkSlots && tt * (cand * region + pair) * 16 <= kWaveLds) {   // + the dummy items of a timestep
                        G = cand;
                        break;
                    }
                }
            }
            if (G > 0 || pi == 1 || !fewer) break;
        }
        if (G == 0) continue;
        const int patches_x = (g0.Wo + pc - 1) / pc;
        const int patches_y = (g0.Ho + pr - 1) / pr;
        const int img_groups = (g0.N + pi - 1) / pi;
        const double lanes = static_cast<double>(img_groups) * patches_x * patches_y * 32.0;
        const double eff = static_cast<double>(g0.N) * g0.Ho * g0.Wo / lanes;
        const double halo = static_cast<double>(region) / (static_cast<double>(pi) * pr * pc);
        // Wide patches store longer runs of a row; stages of 4 slots move in one batch.
        double score = eff / (1.0 + 0.08 * (halo - 1.0)) * (1.0 + 0.004 * std::min(pc, 16));
        if (G * region > 256) score *= 0.97;
        // A frame whose spikes leave as dense tensors is bound by its stores, 2-byte elements side by side along a row: what a pixel costs goes with the 64-byte
        // lines that a patch row touches (of row starts anywhere), and runs that are no multiple of 32 bytes share more of them. us in patches of
        // 8, 14, 16, 28 and 32 columns: 3 -> 64 7x7 stride 2 at 224^2 x 16 62.6, 56.8, 48.5, 51.8, 49.6, at 112^2 x 28 32.1, 32.6, 27.8, 25.1, 24.7, 3x3 at
        // 32^2 x 64 21.4, 22.8, 15.3, 18.1, 14.2, 3 -> 100 at 33^2 x 9 11.2, 9.5, 9.4, 10.8, 10.9.
        const bool dense_frame = g0.in_layout == SNNF_LAYOUT_NCHW && g0.out_layout == SNNF_LAYOUT_NCHW;
        if (dense_frame) score = eff / ((0.85 + 4.8 * (1.0 + (pc - 1) / 32.0) / pc) * (pc % 16 == 0 ? 1.0 : 1.12));
        // Waves own whole tiles: a launch of a little more than one round of waves takes as long as one of two. 88 -> 176 channels at
        // 43^2 x 5 is 1980 tiles of 4 x 8 pixels (31 us) or 2205 of 4 x 7 (53 us) on 2048 waves. Among patches of several rounds the fewer
        // tiles win (256 -> 256 at 14^2 x 128: 3584 of 2 x 14 99 us, 4096 of 4 x 8 103 us).
        const int64_t tiles = static_cast<int64_t>(img_groups) * patches_x * patches_y * oc_tiles, slots = static_cast<int64_t>(cus) * kSpkWaves;
        if (tiles > slots && !dense_frame) score *= 0.6;
        if (score > best.score) best = SpkPlan{pr, pc, pi, rr, rc, region, G, patches_x, patches_y, img_groups, score};
    }
    return best.score > 0.0;
}

// Measured choices for particular layers, registered by the host program (snnf_conv_blocked_tune): patch columns, channel
// groups per stage and waves sharing a tile's K, by layer shape. A choice the kernel cannot run is ignored.
using TunedKey = std::array<int, 13>;
struct TunedPlan { int patch_cols, stage_groups, k_waves; };
std::mutex tuned_mutex;
std::map<TunedKey, TunedPlan>& tuned_plans() {
    static std::map<TunedKey, TunedPlan> plans;
    return plans;
}

size_t c8_step_bytes(int N, int Cin, int H, int W) { return static_cast<size_t>(N) * ((Cin + 7) / 8) * H * W * 16; }

// The workspace of a call on the blocked route: the C8 steps; of fp32 tensors the steps of their low terms and the flags behind them; the
// fp32 membrane that a call of several windows with a 16-bit one passes from window to window (rounded once, at the end).
struct RouteSpace {
    size_t step, lo, flags, flag_stride, carry, total; // bytes; offsets of the low terms, the flags and the membrane
};
RouteSpace route_space(int T, int N, int Cin, int H, int W, bool split, int64_t carried) {
    RouteSpace r = {};
    r.step = c8_step_bytes(N, Cin, H, W);
    r.total = r.step * T;
    if (split) {
        r.lo = r.total;
        r.flags = 2 * r.total;
        r.flag_stride = (r.step / 16 + 255) / 256 * 4;   // one byte per 64 items, in whole dwords
        r.total = r.flags + r.flag_stride * T;
    }
    r.carry = r.total;                                   // (a multiple of 16: no call has both)
    r.total += static_cast<size_t>(carried) * 4;
    return r;
}

// Timesteps in windows of three: no more windows than of four, and a matrix step then multiplies nothing for steps beyond T (3, 5, 6 and 9 timesteps; the rest would take more windows). us, windows of
// four / three, T = 3: 64 -> 64 at 56^2 x 16 on bits 20.6 / 15.8, x 40 35.6 / 26.1, 128 -> 128 at 28^2 x 16 with a residual 19.0 / 15.1, dense 30.9 / 27.3, 512 -> 512 at 7^2 x 7 12.8 / 10.7; T = 6
// 36.1 / 32.9, 69.3 / 61.8, 36.6 / 30.4, 53.3 / 47.6, 23.4 / 19.5; fp32 104 -> 328 at 16^2 x 23, T = 5 78.7 / 66.7. 121 layers: 1.13 in the mean, none slower; the same bits.
bool threes(int T) { return T > 2 && (T + 2) / 3 == (T + 3) / 4; }

// Whether a layer on dense tensors is brought into C8 and run on the blocked kernel (two launches) or stays on the dense kernels. Measured on
// layers of 1 to 64 images, 1 to 512 channels, 1x1 to 7x7, one to eight timesteps (us, dense / here; bf16 and T = 4 unless said):
// * Channel counts that are no multiple of 8 only have the four-wave kernels on dense tensors, which assemble every channel group from
//   scalar loads: they move (126 -> 200 at 12 x 54 stride 2, T = 2 93 / 18, 29 -> 72 at 70^2, 7x7 stride 2 316 / 23, 61 -> 32 1x1 at 39 x 20, T = 3
//   29 / 16), but for large 1x1 layers, which are memory traffic (421 -> 288 at 100^2, T = 8 356 / 416).
// * The matrix kernel's masked variant (planes or channels its tiles do not divide) goes in windows of two timesteps and pays a pass over
//   the weights per window: 600 layers gain a factor of 2 (72 -> 104 at 27 x 35, T = 6, with a residual 59 / 39, 512 -> 512 at 7^2 x 16 55 / 31,
//   16 -> 96 at 25^2 x 8 with a residual 25 / 23, 24 -> 16 at 26^2, 5x5, T = 5 64 / 31). Of one or two timesteps, one window there as well, 1x1
//   layers of any size lose with the copy (256 -> 128 at 97^2 x 16, T = 1 115 / 146, 128 -> 256 stride 2 at 28^2 x 52, T = 1 18 / 24) and so do large strided
//   ones (64 -> 128 at 40^2 x 17, T = 2 16 / 19); 1x1 layers of a stride copy four pixels for one (168 -> 349 at 24 x 75 x 14, T = 6 104 / 123).
// * The pointwise kernel's straight-line variant takes planes of whole tiles of 64 pixels: 24 -> 96 at 56^2 x 32 31 / 73, 128 -> 256 89 / 224.
//   Its general variant is several times slower and loses over 260 layers to a factor of 1.8 (128 -> 64 at 7^2, T = 8 60 / 16, 64 -> 256 at
//   51^2 x 16 with a residual 216 / 127, 128 -> 256 at 28^2 x 32, T = 2 56 / 50).
// * Whole tiles of the matrix kernel take the time of their rounds, full or not, and of their windows of four steps; this kernel's time is
//   nearly proportional to the outputs. So `tile_use` decides (see dense_family), weighed by the products per output, in which this kernel is
//   the better one. The quotient of the two times falls with it from 2 to 0.75 and passes 1 at the lines below. It moves 64 -> 64 at 24^2 x 4 30 / 12, x 38, T = 6 70 / 45, at
//   40^2 x 20 (tiles of four columns) 43 / 33, T = 8 121 / 68, at 56^2 x 21, T = 6 132 / 110, 128 -> 256 stride 2 at 28^2 x 5, T = 8 49 / 40, 1x1 stride 2 x 2
//   31 / 20; 64 -> 64 at 56^2 x 16 34 / 42, 128 -> 128 at 28^2 x 32 52 / 55, 64 -> 128 stride 2 at 56^2 x 16 28 / 37, 1x1 18 / 26, 128 -> 256 stride 2
//   at 28^2 x 16 28 / 34 stay. Where a step's copy takes up to 5 MB, so that the L2 caches hold all of it for the kernel, the line lies higher for layers that fill this kernel's
//   waves (see `fills_waves`); beyond 4 M elements a step the quotient is 0.97. Inputs that the caches don't hold between the copy and the kernel move the lines (64 -> 64 at 56^2 x 88, T = 5
//   with a residual 366 / 437, 128 -> 256 stride 2 at 28^2 x 164, T = 7 395 / 554). Deep layers of few outputs always move (256 -> 256 at 14^2 x 4 29 / 18, 512 -> 512 at 4^2 x 16 37 / 21). Over 22300 layers of
//   whole tiles, planes of four pixels, few pixels and deep layers among them, the rule is 1 % slower than the better kernel in the mean, the dense kernels
//   alone 54 % (256 -> 512 at 2^2 x 40 24 / 14, 64 -> 64 at 16^2 x 2 30 / 11, 256 -> 256 at 14^2 x 16 35 / 31, with a residual 37 / 32).
// * fp32 tensors (two bf16 terms each) run here at two and a half times the speed of the dense kernels over 1500 layers without low terms, and at
//   1.85 times where every input has one: 64 -> 64 at 32^2 x 8 35 / 20, at 56^2 x 16 100 / 73, 512 -> 512 at 7^2 x 4 with a residual 125 / 29, 41 -> 72
//   at 8 x 14 x 15 191 / 20, 122 -> 111 at 15^2, 5x5, T = 5 1068 / 36, 3 -> 64 at 32^2 x 64 34 / 31, 128 -> 256 1x1 at 28^2 x 8 135 / 27. 1x1 layers
//   stay where the copy and the elementwise outputs are their time: on the pointwise kernel those with few products per output and many outputs
//   (64 -> 256 at 56^2 x 16, T = 1 with a residual 66 / 82, 64 -> 128 at 112^2 x 4 80 / 90, 32 -> 192 at 56^2 x 16 116 / 124; but 64 -> 128 at 28^2 x 8
//   79 / 25, 128 -> 256 at 56^2 x 16 281 / 192); on the matrix kernel, which takes up to four steps in one window, those of a stride, of
//   whose copy a quarter is read, unless that kernel would leave the chip idle or they have few outputs or several windows (without low
//   terms / with them everywhere: 96 -> 192 at 112^2 x 36, T = 2 0.54 / 0.34 of its speed, 64 -> 512 at 80^2 x 3 0.80 / 0.54, 48 -> 248 at 125^2 x 4, T = 2
//   0.80 / 0.65; 32 -> 192 at 56^2 1.90 / 1.55, 256 -> 512 at 24^2 x 5, T = 12 4.46 / 2.73), and others of one or two steps and many outputs (192 -> 256
//   at 28^2 x 12, T = 2 0.89 / 0.69; 192 -> 128 x 3 1.37 / 1.12).
// Without a neuron the lines are those of sums that leave as 16-bit values (512 -> 512 at 7^2 x 16 56 / 35).
// `weigh`: above zero a layer only moves where `fills_waves` says so, below only where the kernel reads the dense frames itself.
bool takes_blocked_route(int T, int N, int Cin, int H, int W, int x_dtype, int Cout, int KH, int KW, int stride_h, int stride_w, int pad_h, int pad_w,
                         int v_dtype, bool residual, bool neuron, DenseFamily& family, double& weigh) {
    weigh = 0.0;
    if (x_dtype != SNNF_BF16 && x_dtype != SNNF_F16 && x_dtype != SNNF_F32) return false;
    if ((v_dtype != SNNF_F32 && v_dtype != x_dtype) || T < 1 || T > SNNF_MAX_T_PER_LAUNCH || N < 1 || Cin < 1 || H < 1 || W < 1 || Cout < 1 || KH < 1 || KW < 1 ||
        stride_h < 1 || stride_w < 1 || pad_h < 0 || pad_w < 0 || H + 2 * pad_h < KH || W + 2 * pad_w < KW || 2 * pad_h > KH || 2 * pad_w > KW) return false;
    const bool one = KH == 1 && KW == 1, strided = stride_h > 1 || stride_w > 1;
    const bool pointwise = one && !strided && pad_h == 0 && pad_w == 0;
    const int64_t K = static_cast<int64_t>(Cin) * KH * KW, plane = static_cast<int64_t>(H) * W;
    const int64_t pixels = static_cast<int64_t>(N) * ((H + 2 * pad_h - KH) / stride_h + 1) * ((W + 2 * pad_w - KW) / stride_w + 1);
    const int64_t out = pixels * Cout, outs = T * out, inputs = static_cast<int64_t>(T) * N * Cin * plane;
    double tile_use;
    family = dense_family(T, N, Cin, H, W, x_dtype, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, tile_use);
    if (x_dtype == SNNF_F32) {
        if (one && family == DenseFamily::kMatrixWhole)
            return strided ? (T <= 2 ? tile_use <= 0.4 : T > 4 || outs <= (3 << 21)) : T > 2 || outs <= (3 << 20);
        if (one && strided && family == DenseFamily::kMatrixMasked) return T > 2 || outs <= (1 << 20);
        return !(family == DenseFamily::kPointwise && Cin <= 64 && Cout >= 96 && outs >= (1 << 22));
    }
    const bool deep = K >= 4608 || (K >= 2304 && out <= (1 << 19) && !residual);
    if (!neuron) {
        if (pointwise) return false;
        return family == DenseFamily::kMatrixMasked ? !(T > 4 && Cin < 56) && (T <= 2 ? K >= 1152 : K >= (residual ? 640 : 432)) : family == DenseFamily::kMatrixWhole && deep;
    }
    if (pointwise && Cin < 8) return false;   // a single channel group: next to no products
    switch (family) {
        case DenseFamily::kTInM:
        case DenseFamily::kTimeOuter: return !pointwise || static_cast<int64_t>(T) * N * (Cin + Cout) * plane <= (1 << 25);
        case DenseFamily::kPointwise: return plane % 64 != 0 || (Cout % 32 != 0 && outs <= (1 << 22));
        case DenseFamily::kMatrixMasked:
            // One or two timesteps of a 1x1 layer of stride 1 move where the kernel reads the frames itself: 410 drawn layers, 1.48 in the mean with frames from the caches, 1.35 from
            // memory, 7 and 13 lose more than a twentieth, the worst 0.88 and 0.83 (us, dense / here, 360 -> 24 at 13 x 48 x 17, T = 2
            // 26.2 / 8.1, 136 -> 16 at 68 x 11 x 20, T = 1 13.1 / 7.2, 144 -> 205 at 12 x 54 x 28, T = 1 28.7 / 20.6, 216 -> 88 at 52^2 x 28, T = 2 55.4 / 61.8; of five that
            // keep the copy 464 -> 164 at 34 x 33 x 9, T = 1 21.3 / 34.1).
            if (pointwise && T <= 2 && outs > (1 << 17)) weigh = -1.0;
            if (pointwise && T <= 2) return true;
            if (one) return T <= 2 ? outs <= (1 << 17) : !strided || inputs <= (1 << 24);
            return T > 2 || K >= 1152 || !strided || outs <= (3 << 19);
        case DenseFamily::kMatrixWhole:
            if (deep) return true;
            if (!one && !strided && Cin <= 8) return false;   // (a single channel group: as above)
            if (one) return tile_use * std::sqrt(576.0 / K) <= 0.45;
            // (In windows of three this kernel gains an eighth and the lines lie further up. us, dense / here, with the weighed use: T = 3 64 -> 64 at 56^2 x 9 (0.86) 30.0 / 25.7, x 28 (1.13) 57.0 / 48.7,
            // 32 -> 64 at 32^2 x 90 (1.18) 41.0 / 38.7, x 48 (1.5) 23.2 / 27.2; T = 5 64 -> 64 at 56^2 x 16 (0.96) 63.2 / 53.6, T = 6 (1.15) 63.4 / 58.9, with a residual 69.6 / 73.4; strided T = 3
            // 128 -> 256 at 28^2 x 5 (0.53) 21.1 / 16.0, x 90 (0.61) 91.4 / 96.3, x 48 (0.65) 65.0 / 54.6, x 28 (0.75) 34.4 / 36.3; T = 6 64 -> 128 at 56^2 x 28 (0.56) 94.0 / 78.3, x 48 (0.58) 137.9 / 142.9,
            // 128 -> 256 at 28^2 x 9 (0.72) 43.0 / 32.4, 64 -> 128 at 56^2 x 9 (1.21) 36.1 / 34.0.)
            const bool three = threes(T);
            if (strided) return tile_use * std::sqrt(std::sqrt(576.0 / K)) <= (T <= 4 ? (three ? 0.66 : 0.5) : (inputs < (1 << 24) ? (three ? 1.25 : 0.65) : (three ? 0.57 : 0.45)));
            const double weighed = tile_use * std::sqrt(576.0 / K);
            if (weighed <= (inputs >= (1 << 26) ? 0.7 : (T <= 4 ? (three ? 1.2 : 0.85) : (three ? 1.1 : 0.95)))) return true;
            if (inputs / T > (5 << 19) || weighed > 1.1) return false;
            weigh = weighed;
            return true;
    }
    return false;
}

bool valid_layout(int layout) { return layout == SNNF_LAYOUT_NCHW || layout == SNNF_LAYOUT_C8 || layout == SNNF_LAYOUT_BITS; }

// A projection shortcut whose sums join the main convolution's accumulators: a pointwise convolution (stride s, no padding)
// of a second bit-packed input with as many output channels and output pixels as the main one.
struct Shortcut {
    const void* const* xs;
    int Cin, H, W, stride_h, stride_w;
    const void* packed_weight;
};

// What a launch of the blocked kernel depends on, without its pointers.
struct BlockedCall {
    int T, N, Cin, H, W, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w;
    int x_layout, res_layout, out_layout;              // res_layout: -1 without a residual
    int64_t out_step_stride;
    bool shared, neuron, has_v_init, has_v_out, pool2;
    const Shortcut* shortcut;
    bool split;                                        // fp32 tensors as two bf16 terms
};

struct BlockedPlan {
    SpkGeom g = {};
    SpkPlan patch = {};
    PackGeom pg = {}, pg2 = {};                        // of the weight, and of the shortcut's
    int tt = 0, windows = 0, wk_log2 = 0, oc_tiles = 0, grid = 0;
    size_t lds_bytes = 0;
    bool tuned_patch = false, tuned_split = false;
    bool few = false;                                  // the kernel for few output pixels runs instead
    FewGeom few_g = {};
    size_t few_lds = 0;
};

// Everything that decides whether and how the kernel runs a call; nothing is enqueued. `window`: all timesteps in one window of so many (0: windows of up to four).
int plan_window(const char* who, const BlockedCall& c, BlockedPlan& p, int window, bool may_three = true) {
    const int T = c.T, N = c.N, Cin = c.Cin, H = c.H, W = c.W, Cout = c.Cout, KH = c.KH, KW = c.KW;
    const int stride_h = c.stride_h, stride_w = c.stride_w, pad_h = c.pad_h, pad_w = c.pad_w;
    const bool shared = c.shared, neuron = c.neuron, pool2 = c.pool2;
    const Shortcut* sc = c.shortcut;
    SpkGeom& g = p.g;
    g.N = N; g.Cin = Cin; g.H = H; g.W = W; g.Cout = Cout; g.KH = KH; g.KW = KW;
    g.sh = stride_h; g.sw = stride_w; g.ph = pad_h; g.pw = pad_w;
    g.Ho = (H + 2 * pad_h - KH) / stride_h + 1;
    g.Wo = (W + 2 * pad_w - KW) / stride_w + 1;
    g.C8in = (Cin + 7) / 8;
    g.C8out = (Cout + 7) / 8;
    const int64_t in_items = static_cast<int64_t>(N) * g.C8in * H * W;
    const int64_t out_elems = static_cast<int64_t>(N) * g.C8out * 8 * g.Ho * g.Wo;
    if (in_items >= (1LL << 27) || out_elems >= (1LL << 30) || static_cast<int64_t>(T) * N * g.C8out * g.Ho * g.Wo >= (1LL << 31))
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_shape: tensor too large for 32-bit offsets", who);
    if (c.out_layout == SNNF_LAYOUT_BITS && (c.out_step_stride < 0 || c.out_step_stride >= (1LL << 31) / T))
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_shape: bit-packed output beyond 2 GiB", who);
    const PackGeom& pg = p.pg = make_pack_geom(Cout, Cin, KH, KW, c.split);
    g.gpc = pg.CK / 8;
    g.npairs = pg.npairs;
    g.nocf = pg.nocf;
    g.tap_pairs = pg.CK == 8 ? 1 : 0;
    g.taps = KH * KW;
    g.frag_stride = static_cast<int64_t>(pg.nchunks) * pg.npairs * (kFragBytes / 2);
    g.w_lo_offset = static_cast<int64_t>(pg.nchunks_r) * pg.npairs * (kFragBytes / 2);   // part 1 of the weight (kSplitParts)
    g.narrow = c.split || window > 0 ? 1 : 0;
    g.T = T;
    g.shared_x = shared ? 1 : 0;
    g.in_layout = c.x_layout;
    g.res_layout = c.res_layout;
    g.out_layout = c.out_layout;
    g.analog_out = neuron ? 0 : 1;
    g.out_step_stride = c.out_step_stride;

    // Timesteps side by side: 4 (2 for T == 2, 1 for a single step or a shared frame, 3 where that takes no more windows), fewer when the halo does not fit.
    // Where four don't fit, three only do with few pixels a tile, and two it is (160 -> 40 7x7 stride 2 at 21^2 x 29, T = 6 in patches of 11 x 1 77 us, of 2 x 11 55).
    int& tt = p.tt;
    SpkPlan fours;
    const bool three = may_three && !shared && !pool2 && threes(T) && plan_spk(g, 4, fours);
    tt = window > 0 ? window : (shared || T == 1 ? 1 : (T == 2 ? 2 : (three ? 3 : 4)));
    TunedPlan tuned = {0, 0, 0};
    if (!c.split) {   // (measured on 16-bit activations)
        const TunedKey key = {T, N, Cin, H, W, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, shared ? 1 : 0};
        std::lock_guard<std::mutex> lock(tuned_mutex);
        const auto it = tuned_plans().find(key);
        if (it != tuned_plans().end()) tuned = it->second;
    }
    SpkPlan& pl = p.patch;
    if (pool2 && (!neuron || T != 4 || (g.Ho & 1) || (g.Wo & 1) || c.res_layout >= 0 || c.has_v_init || Cout % 8 != 0))
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_pool: needs four timesteps, a neuron from the zero membrane, no residual, an even %dx%d output plane and whole channel groups",
                    who, g.Ho, g.Wo);
    bool planned = (tuned.patch_cols > 0 || tuned.stage_groups > 0) && plan_spk(g, tt, pl, tuned.patch_cols, tuned.stage_groups, pool2);
    p.tuned_patch = planned;
    for (; !planned && tt >= 1; tt = tt == 3 ? 2 : tt >> 1) {
        planned = plan_spk(g, tt, pl, 0, 0, pool2);
        if (planned) break;
        if (pool2 || window > 0) break;   // the pooled store covers the four steps of one window
    }
    if (!planned)
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_shape: no patch of this layer fits a wave's LDS region (kernel %dx%d, stride %dx%d)",
                    who, KH, KW, stride_h, stride_w);
    if (!p.tuned_patch && !g.tap_pairs) {
        // Few tiles: stages of fewer channel groups where that lets more waves share a tile's K (128 -> 256 at 8^2, one image: stages
        // of 4 groups on 4 waves 13.4 us, of 2 groups on 8 waves 11.9 us; 64 -> 128 at 16^2 13.3 / 11.7).
        const int64_t tiles = static_cast<int64_t>(pl.img_groups) * pl.patches_x * pl.patches_y * (g.narrow ? (Cout + 31) / 32 : (Cout + 63) / 64);
        int share = 1;
        while (share < kSpkWaves && tiles * share * 2 <= static_cast<int64_t>(compute_units()) * kSpkWaves) share *= 2;
        while (pl.G > 2 && (g.C8in + pl.G - 1) / pl.G < share) pl.G >>= 1;
    }
    p.windows = shared ? 1 : (T + tt - 1) / tt;
    if (neuron && !shared && T > std::min(tt, 4) && !c.has_v_out)
        return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: v_out is required when the timesteps take %d windows of %d (it carries the membrane between them)",
                    who, p.windows, tt);
    g.PR = pl.PR; g.PC = pl.PC; g.PI = pl.PI; g.RR = pl.RR; g.RC = pl.RC; g.region = pl.region; g.G = pl.G;
    g.patches_x = pl.patches_x;
    g.patches_img = pl.patches_x * pl.patches_y;
    g.n_patches = pl.img_groups * g.patches_img;
    g.nstages = (g.C8in + g.G - 1) / g.G;
    g.IT = g.G * g.region;
    const int pair = g.in_layout == kSpkSteps ? 2 : 1;
    g.JT = (g.IT / pair + 63) / 64;
    g.lds_wave_bytes = std::max(tt * (g.IT + pair) * 16, 256);   // (a tile's bias passes through it)
    int& oc_tiles = p.oc_tiles;
    oc_tiles = g.narrow ? (Cout + 31) / 32 : (Cout + 63) / 64;
    g.n_items = g.n_patches * oc_tiles;
    // K is shared by as many waves of a workgroup (up to eight, whole stages each) as keep the layer's tiles in one round of waves:
    // 64 -> 64 at 56^2 x 12 is 1176 tiles, 20.2 us unsplit and 27.9 us when two waves share each (2352 of 2048 waves).
    const int cus = compute_units();
    int& wk_log2 = p.wk_log2;
    while (wk_log2 < 3 && static_cast<int64_t>(g.n_items) << (wk_log2 + 1) <= static_cast<int64_t>(cus) * kSpkWaves && g.nstages >= (2 << wk_log2)) ++wk_log2;
    if (tuned.k_waves > 0) {
        int want = 0;
        while ((1 << want) < tuned.k_waves) ++want;
        if (g.nstages >= (1 << want)) {
            wk_log2 = want;
            p.tuned_split = true;
        }
    }
    g.wk_log2 = wk_log2;
    // Tiles of 32 channels where even those fit one round of waves: 256 -> 256 at 14^2 x 4 (112 tiles of 64 channels on eight waves each)
    // 13.9 -> 10.0 us, 512 -> 512 at 7^2 x 8 19.8 -> 13.9, at 4^2 x 32 22.2 -> 17.6. At twice the tiles they would make a second round.
    // The same where a single stage leaves nothing to share (16 -> 64 at 14^2 x 17 10.2 -> 7.6, 16 -> 96 at 8^2 x 3 8.8 -> 6.6, 16 -> 64 at 28^2 x 6,
    // 5x5, T = 6 21.2 -> 14.8; frames: 3 -> 64 at 32^2 x 8 8.5 -> 6.5, 7x7 at 224^2 10.0 -> 8.3, T = 8 16.6 -> 11.3); of one timestep
    // two workgroups share a unit (3 -> 64 at 32^2 x 64, T = 8 15.6 -> 13.7, 16 -> 64 at 40^2 x 30 10.1 -> 8.7). Up to 32 channels always: half of a tile of 64 would be empty (90 layers, factors of 1.13 to 1.5: 64 -> 8 at 28^2 x 73,
    // T = 8 37.5 -> 27.7, 128 -> 32 at 32^2 x 18 22.2 -> 16.6, 128 -> 24 at 14^2 10.7 -> 8.2).
    const bool frame = c.x_layout == SNNF_LAYOUT_NCHW;
    if (!c.split && (tt == 4 || !pool2 || frame) && !p.tuned_split && (wk_log2 > 0 ? !frame : frame || (!pool2 && sc == nullptr)) &&
        ((Cout <= 32 && wk_log2 == 0) || static_cast<int64_t>(g.n_patches) * ((Cout + 31) / 32) << wk_log2 <= static_cast<int64_t>(cus) * kSpkWaves * (tt == 1 && wk_log2 == 0 ? 2 : 1))) {
        g.narrow = 1;
        oc_tiles = (Cout + 31) / 32;
        g.n_items = g.n_patches * oc_tiles;
    }
    const int tiles_per_block = kSpkWaves >> wk_log2;
    // Workgroups that are resident together: one per compute unit, or two where a wave needs at most a quarter of a SIMD's
    // registers (one timestep's accumulators) and two staging areas fit the LDS. The tiles are dealt evenly over as many
    // rounds as that takes.
    if (wk_log2 > 0) g.lds_wave_bytes = std::max(g.lds_wave_bytes, kSpkPartialBytes);
    p.lds_bytes = kSpkHeaderBytes + static_cast<size_t>(kSpkWaves) * g.lds_wave_bytes;
    const int resident = cus * ((tt == 1 && 2 * (p.lds_bytes + 1024) <= kMaxLds) ? 2 : 1);
    const int blocks = (g.n_items + tiles_per_block - 1) / tiles_per_block;
    g.iters = (blocks + resident - 1) / resident;
    int& grid = p.grid;
    grid = (blocks + g.iters - 1) / g.iters;
    // Workgroups full of waves that leave a quarter of the compute units idle in every round, or half of them in the only one: a workgroup
    // on every unit, some of its waves idle in the last round (128 -> 128 at 28^2 x 40, 140 workgroups 55.5 us, 256 workgroups 45.1; 64 -> 64
    // at 24^2, one image, 18 and 36 workgroups 8.5 / 7.5). Fuller rounds stay even: 256 -> 256 at 14^2 x 128, 224 workgroups 100 us, 256 105.
    // Narrow tiles of one wave: two tiles of a patch side by side, which read the same activations.
    const int spread = g.narrow && !c.split && wk_log2 == 0 ? g.n_patches * ((Cout + 63) / 64) : g.n_items;
    // The same where the last of three or more rounds is at most half full (of one timestep, whose workgroups run two to a unit, seven tenths of any round): every
    // unit, and a few waves with a tile more, against fewer units with full rounds. us, full rounds / every unit, by the rounds that all units would take, 64 -> 64 at 56^2: 2.49 (52 images)
    // 45.2 / 41.7, 3.45 56.8 / 53.8, 5.36 83.8 / 81.2, 6.13 (128) 111 / 105; 128 -> 128 at 28^2: 2.30 72.7 / 70.3, 3.50 98.2 / 94.8; 64 -> 128 stride 2 3.06 81.1 / 76.3; stem at 224^2: 1.53
    // (16 images) 32.5 / 31.7, 2.30 42.8 / 38.9, 3.06 55.3 / 51.6, 12.25 175 / 171. Fuller rounds gain nothing (64 -> 64 at 4.98 74.2 / 75.0, 6.89 102.2 / 102.1, stem 6.89 94.1 / 95.4), and of two
    // rounds the second one takes as long for a single tile of a SIMD as for two (256 -> 256 at 14^2, 1.53 90.3 / 95.1, 64 -> 64 at 56^2 x 32 30.8 / 32.1).
    const double rounds = static_cast<double>(g.n_items) / (static_cast<double>(resident) * tiles_per_block), over = rounds - std::floor(rounds);
    const bool part = resident > cus ? rounds > 1.0 && over <= 0.7 : rounds > 2.0 && over <= 0.5;
    if (g.iters > 1 ? grid * 4 < resident * 3 || part : grid * 2 <= cus) grid = std::min(spread, g.iters > 1 ? resident : cus);
    g.grid = grid;
    g.d_ppx = make_spk_div(g.PR * g.PC);
    g.d_PC = make_spk_div(g.PC);
    g.d_region = make_spk_div(g.region);
    g.d_rrrc = make_spk_div(g.RR * g.RC);
    g.d_RC = make_spk_div(g.RC);
    g.d_n_patches = make_spk_div(g.n_patches);
    g.d_patches_img = make_spk_div(g.patches_img);
    g.d_patches_x = make_spk_div(g.patches_x);
    const int hg = g.tap_pairs ? 1 : g.G / 2;
    const int nst = g.tap_pairs ? g.npairs : g.taps * hg;
    g.kw_mul = (KW & (KW - 1)) == 0 ? 65536 / KW : 65536 / KW + 1;
    for (int tap = 0; tap < KH * KW; ++tap)
        if (((tap * g.kw_mul) >> 16) != tap / KW)
            return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_kernel: kernel %dx%d too large", who, KH, KW);
    g.gpc_log2 = 0;
    while ((1 << g.gpc_log2) < g.gpc) ++g.gpc_log2;
    g.hg_log2 = 0;
    while ((1 << g.hg_log2) < hg) ++g.hg_log2;
    g.pair_tap_stride = g.tap_pairs ? 1 : g.gpc / 2;
    if (nst > kSpkMaxSteps)
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_kernel: %d matrix steps per stage exceed %d (kernel %dx%d)", who, nst, kSpkMaxSteps, KH, KW);
    if (sc != nullptr) {
        PackGeom& pg2 = p.pg2;
        pg2 = make_pack_geom(Cout, sc->Cin, 1, 1, false);
        const int gpc2 = pg2.CK / 8;
        if (tt < 3 || g.tap_pairs || gpc2 % g.G != 0 || nst + 4 + hg + 4 > kSpkMaxSteps + 4)
            return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_shortcut: this layer's plan (window %d, %d channel groups per stage, %d steps) has no room for a shortcut",
                        who, tt, g.G, nst);
        g.sc_C8 = sc->Cin / 8;
        g.sc_stages = (g.sc_C8 + g.G - 1) / g.G;
        g.sc_H = sc->H; g.sc_W = sc->W; g.sc_sh = sc->stride_h; g.sc_sw = sc->stride_w;
        g.sc_gpc_log2 = 0;
        while ((1 << g.sc_gpc_log2) < gpc2) ++g.sc_gpc_log2;
        g.sc_npairs = pg2.npairs;
        g.sc_frag_stride = static_cast<int64_t>(pg2.nchunks) * pg2.npairs * (kFragBytes / 2);
    }
    // Layers whose K several waves share, in few tiles: the kernel for few pixels. One that could be pooled takes it with and without its pool or not at
    // all, so that the pooled launch has the sums of the unpooled one.
    if (neuron && !c.split && !shared && sc == nullptr && c.x_layout != kSpkSteps && wk_log2 > 0 && !p.tuned_patch && !p.tuned_split && (c.out_layout != SNNF_LAYOUT_C8 || pool2) && c.res_layout != SNNF_LAYOUT_C8) {
        FewGeom& f = p.few_g;
        f.N = N; f.Cin = Cin; f.C8in = g.C8in; f.H = H; f.W = W; f.Cout = Cout; f.C8out = g.C8out; f.KH = KH; f.KW = KW;
        f.sh = stride_h; f.sw = stride_w; f.ph = pad_h; f.pw = pad_w; f.Ho = g.Ho; f.Wo = g.Wo; f.T = T;
        f.taps = g.taps; f.kw_mul = g.kw_mul;
        f.res_layout = c.res_layout; f.out_layout = c.out_layout; f.pool = pool2 ? 1 : 0;
        const FewGeom blank = f;
        const bool poolable = T == 4 && (g.Ho & 1) == 0 && (g.Wo & 1) == 0 && Cout % 8 == 0 && c.res_layout < 0 && c.out_layout != SNNF_LAYOUT_NCHW;
        p.few = plan_few(f, pg, p.few_lds);
        if (p.few && poolable) {
            FewGeom other = blank;
            size_t other_lds;
            other.pool = pool2 ? 0 : 1;
            p.few = plan_few(other, pg, other_lds);
        }
    }
    return SNNF_OK;
}

// Five and six timesteps take one window where two windows of three would be short: narrow tiles whose K several waves share, with up to 16 matrix steps to each.
// Such a launch lasts as long as one tile's chain of set-up, stages, exchange of sums and epilogue, which it then has once instead of twice. us, two windows / one, T = 6:
// 64 -> 64 at 24^2 x 8 11.9 / 10.1 (bits), 17.2 / 15.9 (dense), 72 -> 240 at 10^2 x 9 19.2 / 17.2, T = 5: 32 -> 296 at 15^2 x 6 with a residual 17.3 / 15.7, 24 -> 27 at 10 x 28 x 11 15.6 / 13.5;
// 11 layers, the smallest gain 1.08. Longer shares lose to the six steps' smaller stages and narrow tiles to wide ones (256 -> 256 at 8^2 x 10 with a
// residual, dense, 18 steps 19.8 / 20.8, 512 -> 512 at 7^2 x 7 25.4 / 28.0, 128 -> 128 at 28^2 x 16 30.4 / 35.5). Eight steps in one window lose there too (512 -> 512
// at 7^2 x 7, T = 8 23.2 / 26.8): nothing is multiplied for steps beyond T, and the activations of a narrow tile come from LDS at its full rate.
int plan_blocked(const char* who, const BlockedCall& c, BlockedPlan& p) {
    if (const int rc = plan_window(who, c, p, 0); rc != SNNF_OK) return rc;
    // Nine timesteps of a 1x1 layer on bits, a wave to a tile: windows of four, four and one. A window of three takes as long to set up as one of four, and the last one of a single step has next to no
    // epilogue (us, three / four, 16 -> 320 at 96^2 x 2 49.5 / 44.8, 24 -> 320 at 111 x 9 x 25 91.8 / 84.4, 64 -> 64 at 96^2 x 8 with a residual 57.1 / 53.4, 96 -> 192 the same; of 64 layers the mean 0.98, where waves
    // share a tile 49 of 1.10).
    if (c.T > 6 && p.tt == 3 && p.g.taps == 1 && p.g.C8in <= 8 && p.wk_log2 == 0 && c.out_layout == SNNF_LAYOUT_BITS && !p.tuned_patch && !p.tuned_split) {
        BlockedPlan four;
        if (plan_window(who, c, four, 0, false) == SNNF_OK) p = four;
        return SNNF_OK;
    }
    if ((c.T != 5 && c.T != 6) || c.shared || c.split || c.shortcut != nullptr || p.tt != 3 || p.few || p.tuned_patch || p.tuned_split || p.g.tap_pairs || !p.g.narrow ||
        p.wk_log2 == 0 || ((p.g.taps * p.g.C8in / 2) >> p.wk_log2) > 16) return SNNF_OK;
    BlockedPlan one;
    if (plan_window(who, c, one, 6) != SNNF_OK || one.wk_log2 == 0) return SNNF_OK;   // (a wave alone has no variant)
    one.few = false;                                   // (the plan above has answered that)
    p = one;
    return SNNF_OK;
}

// Whether a layer of whole tiles beyond the usual line, whose copy is small, moves (see takes_blocked_route): `weigh` is its `tile_use` weighed by the products per output, up
// to 1.1. Of 842 drawn layers there 134 lose, up to a quarter, and what they lose by stands in this kernel's plan: waves without a tile (64 -> 64 at 56^2 x 11 with a residual, 1078 tiles
// on 2048 waves, 37.5 / 43.7), more than two rounds of waves (32 -> 512 at 32^2 x 58, T = 2, with a residual 168 / 190), patches of four columns (64 -> 64 at 48 x 28 x 20 28 / 36), and few
// output channels for a copy (128 -> 64 at 28^2 x 16 with a residual 26 / 28; 24 inputs lose no more often than others). Narrow tiles lose little by idle waves, one
// timestep nothing (116 layers, 1.23). The line takes 471 of the 842 at 1.16 in the mean, 13 of which lose, up to 8 % (40 -> 64 at 16^2 x 25, T = 3 13.8 / 15.0); the others are at 1.03, a third of them below 1.
// 128 -> 128 at 28^2 x 4 20.8 / 17.7, x 16 with a residual 40.8 / 36.5, T = 8 80 / 65, 64 -> 64 at 32^2 x 8 17.0 / 15.2, 64 -> 192 at 28^2 x 48 82 / 70.
bool fills_waves(const BlockedPlan& p, double weigh, int T, int Cout) {
    if (T == 1 || p.few) return true;
    const SpkGeom& g = p.g;
    const double line = weigh * (1.0 + 40.0 / Cout);
    if (g.PC < 8) return false;
    if (g.narrow) return line <= 1.65;
    const double waves = static_cast<double>(g.iters) * compute_units() * kSpkWaves;
    return g.iters <= 2 && line <= 1.55 * std::min(1.0, static_cast<double>(static_cast<int64_t>(g.n_items) << p.wk_log2) / waves);
}

// Whether the kernel reads the dense frames of a call itself (`p`) instead of a launch that brings them into C8 first (`copy`). That launch takes some 3 us and the time of the bytes it moves; without it
// every tile assembles its halo from loads of two pixels of one channel, `loads` of them for a compute unit. What they take goes with the lines that they touch: in long rows (up to 64 elements) a tile's
// rows lie in lines of their own, which come from memory once if the frames are there and from a cache for every further tile of output channels; patches of short rows take more, 1x1 ones
// of a few columns most, whose lines many tiles share, and a wave with a tile of its own waits for its stages in turn. The longer a wave's matrix steps (`steps`, in hundreds), the less of the copy's
// time would have been seen. Fitted to drawn layers, both with frames from the caches, as the layer before leaves them, and from memory: of 1176 and 1229 in 16 bits this takes 793, at 1.25 in the mean
// (7 lose more than a twentieth, the worst 0.86), and 815, at 1.18 (30, the worst 0.68); a line by loads and bytes alone took 892 (26, 0.71) and 937 (103, 0.56), at 1.22 and 1.14. fp32,
// whose pairs take loads of 8 bytes and twice the rounding to two terms: of 672 and 766 332, at 1.23 (5 lose more than a twentieth), and 386, at 1.165 (15, the worst 0.77).
// us, copy / here, T = 4, from the caches: 64 -> 64 at 32^2 x 8 14.6 / 11.5, 128 -> 128 at 28^2 x 16 36.1 / 34.0, at 20^2 x 7 16.0 / 12.1, 256 -> 256 at 14^2 x 16 30.5 / 27.7, 168 -> 56 1x1 at 36^2 x 4 17.0 / 9.8, 72 -> 104 at 27 x 35 x 5
// with a residual, T = 6 28.4 / 25.0, 48 -> 18 1x1 at 9^2 x 9, T = 3 10.7 / 7.1, 88 -> 96 at 104^2 x 2 38.9 / 43.8, fp32 64 -> 64 at 32^2 x 8 16.1 / 14.7, 88 -> 88 at 20^2 x 9, T = 3 16.2 / 11.7, 256 -> 88 1x1 at
// 8^2 x 16 with a residual 13.3 / 9.4, 128 -> 128 at 28^2 x 16 50.4 / 65.7; from memory: 128 -> 128 at 28^2 x 16 35.0 / 34.4, 488 -> 24 1x1 at 16 x 30 x 18, T = 8 64 / 114, 352 -> 24 at 76^2 x 3 with a residual 62 / 85,
// 400 -> 24 at 27 x 79 x 2 25.4 / 33.0, fp32 424 -> 24 1x1 at 35^2 x 17, T = 5 90 / 117.
// Halo rows of whole pairs can make the planner's choice another one. Where fewer waves then share a tile's K, or stages are shorter, the copy stays (7x7 stride 2 116 -> 72 at 34 x 27 x 25, T = 1, two waves for four
// 25.7 / 40.1, 376 -> 32 at 40 x 54 x 12 with a residual 80 / 119; fp32 384 -> 19 1x1 at 69 x 33 x 5 with a residual, stages of four groups for eight, 37.2 / 48.8).
// 1x1 layers of many channels in patches of up to four columns of long rows touch a line of every channel and row for a pair or two of it. Where the frames are larger than the L2 caches hold beside each
// other, the line is gone before the next tile asks for it, and the copy stays, or the dense kernel where the route has no copy (of 573 drawn 1x1 layers that go past the lines below ten are
// stopped by this one, 0.80 in the mean: us, copy or dense / here, 168 -> 104 at 110 x 58 x 8 with a residual, T = 1 35.8 / 95.1, 456 -> 86 at 32 x 83 x 6, T = 2 31.3 / 54.7, 160 -> 29 at 67 x 52 x 18, T = 1 20.8 / 33.2,
// 112 -> 24 at 16 x 57 x 31, T = 4 34.0 / 43.1, fp32 432 -> 30 at 80 x 52 x 18, T = 1 64 / 91; 7.5 MB, 306 -> 60 at 7 x 35 x 25, T = 2 16.4 / 10.7).
// Strided layers of up to two channel groups are not among the measured and keep the copy, as do rows of one pixel, which have no pairs.
bool reads_steps(const BlockedPlan& p, const BlockedPlan& copy, int T, bool split) {
    const SpkGeom& g = p.g;
    if (g.W < 2 || (g.C8in <= 2 && (g.sh > 1 || g.sw > 1))) return false;
    if (p.wk_log2 < copy.wk_log2 || g.G < copy.g.G) return false;
    const int cus = compute_units();
    const double units = std::min(p.grid, cus);
    const double loads = static_cast<double>(g.n_items) / units * g.C8in * g.region * T / 16.0;
    const double megabytes = static_cast<double>(g.N) * g.C8in * g.H * g.W * T * 16e-6;      // of one term
    const double shares = static_cast<double>(static_cast<int64_t>(g.n_items) << p.wk_log2) / (static_cast<double>(cus) * kSpkWaves);      // of tiles, to a wave
    const double steps = 0.01 * g.taps * g.C8in / 2.0 * p.tt * p.windows * (g.narrow ? 1 : 2) * std::max(std::ceil(shares) / (1 << p.wk_log2), 2.0 * shares / (1 << p.wk_log2));
    if (g.taps == 1 && g.PC <= 4 && g.W >= 20 && g.C8in >= 10 && megabytes * (split ? 2.0 : 1.0) > 8.0) return false;
    if (split) return 3.0 + 0.25 * megabytes > loads * (0.0075 + (p.wk_log2 == 0 ? 0.0022 : 0.0) + (g.PC < 8 ? 0.0006 : 0.0) + (g.taps == 1 ? 0.0016 : 0.0)) + 0.3 * steps;
    const bool strided = g.sh > 1 || g.sw > 1;
    return 3.0 + megabytes * (0.74 - 0.37 / p.oc_tiles) > loads * (0.0031 + (p.wk_log2 == 0 ? 0.0031 : 0.0) + (g.PC < 8 ? 0.0019 : 0.0) + (g.taps == 1 && g.PC <= 4 ? 0.0073 : 0.0) -
                                                                  (strided ? 0.0014 : 0.0) + 0.0075 * std::min(g.W, 64) / 64.0) + 0.37 * steps;
}

// The same for the kernel of few pixels: a workgroup's threads bring in its halo item by item, eight loads each, which takes what the copy does at some 2300 items of all timesteps.
// Workgroups of one column fragment, the smallest launches: the others keep the copy.
// us, copy / here, 47 layers: 32 -> 64 at 12^2, T = 4 7.7 / 5.9 (256 items), 128 -> 256 at 8^2 8.1 / 6.9 (1024), 128 -> 256 at 8^2, T = 8 10.4 / 10.0 (2048); 512 -> 512 at 2^2 10.9 / 12.7 (4096), at 7^2 12.2 / 16.6 (6912).
bool few_reads_steps(const BlockedPlan& p, bool split) { return p.few && !split && p.few_g.frags == 1 && static_cast<int64_t>(p.few_g.Gs) * p.few_g.region * p.few_g.T <= 2304; }

const char* family_name(DenseFamily f) {
    return f == DenseFamily::kTInM ? "t_in_m" : (f == DenseFamily::kTimeOuter ? "time_outer" : (f == DenseFamily::kPointwise ? "pointwise" : "matrix"));
}

// (kStepsRoute: the blocked route, whose kernel reads the dense frames itself; one launch.)
enum DenseRouteKind { kNoRoute, kCopyRoute, kFrameRoute, kStepsRoute };
void plan_text(char* text, const BlockedPlan& p, const char* kernel, int epilogue, int window, DenseRouteKind route) {
    const SpkGeom& g = p.g;
    snprintf(text, 256,
             "kernel=%s variant=%d window=%d launches=%d tile=%dx%dx%d halo=%dx%d waves=8x1x%d oc_tiles=%d oc_tile=%d px_tiles=%d "
             "stage_chunks=%d run=0 lds=%zu grid=%d tuned=%d shortcut_stages=%d%s",
             kernel, (p.wk_log2 > 0 ? 50 : 40) + p.tt + epilogue, window, route == kCopyRoute ? 2 : 1, g.PI, g.PR, g.PC, g.RR, g.RC, 1 << p.wk_log2, p.oc_tiles,
             g.narrow ? 32 : 64, g.n_patches, g.G, p.lds_bytes, p.grid, (p.tuned_patch ? 1 : 0) + (p.tuned_split ? 2 : 0), g.sc_stages,
             route == kCopyRoute ? " route=c8 ran=blocked" : (route == kFrameRoute ? " route=frame ran=blocked" : (route == kStepsRoute ? " route=c8 ran=blocked reads=frames" : "")));
    // A launch of few pixels: the workgroups (images x rows x columns x channels x their number) that run instead of the tiles above.
    if (p.few) {
        const size_t n = strlen(text);
        snprintf(text + n, 256 - n, " few=%dx%dx%dx16x%d", p.few_g.PI, p.few_g.PR, p.few_g.PC, p.few_g.grid);
    }
}

// Whether a layer takes the blocked route: where the rule sends it there and the kernel then runs it. A layer that the planner refuses
// (offsets, a kernel of too many steps, no patch that fits) gets no scratch memory asked for. Without a neuron the dense route has the
// matrix kernel only; what it refuses stays refused. The answer depends on the layer and the table of tuned plans alone and is
// kept per layer with the plan and its text (made anew in each call they took 0.6 of its 11.5 us; it asks twice).
using RouteKey = std::array<int, 16>;
struct KeptPlan {
    BlockedPlan plan;
    char text[2][256];                                 // with the general and with the dense epilogue
    bool few_steps;                                    // the kernel for few pixels reads the dense frames itself (`few_reads_steps`)
    BlockedPlan steps;                                 // of the kernel on the dense frames themselves, where the dense epilogue applies (see `reads_steps`; grid 0: never)
    char steps_text[256];
    bool steps_only;                                   // a call that doesn't read its frames stays on the dense kernels (one window)
};
struct Route { bool taken; DenseFamily family; std::shared_ptr<const KeptPlan> kept; };
std::mutex routes_mutex;
std::map<RouteKey, Route>& routes() {
    static std::map<RouteKey, Route> known;
    return known;
}
constexpr size_t kMaxRoutes = 4096;

// Outputs (elements, all steps) up to which the blocked kernel takes a frame's layer. It is bound by its stores, 2-byte elements in runs of a patch row, which share lines with the next
// patch's, and falls behind where many are under way (that the caches then no longer hold them until they are whole is a guess). Quotients of the dense kernel's time and this one's, over 200 layers, by millions of outputs:
// * strided whole tiles of the matrix kernel (stems): 1.18 from 40 to 63 (the smallest 1.05), 0.98 to 84, 1.05 to 101 (8 of these 13 up to 1.00, down to 0.90), 0.93 beyond: 3 -> 64 7x7
//   stride 2 at 224^2 x 18 66 / 60 us, x 20 75 / 82, x 24 96 / 96, x 28 113 / 122, T = 8, x 10 53 / 59;
// * 1x1 on the time-outer kernel: 2.2 to 84 (the smallest 1.6), 0.64 to 5 at 84 to 100, half of them below 1 beyond (4 -> 96 at 96 x 25 x 50, T = 8 81 / 126);
// * whole tiles of stride 1 1.14 to 63, 1.4 to 84, 1.07 to 101, 0.94 to 1.45 beyond; layers that tiles do not divide 2.2, 1.8 (one of 7 loses, 0.95), 1.6 and, beyond, 1.36 (29 layers, two of which lose: 0.80, 0.90).
int64_t most_frame_outputs(DenseFamily family, bool strided) {
    if (family == DenseFamily::kTInM || family == DenseFamily::kTimeOuter) return 5ll << 24;
    return family == DenseFamily::kMatrixWhole && strided ? 15ll << 22 : 3ll << 25;
}

// `frame`: one input of at most eight channels for all timesteps, which the kernel reads as it is.
Route blocked_route(int T, int N, int Cin, int H, int W, int x_dtype, int Cout, int KH, int KW, int stride_h, int stride_w, int pad_h, int pad_w,
                    int v_dtype, bool residual, bool neuron, bool frame = false) {
    if (!valid_dtype(x_dtype) || (v_dtype != SNNF_F32 && v_dtype != x_dtype)) return {false, DenseFamily::kTInM, nullptr};
    const bool split = x_dtype == SNNF_F32;
    const RouteKey key = {T, N, Cin, H, W, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, residual ? 1 : 0, neuron ? 1 : 0, split ? 1 : 0, frame ? 1 : 0};
    {
        std::lock_guard<std::mutex> lock(routes_mutex);
        const auto it = routes().find(key);
        if (it != routes().end()) return it->second;
    }
    Route route = {false, DenseFamily::kTInM, nullptr};
    double weigh;
    route.taken = takes_blocked_route(T, N, Cin, H, W, x_dtype, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, v_dtype, residual, neuron, route.family, weigh) &&
                  (neuron || (!split && (route.family == DenseFamily::kMatrixMasked || route.family == DenseFamily::kMatrixWhole)));
    if (frame)                                         // (see takes_frame)
        route.taken = route.family != DenseFamily::kPointwise &&
                      static_cast<int64_t>(T) * N * Cout * ((H + 2 * pad_h - KH) / stride_h + 1) * ((W + 2 * pad_w - KW) / stride_w + 1) <=
                          most_frame_outputs(route.family, stride_h > 1 || stride_w > 1);
    if (route.taken) {
        const auto kept = std::make_shared<KeptPlan>();
        BlockedPlan& plan = kept->plan;
        route.taken = plan_blocked("snnf_conv_lif_scratch_bytes", BlockedCall{T, N, Cin, H, W, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w,
                                   frame ? SNNF_LAYOUT_NCHW : SNNF_LAYOUT_C8, residual ? SNNF_LAYOUT_NCHW : -1, SNNF_LAYOUT_NCHW, 0, frame, neuron, false, neuron, false,
                                   nullptr, split}, plan) == SNNF_OK &&
                      (frame || weigh <= 0.0 || fills_waves(plan, weigh, T, Cout));
        if (route.taken) {
            for (int dense_epi = 0; dense_epi < 2; ++dense_epi) plan_text(kept->text[dense_epi], plan, family_name(route.family), dense_epi ? 40 : 0, frame ? T : plan.tt,
                                                                                  frame ? kFrameRoute : (few_reads_steps(plan, split) ? kStepsRoute : kCopyRoute));
            kept->few_steps = !frame && few_reads_steps(plan, split);
            if (!frame && neuron && !plan.few) {
                BlockedPlan direct;
                if (plan_blocked("snnf_conv_lif", BlockedCall{T, N, Cin, H, W, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, kSpkSteps, residual ? SNNF_LAYOUT_NCHW : -1,
                                 SNNF_LAYOUT_NCHW, 0, false, true, false, true, false, nullptr, split}, direct) == SNNF_OK && reads_steps(direct, plan, T, split) &&
                    direct.windows <= std::max(plan.windows, plan.tt > 4 ? 2 : 1)) {   // (the scratch memory holds what passes from window to window of `plan`)
                    kept->steps = direct;
                    plan_text(kept->steps_text, direct, family_name(route.family), 40, direct.tt, kStepsRoute);
                }
            }
            kept->steps_only = weigh < 0.0;
            if (kept->steps_only && (kept->steps.grid == 0 || kept->steps.windows > 1)) route.taken = false;
            else route.kept = kept;
        }
    }
    std::lock_guard<std::mutex> lock(routes_mutex);
    if (routes().size() >= kMaxRoutes) routes().clear();
    routes()[key] = route;
    return route;
}

// fp32 elements that pass from window to window beside a 16-bit membrane, and room for them in calls of more than four timesteps.
int64_t carried_membrane(const Route& r, int v_dtype, int N, int H, int W, int Cout, int KH, int KW, int stride_h, int stride_w, int pad_h, int pad_w) {
    if (v_dtype == SNNF_F32 || (r.kept->plan.windows <= 1 && r.kept->plan.tt <= 4)) return 0;   // (one window of six keeps the answer that two had)
    return static_cast<int64_t>(N) * Cout * ((H + 2 * pad_h - KH) / stride_h + 1) * ((W + 2 * pad_w - KW) / stride_w + 1);
}

// The scratch memory of a layer. A kernel that always reads the frames itself needs none: a token asks for the route.
RouteSpace scratch_space(const Route& r, int T, int N, int Cin, int H, int W, int x_dtype, int v_dtype, bool neuron, int Cout, int KH, int KW, int stride_h, int stride_w, int pad_h, int pad_w) {
    if (!r.kept->steps_only) return route_space(T, N, Cin, H, W, x_dtype == SNNF_F32, neuron ? carried_membrane(r, v_dtype, N, H, W, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w) : 0);
    RouteSpace token = {};
    token.step = 16;
    token.total = token.carry = static_cast<size_t>(T) * token.step;
    return token;
}

// A call on dense tensors that runs here: its inputs, which are brought into C8 first (null: a frame, which is read as it is), and its plan.
struct DenseRoute {
    const void* const* xs;
    const KeptPlan* kept;
    RouteSpace space;
    int v_dtype;
    bool apart;                                        // the call writes nothing where its inputs lie, so that the kernel may read them as they are
};

}  // namespace

int launch_steps_to_c8(const StepPtrs& xs, int T, void* dst, int N, int C, int H, int W, hipStream_t stream);   // snnf_layout.hip
int launch_steps_to_c8_split(const StepPtrs& xs, int T, void* dst, void* flags, int64_t lo_offset, int64_t flag_stride, int N, int C, int H, int W,
                             hipStream_t stream);

char* conv_plan_buffer();   // the thread's plan text (snnf_conv_igemm.hip), shared with snnf_conv_last_plan()

namespace {
int conv_lif_blocked_impl(const char* who, const void* const* xs, int x_layout, const void* const* residuals, int res_layout, int T,
                          int N, int Cin, int H, int W, int x_dtype, const void* packed_weight, int Cout, int KH,
                          int KW, int stride_h, int stride_w, int pad_h, int pad_w, const void* v_init, void* out,
                          int out_layout, int64_t out_step_stride, void* v_out, int neuron, float v_threshold,
                          float v_reset, float tau, void* stream, const Shortcut* sc, bool pool2 = false, const DenseRoute* dense = nullptr);
}  // namespace

}  // namespace snnf

extern "C" int snnf_conv_blocked_tune(int T, int N, int Cin, int H, int W, int Cout, int KH, int KW, int stride_h, int stride_w,
                                      int pad_h, int pad_w, int shared_frame, int patch_cols, int stage_groups, int k_waves) {
    using namespace snnf;
    if (patch_cols < 0 || patch_cols > 32 || stage_groups < 0 || k_waves < 0 || k_waves > kSpkWaves || (k_waves & (k_waves - 1)) != 0)
        return fail(SNNF_ERR_INVALID_ARGUMENT, "snnf_conv_blocked_tune: patch_cols=%d stage_groups=%d k_waves=%d out of range", patch_cols,
                    stage_groups, k_waves);
    const TunedKey key = {T, N, Cin, H, W, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, shared_frame ? 1 : 0};
    {
        std::lock_guard<std::mutex> lock(tuned_mutex);
        if (patch_cols == 0 && stage_groups == 0 && k_waves == 0) tuned_plans().erase(key);
        else tuned_plans()[key] = TunedPlan{patch_cols, stage_groups, k_waves};
    }
    std::lock_guard<std::mutex> lock(routes_mutex);
    routes().clear();
    return SNNF_OK;
}

extern "C" int snnf_conv_lif_blocked(const void* const* xs, int x_layout, const void* const* residuals, int res_layout, int T,
                                     int N, int Cin, int H, int W, int x_dtype, const void* packed_weight, int Cout, int KH,
                                     int KW, int stride_h, int stride_w, int pad_h, int pad_w, const void* v_init, void* out,
                                     int out_layout, int64_t out_step_stride, void* v_out, int neuron, float v_threshold,
                                     float v_reset, float tau, void* stream) {
    return snnf::conv_lif_blocked_impl("snnf_conv_lif_blocked", xs, x_layout, residuals, res_layout, T, N, Cin, H, W, x_dtype, packed_weight,
                                       Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, v_init, out, out_layout, out_step_stride, v_out,
                                       neuron, v_threshold, v_reset, tau, stream, nullptr);
}

extern "C" int snnf_conv_lif_blocked_shortcut(const void* const* xs, const void* const* shortcut_xs, int T, int N, int Cin, int H, int W,
                                              int x_dtype, const void* packed_weight, int Cout, int KH, int KW, int pad_h, int pad_w,
                                              int shortcut_Cin, int shortcut_H, int shortcut_W, int shortcut_stride_h, int shortcut_stride_w,
                                              const void* shortcut_packed_weight, const void* v_init, void* out, int out_layout,
                                              int64_t out_step_stride, void* v_out, int neuron, float v_threshold, float v_reset, float tau,
                                              void* stream) {
    using namespace snnf;
    const char* who = "snnf_conv_lif_blocked_shortcut";
    if (shortcut_xs == nullptr || shortcut_packed_weight == nullptr)
        return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: shortcut_xs and shortcut_packed_weight must be non-null", who);
    const Shortcut sc = {shortcut_xs, shortcut_Cin, shortcut_H, shortcut_W, shortcut_stride_h, shortcut_stride_w, shortcut_packed_weight};
    return conv_lif_blocked_impl(who, xs, SNNF_LAYOUT_BITS, nullptr, SNNF_LAYOUT_BITS, T, N, Cin, H, W, x_dtype, packed_weight, Cout, KH, KW, 1, 1,
                                 pad_h, pad_w, v_init, out, out_layout, out_step_stride, v_out, neuron, v_threshold, v_reset, tau, stream, &sc);
}

extern "C" int snnf_conv_lif_blocked_avgpool(const void* const* xs, int x_layout, int T, int N, int Cin, int H, int W, int x_dtype,
                                             const void* packed_weight, int Cout, int KH, int KW, int stride_h, int stride_w, int pad_h,
                                             int pad_w, void* out, int64_t out_step_stride, void* v_out, float v_threshold, float v_reset,
                                             float tau, void* stream) {
    return snnf::conv_lif_blocked_impl("snnf_conv_lif_blocked_avgpool", xs, x_layout, nullptr, 0, T, N, Cin, H, W, x_dtype, packed_weight, Cout, KH,
                                       KW, stride_h, stride_w, pad_h, pad_w, nullptr, out, SNNF_LAYOUT_C8, out_step_stride, v_out, 1, v_threshold,
                                       v_reset, tau, stream, nullptr, true);
}

extern "C" size_t snnf_conv_lif_workspace_bytes(int T, int N, int Cin, int H, int W, int x_dtype, int Cout, int KH, int KW, int stride_h,
                                                int stride_w, int pad_h, int pad_w, int v_dtype, int residual) {
    if ((x_dtype != SNNF_BF16 && x_dtype != SNNF_F16) || v_dtype != SNNF_F32) return 0;
    return snnf_conv_lif_scratch_bytes(T, N, Cin, H, W, x_dtype, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, v_dtype, residual);
}

extern "C" size_t snnf_conv_lif_scratch_bytes(int T, int N, int Cin, int H, int W, int x_dtype, int Cout, int KH, int KW, int stride_h,
                                              int stride_w, int pad_h, int pad_w, int v_dtype, int residual) {
    using namespace snnf;
    const Route route = blocked_route(T, N, Cin, H, W, x_dtype, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, v_dtype, residual != 0, true);
    if (!route.taken) return 0;
    return scratch_space(route, T, N, Cin, H, W, x_dtype, v_dtype, true, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w).total;
}

extern "C" size_t snnf_conv_bias_workspace_bytes(int T, int N, int Cin, int H, int W, int x_dtype, int Cout, int KH, int KW, int stride_h,
                                                 int stride_w, int pad_h, int pad_w, int residual) {
    using namespace snnf;
    if (!blocked_route(T, N, Cin, H, W, x_dtype, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, SNNF_F32, residual != 0, false).taken) return 0;
    return route_space(T, N, Cin, H, W, false, 0).total;
}

namespace snnf {
namespace {
// The neuron of the dense epilogue.
bool dense_epilogue_neuron(const LifParams& lif) { return lif.charge_mode == CHARGE_SCALE && lif.inv_tau == 0.5f && !lif.soft_reset; }

// One dense 16-bit frame of at most eight channels for all timesteps (the first layer of a network) around the usual neuron (tau 2, hard reset) goes to the
// blocked kernel, which reads the frame as it is and needs no scratch memory (us, matrix kernel / here, T = 4, bf16): 3 -> 64 7x7 stride 2 at 224^2 x 16 62.8 / 48.5, one
// image 14.6 / 9.9, 3x3 at 32^2 x 64 19.7 / 14.2, one image 11.5 / 6.9, 3 -> 32 stride 2 at 128^2 x 32 33.3 / 14.6, 1 -> 64 5x5 at 28^2 x 50 18.6 / 14.6, 4 -> 96 at 50^2 x 20
// 40.3 / 20.3, 8 -> 128 at 56^2 x 16 35.5 / 25.4; T = 8 3 -> 64 3x3 at 32^2 x 64 25.8 / 18.7, 4 -> 96 60.3 / 31.2. What the pointwise kernel takes stays there (8 -> 256 1x1 at
// 56^2 x 16 33.4 / 50.9), and more outputs than `most_frame_outputs`. Other neurons take its general epilogue, which is slower than the matrix kernel's
// (77.5 at 224^2 x 16), and stay.
bool takes_frame(bool shared, int T, int Cin, int x_dtype, int v_dtype, bool residual, const LifParams& lif) {
    return shared && T <= SNNF_MAX_T_PER_LAUNCH && Cin <= 8 && (x_dtype == SNNF_BF16 || x_dtype == SNNF_F16) && v_dtype == SNNF_F32 && !residual &&
           dense_epilogue_neuron(lif);
}

// The blocked route of a call on dense tensors: SNNF_ERR_UNSUPPORTED (nothing enqueued) when it does not apply.
int run_blocked_route(const void* const* xs, const void* const* residuals, int T, int N, int Cin, int H, int W, int x_dtype, const void* packed_weight,
                      int Cout, int KH, int KW, int stride_h, int stride_w, int pad_h, int pad_w, const void* v_init, int v_dtype, void* out,
                      int64_t out_step_stride, void* v_out, int neuron, float v_threshold, float v_reset, float tau, void* workspace,
                      size_t workspace_bytes, void* stream) {
    if (xs == nullptr || (neuron && v_out == nullptr) || out_step_stride < 0 || T < 1 || T > SNNF_MAX_T_PER_LAUNCH || N < 1 || Cin < 1 || H < 1 || W < 1 || Cout < 1 ||
        KH < 1 || KW < 1 || stride_h < 1 || stride_w < 1 || pad_h < 0 || pad_w < 0 || H + 2 * pad_h < KH || W + 2 * pad_w < KW || 2 * pad_h > KH || 2 * pad_w > KW || tau == 0.0f)
        return SNNF_ERR_UNSUPPORTED;
    bool shared = T > 1;
    for (int t = 0; t < T; ++t) {
        if (xs[t] == nullptr) return SNNF_ERR_UNSUPPORTED;
        shared = shared && xs[t] == xs[0];
    }
    if (neuron && takes_frame(shared, T, Cin, x_dtype, v_dtype, residuals != nullptr, make_lif_params(v_threshold, v_reset, tau))) {
        const Route frame = blocked_route(T, N, Cin, H, W, x_dtype, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, v_dtype, false, true, true);
        if (!frame.taken) return SNNF_ERR_UNSUPPORTED;
        const DenseRoute route = {nullptr, frame.kept.get(), RouteSpace{}, v_dtype, false};
        return conv_lif_blocked_impl("snnf_conv_lif", xs, SNNF_LAYOUT_NCHW, nullptr, SNNF_LAYOUT_NCHW, T, N, Cin, H, W, x_dtype, packed_weight, Cout, KH, KW, stride_h, stride_w,
                                     pad_h, pad_w, v_init, out, SNNF_LAYOUT_NCHW, out_step_stride * dtype_size(x_dtype), v_out, 1, v_threshold, v_reset, tau, stream, nullptr,
                                     false, &route);
    }
    if (workspace == nullptr || !aligned_to(workspace, 16) || shared) return SNNF_ERR_UNSUPPORTED;   // one frame for all timesteps is convolved once on the dense kernels too
    const Route taken = blocked_route(T, N, Cin, H, W, x_dtype, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, v_dtype, residuals != nullptr, neuron != 0);
    if (!taken.taken) return SNNF_ERR_UNSUPPORTED;
    const RouteSpace space = scratch_space(taken, T, N, Cin, H, W, x_dtype, v_dtype, neuron != 0, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w);
    if (workspace_bytes < space.total) return SNNF_ERR_UNSUPPORTED;
    const int size = dtype_size(x_dtype);
    const auto to = reinterpret_cast<uintptr_t>(out), v = reinterpret_cast<uintptr_t>(v_out);
    const uintptr_t neurons = static_cast<uintptr_t>(N) * Cout * ((H + 2 * pad_h - KH) / stride_h + 1) * ((W + 2 * pad_w - KW) / stride_w + 1);
    const uintptr_t to_end = to + (static_cast<uintptr_t>(T - 1) * static_cast<uintptr_t>(out_step_stride) + neurons) * size;
    const bool apart = std::all_of(xs, xs + T, [&](const void* x) {
        const auto in = reinterpret_cast<uintptr_t>(x), in_end = in + static_cast<uintptr_t>(N) * Cin * H * W * size;
        return aligned_to(x, size) && (in >= to_end || to >= in_end) && (v_out == nullptr || in >= v + neurons * dtype_size(v_dtype) || v >= in_end);
    });
    if (taken.kept->steps_only && !(apart && dense_epilogue_neuron(make_lif_params(v_threshold, v_reset, tau)))) return SNNF_ERR_UNSUPPORTED;
    const void* inner[SNNF_MAX_T_PER_LAUNCH];
    for (int t = 0; t < T; ++t) inner[t] = static_cast<const char*>(workspace) + t * space.step;
    const DenseRoute route = {xs, taken.kept.get(), space, v_dtype, apart};
    return conv_lif_blocked_impl(neuron ? "snnf_conv_lif" : "snnf_conv_bias", inner, SNNF_LAYOUT_C8, residuals, SNNF_LAYOUT_NCHW, T, N, Cin, H, W, x_dtype,
                                 packed_weight, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, v_init, out, SNNF_LAYOUT_NCHW, out_step_stride * dtype_size(x_dtype), v_out,
                                 neuron, v_threshold, v_reset, tau, stream, nullptr, false, &route);
}
}  // namespace
}  // namespace snnf

extern "C" int snnf_conv_lif_ws(const void* const* xs, const void* const* residuals, int T, int N, int Cin, int H, int W, int x_dtype,
                                const void* packed_weight, int Cout, int KH, int KW, int stride_h, int stride_w, int pad_h, int pad_w,
                                const void* v_init, int v_dtype, void* spikes, int64_t spike_step_stride, void* v_out, float v_threshold,
                                float v_reset, float tau, void* workspace, size_t workspace_bytes, void* stream) {
    const int rc = snnf::run_blocked_route(xs, residuals, T, N, Cin, H, W, x_dtype, packed_weight, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, v_init,
                                           v_dtype, spikes, spike_step_stride, v_out, 1, v_threshold, v_reset, tau, workspace, workspace_bytes, stream);
    if (rc != SNNF_ERR_UNSUPPORTED) return rc;
    return snnf_conv_lif(xs, residuals, T, N, Cin, H, W, x_dtype, packed_weight, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, v_init, v_dtype, spikes,
                         spike_step_stride, v_out, v_threshold, v_reset, tau, stream);
}

extern "C" int snnf_conv_bias_ws(const void* const* xs, const void* const* residuals, int T, int N, int Cin, int H, int W, int x_dtype,
                                 const void* packed_weight, int Cout, int KH, int KW, int stride_h, int stride_w, int pad_h, int pad_w, void* out,
                                 int64_t out_step_stride, void* workspace, size_t workspace_bytes, void* stream) {
    const int rc = snnf::run_blocked_route(xs, residuals, T, N, Cin, H, W, x_dtype, packed_weight, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, nullptr,
                                           SNNF_F32, out, out_step_stride, nullptr, 0, 1.0f, 0.0f, 2.0f, workspace, workspace_bytes, stream);
    if (rc != SNNF_ERR_UNSUPPORTED) return rc;
    return snnf_conv_bias(xs, residuals, T, N, Cin, H, W, x_dtype, packed_weight, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, out, out_step_stride, stream);
}

namespace snnf {
namespace {
int conv_lif_blocked_impl(const char* who, const void* const* xs, int x_layout, const void* const* residuals, int res_layout, int T,
                          int N, int Cin, int H, int W, int x_dtype, const void* packed_weight, int Cout, int KH,
                          int KW, int stride_h, int stride_w, int pad_h, int pad_w, const void* v_init, void* out,
                          int out_layout, int64_t out_step_stride, void* v_out, int neuron, float v_threshold,
                          float v_reset, float tau, void* stream, const Shortcut* sc, bool pool2, const DenseRoute* dense) {
    if (xs == nullptr || packed_weight == nullptr || out == nullptr)
        return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: xs, packed_weight and out must be non-null", who);
    if (T < 1 || N < 1 || Cin < 1 || H < 1 || W < 1 || Cout < 1 || KH < 1 || KW < 1 || stride_h < 1 || stride_w < 1 || pad_h < 0 || pad_w < 0)
        return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: bad extent (T=%d N=%d Cin=%d H=%d W=%d Cout=%d K=%dx%d s=%dx%d p=%dx%d)", who,
                    T, N, Cin, H, W, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w);
    if (T > SNNF_MAX_T_PER_LAUNCH)
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_temporal_length: T=%d exceeds %d", who, T, SNNF_MAX_T_PER_LAUNCH);
    const bool split = dense != nullptr && x_dtype == SNNF_F32;
    if (x_dtype != SNNF_BF16 && x_dtype != SNNF_F16 && !split)
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_dtype: the internal layouts hold bf16 or fp16 activations", who);
    if (x_layout != SNNF_LAYOUT_C8 && x_layout != SNNF_LAYOUT_BITS && x_layout != SNNF_LAYOUT_NCHW)
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_layout: inputs must be in C8 or BITS layout (or one dense frame of at most 8 channels)", who);
    if (!valid_layout(out_layout) || (residuals != nullptr && !valid_layout(res_layout)))
        return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: unknown layout code", who);
    if (!neuron && out_layout == SNNF_LAYOUT_BITS)
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_layout: an output without a neuron cannot be bit-packed", who);
    if (neuron && !(tau != 0.0f)) return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_tau: tau must be nonzero", who);
    if (H + 2 * pad_h < KH || W + 2 * pad_w < KW)
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_kernel: kernel larger than padded input", who);
    if (2 * pad_h > KH || 2 * pad_w > KW)
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_padding: padding %dx%d too large for kernel %dx%d", who, pad_h, pad_w, KH, KW);
    // Bytes a tensor in a layout is accessed by: bit-packed tensors by single bytes, blocked inputs by 16-byte groups, blocked
    // outputs and residuals by 4 channels (8 bytes), dense tensors by elements.
    auto need_align = [x_dtype](int layout, bool as_input) -> size_t { return layout == SNNF_LAYOUT_BITS ? 1 : (layout == SNNF_LAYOUT_C8 ? (as_input ? 16 : 8) : static_cast<size_t>(dtype_size(x_dtype))); };
    const size_t v_align = dense != nullptr && dense->v_dtype != SNNF_F32 ? 2 : 4;
    if (!aligned_to(packed_weight, 16) || !aligned_to(out, need_align(out_layout, false)) || (out_step_stride % need_align(out_layout, false)) != 0 ||
        (v_init != nullptr && !aligned_to(v_init, v_align)) || (v_out != nullptr && !aligned_to(v_out, v_align)))
        return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: packed_weight, out (and its step stride) or a membrane pointer is misaligned", who);
    bool shared = T > 1;
    for (int t = 0; t < T; ++t) {
        if (xs[t] == nullptr || !aligned_to(xs[t], need_align(x_layout, true)))
            return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: xs[%d] is null or misaligned for its layout", who, t);
        if (residuals != nullptr && (residuals[t] == nullptr || !aligned_to(residuals[t], need_align(res_layout, false))))
            return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: residuals[%d] is null or misaligned for its layout", who, t);
        shared = shared && xs[t] == xs[0];
    }
    if (x_layout == SNNF_LAYOUT_NCHW && (!shared || Cin > 8))
        return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_layout: a dense input must be one frame of at most 8 channels shared by all timesteps (Cin=%d)", who, Cin);
    if (sc != nullptr) {
        // The shortcut's sums are K steps of the main tile: same output pixels (a main convolution that keeps the plane, the
        // shortcut's stride taking its own input down to it), whole pairs of channel groups, bit-packed input like the main one.
        if (sc->Cin < 1 || sc->H < 1 || sc->W < 1 || sc->stride_h < 1 || sc->stride_w < 1)
            return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: bad shortcut extent (Cin=%d H=%d W=%d s=%dx%d)", who, sc->Cin, sc->H, sc->W, sc->stride_h, sc->stride_w);
        if (KH != 2 * pad_h + 1 || KW != 2 * pad_w + 1 || (sc->H - 1) / sc->stride_h + 1 != H || (sc->W - 1) / sc->stride_w + 1 != W)
            return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_shortcut: the main convolution must keep its %dx%d plane and the shortcut (%dx%d, stride %dx%d) must land on it",
                        who, H, W, sc->H, sc->W, sc->stride_h, sc->stride_w);
        if (sc->Cin % 16 != 0 || Cin % 16 != 0 || shared || T < 3)
            return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_shortcut: needs channel counts that are multiples of 16, at least 3 timesteps and an input per timestep", who);
        if (!aligned_to(sc->packed_weight, 16))
            return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: shortcut_packed_weight is misaligned", who);
        if (static_cast<int64_t>(N) * (sc->Cin / 8) * sc->H * sc->W >= (1LL << 27))
            return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_shape: shortcut input too large for 32-bit offsets", who);
        for (int t = 0; t < T; ++t)
            if (sc->xs[t] == nullptr) return fail(SNNF_ERR_INVALID_ARGUMENT, "%s: shortcut_xs[%d] is null", who, t);
    }

    BlockedPlan made;
    if (dense == nullptr) {
        if (const int rc = plan_blocked(who, BlockedCall{T, N, Cin, H, W, Cout, KH, KW, stride_h, stride_w, pad_h, pad_w, x_layout,
                                                         residuals != nullptr ? res_layout : -1, out_layout, out_step_stride, shared, neuron != 0,
                                                         v_init != nullptr, v_out != nullptr, pool2, sc, split}, made); rc != SNNF_OK)
            return rc;
    }
    // (Of a dense call xs are the C8 buffers. The plan of the frames is one of its own: its patches, stages and shares of K can be others than the copy's, and fp32's low terms follow a wave's own stages,
    // so the order of a sum's additions can depend on whether the call may read them as they are.)
    const LifParams lif_params = make_lif_params(v_threshold, v_reset, tau);
    const bool usual = dense_epilogue_neuron(lif_params);
    // (Frames that the call writes to, spikes or membrane, are copied first.)
    const bool frames = dense != nullptr && dense->xs != nullptr && dense->apart;
    const bool steps = frames && dense->kept->steps.grid > 0 && usual && v_out != nullptr &&
                       (dense->kept->steps.windows == 1 || dense->v_dtype == SNNF_F32 || x_dtype == SNNF_F32 || dense->space.total > dense->space.carry);
    const bool few_steps = frames && dense->kept->few_steps;
    const BlockedPlan& p = dense == nullptr ? made : (steps ? dense->kept->steps : dense->kept->plan);
    const SpkGeom& g = p.g;

    SpkLaunch L = {};
    for (int t = 0; t < T; ++t) {
        L.xs.p[t] = steps || few_steps ? dense->xs[t] : xs[t];
        if (residuals != nullptr) L.residuals.p[t] = residuals[t];
        if (sc != nullptr) L.residuals.p[t] = sc->xs[t];   // the second input travels in the residual's place (a shortcut launch has no residual)
    }
    if (sc != nullptr) {
        L.wpacked2 = static_cast<const uint16_t*>(sc->packed_weight);
        L.bias2 = reinterpret_cast<const float*>(L.wpacked2 + packed_weight_elems(p.pg2));
    }
    L.g = g;
    L.g.out_step_stride = out_step_stride;
    L.wpacked = static_cast<const uint16_t*>(packed_weight);
    L.bias = reinterpret_cast<const float*>(L.wpacked + packed_weight_elems(p.pg));
    L.g.v_in_place = neuron && v_init != nullptr && v_init == v_out ? 1 : 0;
    L.v_start = neuron && L.g.v_in_place == 0 ? v_init : nullptr;
    L.out = out;
    L.v_store = neuron ? v_out : nullptr;
    if (dense != nullptr && neuron && dense->v_dtype != SNNF_F32) {
        L.g.v16 = 1;
        L.v_scratch = reinterpret_cast<float*>(static_cast<char*>(const_cast<void*>(xs[0])) + dense->space.carry);
    }
    L.lif = lif_params;
    L.grid = p.grid;
    L.lds_bytes = p.lds_bytes;
    L.stream = as_stream(stream);
    const bool fast_epi = neuron && (out_layout == SNNF_LAYOUT_BITS || pool2) && (residuals == nullptr || res_layout == SNNF_LAYOUT_BITS) &&
                          L.lif.charge_mode == CHARGE_SCALE && L.lif.inv_tau == 0.5f && L.lif.v_reset == 0.0f &&
                          L.lif.v_threshold >= 1e-30f && L.lif.v_threshold <= 1e30f &&   // its multiples by 2^t stay normal numbers
                          v_init == nullptr && (p.windows == 1 || p.tt >= 3) && Cout % 8 == 0;
    // Dense tensors around the neuron: no range limit on the threshold, any reset potential, initial membrane, windows and channels.
    // (A frame for all timesteps: without a residual, with or without a membrane.)
    const bool frame_epi = x_layout == SNNF_LAYOUT_NCHW && shared && residuals == nullptr;
    const bool dense_epi = neuron && (frame_epi || (x_layout == SNNF_LAYOUT_C8 && !shared && L.v_store != nullptr)) && out_layout == SNNF_LAYOUT_NCHW &&
                           (residuals == nullptr || res_layout == SNNF_LAYOUT_NCHW) && usual;
    if (steps) memcpy(snnf::conv_plan_buffer(), dense->kept->steps_text, 256);
    else if (dense != nullptr) memcpy(snnf::conv_plan_buffer(), dense->kept->text[dense_epi ? 1 : 0], 256);
    else plan_text(snnf::conv_plan_buffer(), p, "blocked", fast_epi ? 20 : (dense_epi ? 40 : 0), shared ? T : p.tt, kNoRoute);
    L.fast_epilogue = fast_epi;
    L.multi_window = p.windows > 1;
    L.dense_epilogue = dense_epi;
    if (steps && split) return launch_conv_spk_f32_steps(L, p.tt);
    if (steps) return x_dtype == SNNF_BF16 ? launch_conv_spk_bf16_steps(L, p.tt) : launch_conv_spk_f16_steps(L, p.tt);
    if (dense != nullptr && dense->xs != nullptr && !few_steps) {   // the plan stands: bring the dense inputs into the C8 buffers behind `xs`
        StepPtrs from = {};
        for (int t = 0; t < T; ++t) from.p[t] = dense->xs[t];
        char* const base = static_cast<char*>(const_cast<void*>(xs[0]));
        if (split) {
            L.g.lo_offset = static_cast<int64_t>(dense->space.lo);
            L.g.flag_stride = static_cast<int64_t>(dense->space.flag_stride);
            L.lo_flags = reinterpret_cast<const unsigned char*>(base + dense->space.flags);
            if (const int rc = launch_steps_to_c8_split(from, T, base, base + dense->space.flags, L.g.lo_offset, L.g.flag_stride, N, Cin, H, W, L.stream); rc != SNNF_OK)
                return rc;
            return launch_conv_spk_f32(L, p.tt);
        }
        if (const int rc = launch_steps_to_c8(from, T, base, N, Cin, H, W, L.stream); rc != SNNF_OK) return rc;
    }
    if (pool2) {
        if (!fast_epi || p.windows != 1 || (p.tt != 4 && !shared))
            return fail(SNNF_ERR_UNSUPPORTED, "%s: unsupported_pool: the pooled output needs the usual neuron (tau 2, hard reset to 0) and the four steps in one window", who);
    }
    if (p.few) {
        FewLaunch F = {L.xs, L.residuals, p.few_g, L.wpacked, L.bias, L.v_start, L.out, L.v_store, L.lif, p.few_lds, L.stream};
        F.g.out_step_stride = out_step_stride;
        F.g.v16 = L.g.v16;
        F.g.v_in_place = L.g.v_in_place;
        return launch_conv_few(F, x_dtype == SNNF_F16, few_steps ? kSpkSteps : x_layout);
    }
    if (pool2) {
        if (x_layout == SNNF_LAYOUT_NCHW) return x_dtype == SNNF_BF16 ? launch_conv_spk_bf16_frame(L, true) : launch_conv_spk_f16_frame(L, true);
        return x_dtype == SNNF_BF16 ? launch_conv_spk_bf16_pooled(L, p.tt) : launch_conv_spk_f16_pooled(L, p.tt);
    }
    if (sc != nullptr && p.tt == 3) return x_dtype == SNNF_BF16 ? launch_conv_spk_bf16_three_shortcut(L) : launch_conv_spk_f16_three_shortcut(L);
    if (sc != nullptr) return x_dtype == SNNF_BF16 ? launch_conv_spk_bf16_shortcut(L) : launch_conv_spk_f16_shortcut(L);
    if (x_layout == SNNF_LAYOUT_NCHW) return x_dtype == SNNF_BF16 ? launch_conv_spk_bf16_frame(L, false) : launch_conv_spk_f16_frame(L, false);
    if (p.tt == 6) return x_dtype == SNNF_BF16 ? launch_conv_spk_bf16_long(L) : launch_conv_spk_f16_long(L);
    if (p.tt == 3) return x_dtype == SNNF_BF16 ? launch_conv_spk_bf16_three(L) : launch_conv_spk_f16_three(L);
    if (x_layout == SNNF_LAYOUT_BITS) return x_dtype == SNNF_BF16 ? launch_conv_spk_bf16_bits(L, p.tt) : launch_conv_spk_f16_bits(L, p.tt);
    return x_dtype == SNNF_BF16 ? launch_conv_spk_bf16_c8(L, p.tt) : launch_conv_spk_f16_c8(L, p.tt);
}

}  // namespace
}  // namespace snnf
