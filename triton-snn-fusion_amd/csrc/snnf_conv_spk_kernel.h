// Dense convolution + bias (+ residual) + LIF on activations in the library's internal layouts: channel-blocked 16-bit
// values ([N][C/8][H][W][8], "C8") or bit-packed spikes ([N][C/8][H][W] bytes, bit j = channel 8 c8 + j, "BITS"). These
// layouts exist between consecutive fused operators of one network; the operator boundary keeps dense NCHW.
//
// Same implicit GEMM as the NCHW kernels (M = output channels from packed weight fragments, N = pixels, K = taps x
// channel groups of 8, v_mfma_f32_32x32x16, fp32 accumulate, TT timesteps side by side against one weight fragment), but:
//   * a group of 8 channels of one pixel is 16 contiguous bytes in C8 and one byte in BITS, i.e. already the matrix
//     operand of a lane: staging is one load and one 16-byte LDS write per item, no transposition; a spike byte is
//     expanded to eight 16-bit ones with 9 integer instructions on its way into LDS;
//   * every wave is its own pipeline: it owns a patch of 32 output pixels x 64 output channels x TT timesteps, stages
//     the halo of its patch into a private LDS region and never meets a workgroup barrier in the matrix loop, so the
//     eight waves of a compute unit drift apart and one wave's staging and epilogue overlap another's matrix work;
//   * spikes leave as bits: the accumulator layout gives a lane 4 consecutive channels of its pixel, the two halves of
//     a wave exchange their nibbles with one cross-lane move and store bytes; the membrane is fp32 NCHW and optional;
//   * deep layers with few pixels split K over WK waves of a workgroup (whole LDS stages each) and add their partial
//     sums through LDS in a fixed order;
//   * neighbours of a convolution that fit its tile join its launch: the 1x1 projection shortcut of a residual block as
//     further K steps on a second input (SC), the 2x2 average pool of the spikes as a reduce-scatter between the four
//     lanes of a window (POOL), and a network's dense input frame of at most 8 channels read as it is (IN = NCHW).
#pragma once

#include <type_traits>

#include "snnf_conv_common.h"

namespace snnf {

typedef __bf16 sk_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 sk_f16x8 __attribute__((ext_vector_type(8)));
typedef float sk_f32x16 __attribute__((ext_vector_type(16)));
typedef float sk_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t sk_u32x4 __attribute__((ext_vector_type(4)));

constexpr int kSpkWaves = 8;                      // waves per workgroup, one workgroup per compute unit
#ifndef SPK_SLOTS
#define SPK_SLOTS 8
#endif
constexpr int kSpkSlots = SPK_SLOTS;                      // staging items per lane and timestep, at most
constexpr int kSpkPartialBytes = 16 * 64 * 16;     // split-K: a wave parks 4 quads x up to 4 timesteps of partial sums in its region
constexpr int kSpkSteps = 16;                     // an input layout of this kernel alone (no code of the library's): dense frames, one per timestep
constexpr int kSpkMaxSteps = 60;                  // matrix steps per stage, at most (the step table holds 4 more)
constexpr size_t kSpkTableBytes = (kSpkMaxSteps + 4) * 16;      // the workgroup's step table at the start of LDS
constexpr int kSpkDescs = 64 * kSpkSlots;                       // staging items of one timestep, at most
constexpr size_t kSpkDescBytes = kSpkDescs * 8;                 // the workgroup's staging descriptors behind the step table
constexpr size_t kSpkPosBytes = 32 * 8;            // where each of the 32 pixels of a tile sits inside the patch, and its top-left input in the staged halo
constexpr size_t kSpkHeaderBytes = kSpkTableBytes + kSpkDescBytes + kSpkPosBytes;   // what precedes the waves' staging regions in LDS

// n / d for 0 <= n < 2^31 as one multiply-high and a shift, for every d from 1: with s = ceil(log2 d) and mul = ceil(2^(31+s) / d), 2 n mul / 2^32 / 2^s
// exceeds n / d by less than 1 / d. (fast_div's general form takes another multiply or a select for a divisor of 1.)
struct SpkDiv {
    uint32_t mul;
    int shift;
};
inline SpkDiv make_spk_div(int d) {
    int s = 0;
    while ((1LL << s) < d) ++s;
    return {static_cast<uint32_t>(((1ULL << (31 + s)) + static_cast<uint64_t>(d) - 1) / static_cast<uint64_t>(d)), s};
}
__device__ __forceinline__ int sk_div(int n, const SpkDiv& f) { return static_cast<int>(__umulhi(static_cast<uint32_t>(n) * 2u, f.mul) >> f.shift); }

struct SpkGeom {
    int N, Cin, H, W, Cout, KH, KW, sh, sw, ph, pw, Ho, Wo;
    int C8in, C8out;
    int PR, PC, PI;              // patch of a wave: PR x PC output pixels of PI images (PI > 1: whole planes)
    int patches_x, patches_img;  // patches per output row band, per image (patches_x * patches_y)
    int n_patches;               // image groups x patches per image
    int RR, RC;                  // halo rows / columns per image
    int region;                  // PI * RR * RC: 16-byte items per channel group and timestep
    int G;                       // channel groups per LDS stage
    int nstages;                 // ceil(C8in / G)
    int IT, JT;                  // staging items per timestep (G * region) and slots per lane (ceil(IT / 64))
    int gpc;                     // channel groups per packed chunk (CK / 8)
    int npairs;                  // k-slot pairs per packed chunk
    int nocf;                    // 32-row weight fragments
    int tap_pairs;               // packed chunks of 8 channels: a pair of k-slots is two taps of one group
    int taps;
    int T;                       // timesteps
    int shared_x;                // one input frame for all T timesteps (TT == 1): convolved once
    int kw_mul;                  // tap / KW == (tap * kw_mul) >> 16 for every tap of the kernel (branch-free on the scalar unit)
    int gpc_log2;                // log2(gpc)
    int hg_log2;                 // log2 of the k-slot pairs per tap and stage (G / 2; 0 with tap pairs)
    int pair_tap_stride;         // packed pairs between consecutive taps of one group pair (gpc / 2; 1 with tap pairs)
    int wk_log2;                 // split-K: waves per tile
    int n_items, iters;          // (patch, channel tile) pairs; loop trips per wave
    int narrow;                  // tiles of 32 output channels instead of 64
    int in_layout, res_layout, out_layout;   // snnf_layout codes; res_layout < 0: no residual
    int analog_out;              // no neuron: the sums themselves are written (C8 or NCHW)
    int grid;                    // workgroups of the launch (read from here: the hidden arguments lie in a cache line of their own)
    int64_t out_step_stride;     // bytes between timesteps of `out`
    int lds_wave_bytes;          // private staging region of a wave (a multiple of 16)
    int64_t frag_stride;         // 16-bit elements between consecutive 32-row fragments of the packed weight
    // A second, pointwise operand pair that shares the accumulators (the projection shortcut of a residual block: its sums
    // are further K steps of the same output tile). Its input has sc_C8 channel groups on an sc_H x sc_W plane and is
    // sampled at (sc_sh * ih, sc_sw * iw) for the pixel (ih, iw) of the main input; its stages follow the main ones.
    int sc_stages;               // 0: none
    int sc_C8, sc_H, sc_W, sc_sh, sc_sw;
    int sc_gpc_log2, sc_npairs;  // channel groups (log2) and k-slot pairs per packed chunk of the second weight
    int64_t sc_frag_stride;
    // fp32 tensors (SPLIT): the low bf16 terms of the activations lie `lo_offset` bytes behind the high ones, those of the weights
    // `w_lo_offset` elements behind. One byte per 64 items of the C8 tensor tells whether any of them has a low term; only those are written.
    int64_t lo_offset, w_lo_offset;
    int64_t flag_stride;         // bytes of the flags of one timestep (a multiple of 4)
    int v16;                     // v_start and v_store hold the activation dtype; the windows in between pass v_scratch on
    int v_in_place;              // the initial membrane lies in v_store
    SpkDiv d_ppx, d_PC, d_region, d_rrrc, d_RC, d_n_patches, d_patches_img, d_patches_x;
};

struct SpkLaunch {
    StepPtrs xs;
    StepPtrs residuals;
    SpkGeom g;
    const uint16_t* wpacked;
    const float* bias;
    const void* v_start;        // initial membrane (null: zero, or in v_store: see SpkGeom::v_in_place)
    void* out;
    void* v_store;              // final membrane, and fp32 ones between the windows of a call
    float* v_scratch;           // those of a call with a 16-bit membrane, else null
    LifParams lif;
    const uint16_t* wpacked2;   // packed weight and bias of the shortcut (sc_stages > 0), else null
    const float* bias2;
    const unsigned char* lo_flags;   // SPLIT: see SpkGeom::lo_offset
    int grid;
    size_t lds_bytes;
    hipStream_t stream;
    bool dense_epilogue;  // straight-line epilogue with dense spikes (and residual): a neuron of tau 2 with a hard reset, dense tensors around it
    bool multi_window;    // ... with more than one window
    bool fast_epilogue;   // the straight-line epilogue applies: bit-packed output, no or a bit-packed residual, the usual neuron
                          // (tau 2, hard reset to 0), zero initial membrane, whole channel groups
};

template <bool F16>
__device__ __forceinline__ sk_f32x16 sk_mfma(sk_u32x4 a, sk_u32x4 b, sk_f32x16 c) {
    if constexpr (F16) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(sk_f16x8, a), __builtin_bit_cast(sk_f16x8, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(sk_bf16x8, a), __builtin_bit_cast(sk_bf16x8, b), c, 0, 0, 0);
    }
}

// The way from a kernel's start to its first requests is bound by the number of instructions and the round trips it waits for: at 512 -> 512, 7^2 x 16 it took
// 8.6 k of a launch's 43 k cycles, with a condition and a wait per quad of biases, branches around each comparison of a descriptor, divisions by 1 as a
// special case and 90 scalars of the epilogue worked out and spilled in front, and takes 5.9 k as it stands (20.6 -> 20.1 us at 64 -> 64, 56^2 x 16,
// 21.4 -> 20.1 at 512 -> 512, 7^2 x 16, 12.4 -> 11.7 at 4^2, one image, 18.5 -> 17.1 at 64 -> 128 stride 2).
// A uniform value that is computed where it stands: the compiler otherwise works out everything that depends on the kernel arguments alone ahead
// of all loops, and keeps it in (and reads it back from) lanes of vector registers.
__device__ __forceinline__ int sk_here(int x) {
    asm volatile("" : "+s"(x));
    return x;
}

// Which part of a tile's K a wave has. Waves w and w + 4 share a SIMD: the first parts, which have a stage more where the stages don't divide evenly, go
// to different SIMDs (72 -> 104 at 28^2 x 5 with a residual, five stages on four waves, 13.2 -> 11.9 us: four stages on the first SIMD and two on each of
// the others; 80 -> 128 at 20^2 x 6 9.6 -> 9.1; even splits are the same).
__device__ __forceinline__ int sk_share(int wave, int WK) { return (wave & (WK - 1)) ^ (WK < 8 && wave >= 4 ? WK >> 1 : 0); }

// Entry i of a table of pointers passed by value as a kernel argument, read from the kernel-argument segment (arguments
// start at offset 0 of that segment, in declaration order and naturally aligned): indexing the by-value struct with a
// runtime index would copy it to scratch memory.
typedef const void* sk_cvp;
typedef const __attribute__((address_space(1))) unsigned char* sk_global_bytes;
__device__ __forceinline__ const void* sk_kernarg_ptr(int table_offset_bytes, int i) {
    typedef const __attribute__((address_space(4))) unsigned char* ka_bytes;
    typedef const __attribute__((address_space(4))) sk_cvp* ka_entry;
    ka_bytes ka = (ka_bytes)__builtin_amdgcn_kernarg_segment_ptr();
    return *(ka_entry)(ka + table_offset_bytes + i * 8);
}

// The kernel's arguments as they lie in the kernel-argument segment (the order of its parameters).
struct SpkArgs {
    StepPtrs xs, residuals;
    SpkGeom g;
    const void *wpacked, *bias, *v_start, *out, *v_store;
    LifParams lif;
    const void *wpacked2, *bias2, *v_scratch, *lo_flags;
};
__device__ __forceinline__ const __attribute__((address_space(4))) SpkArgs& sk_kernarg_spk() {
    auto ka = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ka));       // (opaque: what is derived from it is computed where it is used)
    return *(const __attribute__((address_space(4))) SpkArgs*)ka;
}

// Eight spike bits -> eight 16-bit ones or zeros (ONE = the dtype's 1.0), channel j in element j. `twice` holds the byte in both halves
// (bit j at bits j and 16 + j, from one byte permutation that also drops the bytes of padding): per pair of channels one mask and one
// packed multiplication, by the 1.0 shifted down by the bit's place (both dtypes' 1.0 end in seven zero bits or more).
typedef uint16_t sk_u16x2 __attribute__((ext_vector_type(2)));
template <uint32_t ONE>
__device__ __forceinline__ sk_u32x4 sk_expand_bits(uint32_t twice) {
    static_assert((ONE & 0x7fu) == 0, "the dtype's 1.0 is shifted down by up to seven bits");
    sk_u32x4 d;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const sk_u16x2 bits = __builtin_bit_cast(sk_u16x2, twice & ((1u << (2 * k)) | (0x20000u << (2 * k))));
        const sk_u16x2 one = {static_cast<uint16_t>(ONE >> (2 * k)), static_cast<uint16_t>(ONE >> (2 * k + 1))};
        d[k] = __builtin_bit_cast(uint32_t, static_cast<sk_u16x2>(bits * one));
    }
    return d;
}

// NARROW: tiles of 32 output channels (one weight fragment) for layers of up to 32 channels and for launches of few tiles: twice the workgroups,
// each with half the matrix instructions and half the weights in its chain of steps, which is what such a launch lasts (512 -> 512 at
// 4^2, one image: 288 steps on eight waves, 19.1 -> 12.6 us; 64 -> 64 at 56^2 11.7 -> 8.7 us; of one timestep 512 -> 512 at 4^2 10.8 -> 7.5).
// MULTI: the straight-line epilogue of calls of several windows, which pass the membrane on through memory (a variant of its own: the
// loads of that membrane cost the calls of one window 3 to 5 %). 64 -> 64 at 56^2 x 16, T = 8, with a residual 70.2 -> 39.6 us against the
// general epilogue, 128 -> 128 at 20^2 x 3, T = 6 18.4 -> 14.9, 512 -> 512 at 7^2 x 7, T = 8 29.0 -> 25.0.
// IN = kSpkSteps: dense frames, one per timestep, as they are: a lane brings two neighbouring pixels of 8 channels into LDS, from eight loads of 4 bytes that hold
// one channel each (at any even address). Which calls take it instead of a launch that brings them into C8 first: see `reads_steps`.
// SPLIT (XT = float): fp32 tensors as two bf16 terms. The tile is a narrow one whose two weight fragments are the high and the low terms
// of the same 32 channels, both multiplied with the high terms of the activations; stages of the low activation terms follow where the
// tile's halo has any (spikes, averages of spikes and 8-bit pixels have none).
template <typename XT, int TT, int IN, bool SK, bool FAST, bool SC = false, bool POOL = false, bool NARROW = false, bool DENSE = false, bool MULTI = false>
__global__ __launch_bounds__(kSpkWaves * 64, 1) __attribute__((amdgpu_waves_per_eu(TT == 1 ? 4 : 2, TT == 1 ? 4 : 2))) void conv_spk_kernel(
    const StepPtrs xs, const StepPtrs residuals, const SpkGeom g, const uint16_t* __restrict__ wpacked,
    const float* __restrict__ bias, const void* __restrict__ v_start, unsigned char* __restrict__ out,
    void* __restrict__ v_store, const LifParams lif, const uint16_t* __restrict__ wpacked2, const float* __restrict__ bias2,
    float* __restrict__ v_scratch, const unsigned char* __restrict__ lo_flags) {
    extern __shared__ __align__(16) unsigned char lds[];
    // ---- every cache line of the kernel arguments is touched once, in one round trip: the compiler loads the arguments
    // where they are used, all over the prologue, and each of those loads then hits the scalar cache instead of waiting
    // for memory in turn.
    {
        auto ka = __builtin_amdgcn_kernarg_segment_ptr();
        // The explicit arguments are two step tables, the geometry, nine pointers and the neuron: the last dword that is
        // touched must lie inside them (what follows is the hidden-argument area, which the compiler may leave out).
        constexpr size_t kExplicitArgBytes = sizeof(SpkArgs);
        static_assert(0x280 + 4 <= kExplicitArgBytes && kExplicitArgBytes <= 0x2c0, "argument prefetch does not end in the last cache line of the explicit arguments");
        uint32_t d0, d1, d2, d3, d4, d5, d6, d7, d8, d9;
        asm volatile(
            "s_load_dword %0, %10, 0x40\n\ts_load_dword %1, %10, 0x80\n\ts_load_dword %2, %10, 0xc0\n\ts_load_dword %3, %10, 0x100\n\t"
            "s_load_dword %4, %10, 0x140\n\ts_load_dword %5, %10, 0x180\n\ts_load_dword %6, %10, 0x1c0\n\ts_load_dword %7, %10, 0x200\n\t"
            "s_load_dword %8, %10, 0x240\n\ts_load_dword %9, %10, 0x280\n\ts_waitcnt lgkmcnt(0)"
            : "=&s"(d0), "=&s"(d1), "=&s"(d2), "=&s"(d3), "=&s"(d4), "=&s"(d5), "=&s"(d6), "=&s"(d7), "=&s"(d8), "=&s"(d9)
            : "s"(ka));
    }
    __builtin_amdgcn_sched_barrier(0);

    static_assert(!SC || (IN == SNNF_LAYOUT_BITS && (TT == 3 || TT == 4)), "the shortcut variants take bit-packed inputs, three or four timesteps at a time");
    static_assert(!POOL || (FAST && (TT == 4 || TT == 1)), "the pooled output belongs to the straight-line epilogue of four steps");
    static_assert(IN != SNNF_LAYOUT_NCHW || (TT == 1 && !SK), "a dense input is one frame for all timesteps, of one channel group");
    constexpr bool SPLIT = std::is_same<XT, float>::value;
    static_assert(IN != kSpkSteps || DENSE, "dense frames per timestep belong to the dense epilogue");
    static_assert(!NARROW || SK || (!SC && (!POOL || IN == SNNF_LAYOUT_NCHW)), "narrow tiles of one wave: not of a shortcut, and pooled only of a dense frame");
    static_assert(!SPLIT || (NARROW && (IN == SNNF_LAYOUT_C8 || IN == kSpkSteps) && !FAST && !SC && !POOL), "fp32 tensors: narrow tiles on two C8 tensors or dense frames, dense tensors out");
    static_assert(!MULTI || (FAST && !POOL), "several windows belong to the straight-line epilogue");
    static_assert(TT <= 4 || (NARROW && SK && !SPLIT && !SC && !POOL && !MULTI), "more than four timesteps side by side: narrow tiles of 16-bit tensors whose K waves share, one window");
    static_assert(!DENSE || (IN != SNNF_LAYOUT_BITS && !FAST && !SC && !POOL), "the dense epilogue belongs to calls on dense tensors");
    // No two of the membrane arguments are the same memory: a call in place passes no v_start, and only one with a 16-bit membrane has a
    // v_scratch. (Promising nothing here instead cost the straight-line epilogue 2 %: ResNet-18, 16 images of 224x224 361 -> 369 us.)
    float* const v_out = static_cast<float*>(v_store);
    const void* const v_init = g.v_in_place ? v_store : v_start;
    float* const v_carry = g.v16 ? v_scratch : v_out;
    constexpr int NF = NARROW ? 1 : 2;         // 32-channel weight fragments of a tile
    constexpr int TG = 4 * NF;                 // channel groups of 8 of a tile
    constexpr int TL = TT > 4 ? 4 : TT;        // timesteps whose activations a matrix step holds at a time
    // A dense frame with dense spikes is computed in the form of the matrix kernel (which takes other neurons, and frames per timestep of whole tiles): the bias
    // behind the sums, the charge as v + (x - v) / 2. One frame T times and T equal frames then have the same bits where that kernel also adds a sum's products in this
    // order (3 -> 64 3x3 at 32^2, 7x7 stride 2 at 224^2 x 16). On other channels and kernels (8 -> 64, 1 -> 64 5x5), and where equal frames take the copy route, whose sums
    // start from the bias (3 -> 64 at 33^2), they differ in a membrane's last bits where sums round.
    constexpr bool LATE_BIAS = DENSE && IN == SNNF_LAYOUT_NCHW;
    constexpr bool F16 = dtype_of<XT>::value == SNNF_F16;
    constexpr uint32_t ONE = F16 ? 0x3c00u : 0x3f80u;
    constexpr int kResTable = static_cast<int>(sizeof(StepPtrs));
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int half = lane >> 5;
    const int l32 = lane & 31;
    unsigned char* const wlds = lds + kSpkHeaderBytes + wave * g.lds_wave_bytes;
    const int region16 = g.region * 16;        // bytes of one channel group of the halo
    constexpr int PAIR = IN == kSpkSteps ? 2 : 1;          // items that a lane stages at a time: neighbours in a halo row (whose length is even)
    const int tile_t = g.G * region16 + 16 * PAIR;    // bytes of one timestep's stage: its items and dummy ones that absorb the writes of idle staging slots

    const int WK = SK ? (1 << g.wk_log2) : 1;
    const int wk = SK ? sk_share(wave, WK) : 0;
    const int tile_in_block = SK ? (wave >> g.wk_log2) : wave;
    const int tiles_per_block = SK ? (kSpkWaves >> g.wk_log2) : kSpkWaves;
    const int nsteps_t = g.shared_x ? 1 : g.T;          // timesteps with a convolution of their own
    const int hg = g.tap_pairs ? 1 : (g.G >> 1);        // k-slot pairs per tap and stage
    const int nst = g.tap_pairs ? g.npairs : g.taps * hg;   // matrix steps per stage

    // ---- step table of the workgroup: for step i of a stage, the byte offset of its weight fragments from the stage's
    // first pair and the LDS offset of its activations (tap and channel group of the half's k-slot), once for the lower and
    // once for the upper half of a wave: a lane reads the 8 bytes of its half. The matrix loop then needs no index
    // arithmetic. Steps beyond the last repeat it (prefetch only).
    {
        sk_u32x4* __restrict__ table = reinterpret_cast<sk_u32x4*>(lds);
        const int tid_t = tid - 7 * 64;          // (at most 64 entries)
        if (tid_t >= 0 && tid_t < nst + 4) {
            const int i = min(tid_t, nst - 1);
            sk_u32x4 e;
            if (g.tap_pairs) {
                const int tap0 = 2 * i, tap1 = min(2 * i + 1, g.taps - 1);   // an odd tap count leaves the last k-slot empty (zero weights)
                const int kh0 = (tap0 * g.kw_mul) >> 16, kh1 = (tap1 * g.kw_mul) >> 16;
                e[0] = static_cast<uint32_t>(i * kFragBytes);
                e[1] = static_cast<uint32_t>((kh0 * g.RC + (tap0 - kh0 * g.KW)) * 16);
                e[3] = static_cast<uint32_t>((kh1 * g.RC + (tap1 - kh1 * g.KW)) * 16);
            } else {
                const int tap = i >> g.hg_log2;
                const int gp = i & (hg - 1);
                const int kh = (tap * g.kw_mul) >> 16;
                const int tapoff = (kh * g.RC + (tap - kh * g.KW)) * 16;
                e[0] = static_cast<uint32_t>((tap * g.pair_tap_stride + gp) * kFragBytes);
                e[1] = static_cast<uint32_t>(tapoff + (2 * gp) * region16);
                e[3] = static_cast<uint32_t>(tapoff + (2 * gp + 1) * region16);
            }
            e[2] = e[0];
            table[tid_t] = e;
        }
        if constexpr (SC) {
            // The shortcut's stages: one tap, the centre of the main kernel (the lane's own pixel), on the same halo; entries
            // behind the main table's.
            const int i2 = tid_t - (nst + 4);
            if (i2 >= 0 && i2 < hg + 4) {
                const int gp = min(i2, hg - 1);
                const int tapoff = (g.ph * g.RC + g.pw) * 16;
                sk_u32x4 e;
                e[0] = static_cast<uint32_t>(gp * kFragBytes);
                e[1] = static_cast<uint32_t>(tapoff + (2 * gp) * region16);
                e[2] = e[0];
                e[3] = static_cast<uint32_t>(tapoff + (2 * gp + 1) * region16);
                table[tid_t] = e;
            }
        }
        // ---- staging descriptors of the workgroup: item e of a timestep's stage = (channel group gq, image ii, halo row r, halo
        // column c); its element offset from the stage's first item and the four coordinates, packed. Built once; the staging
        // of every stage of every tile reads them back instead of dividing (three divisions per item otherwise). Items beyond
        // the stage carry channel group 255, which no stage has.
        Pack<uint32_t, 2>* __restrict__ desc_w = reinterpret_cast<Pack<uint32_t, 2>*>(lds + kSpkTableBytes);
        for (int e = tid; e < kSpkDescs; e += kSpkWaves * 64) {
            Pack<uint32_t, 2> d;
            d.v[0] = 0u;
            d.v[1] = 0xff000000u;
            if (e * PAIR < g.IT) {
                const int gq = sk_div(e * PAIR, g.d_region);
                const int rem = e * PAIR - gq * g.region;
                const int ii = sk_div(rem, g.d_rrrc);
                const int rem2 = rem - ii * (g.RR * g.RC);
                const int r = sk_div(rem2, g.d_RC);
                const int c = rem2 - r * g.RC;
                if constexpr (IN == SNNF_LAYOUT_NCHW || IN == kSpkSteps) d.v[0] = static_cast<uint32_t>(((ii * g.Cin + gq * 8) * g.H + r) * g.W + c);   // elements of a dense frame
                else d.v[0] = static_cast<uint32_t>(((ii * g.C8in + gq) * g.H + r) * g.W + c);
                d.v[1] = static_cast<uint32_t>(r) | (static_cast<uint32_t>(c) << 8) | (static_cast<uint32_t>(ii) << 16) | (static_cast<uint32_t>(gq) << 24);
            }
            desc_w[e] = d;
        }
        // ---- where pixel p of a tile sits inside the patch: image, row and column, packed. Every item reads its lane's entry
        // back: kept in registers these values would live (or be spilled) across the matrix loop of every variant.
        // (Built by the sixth wave and the step table by the eighth: the first ones have the descriptors of a usual stage.)
        if (tid >= 5 * 64 && tid < 5 * 64 + 32) {
            const int p32 = tid - 5 * 64;
            const int ppx = g.PR * g.PC;
            const int pi = sk_div(p32, g.d_ppx);
            const int prem = p32 - pi * ppx;
            const int prow = sk_div(prem, g.d_PC);
            const int pcol = prem - prow * g.PC;
            Pack<uint32_t, 2> e;
            e.v[0] = static_cast<uint32_t>(pi) | (static_cast<uint32_t>(prow) << 8) | (static_cast<uint32_t>(pcol) << 16);
            e.v[1] = pi < g.PI ? static_cast<uint32_t>(((pi * g.RR + prow * g.sh) * g.RC + pcol * g.sw) * 16) : 0u;
            reinterpret_cast<Pack<uint32_t, 2>*>(lds + kSpkTableBytes + kSpkDescBytes)[p32] = e;
        }
        __syncthreads();
    }
    const Pack<uint32_t, 2>* __restrict__ desc = reinterpret_cast<const Pack<uint32_t, 2>*>(lds + kSpkTableBytes);
    const Pack<uint32_t, 2>* __restrict__ table = reinterpret_cast<const Pack<uint32_t, 2>*>(lds + 8 * half);   // entry i of this half: table[2 * i]

    // Workgroups are handed to the eight XCDs in turn (workgroup b runs on XCD b % 8) and every XCD has an L2 of its own.
    // Items are ordered output-channel tile first, so the workgroups of one XCD take a contiguous range of them: an XCD then
    // reads the weights of few output-channel tiles (one, for a 512-channel layer) instead of the whole tensor.
    const int nb = g.grid;
    const int xcd = static_cast<int>(blockIdx.x) & 7;
    const int block_l = xcd * (nb >> 3) + min(xcd, nb & 7) + (static_cast<int>(blockIdx.x) >> 3);
    for (int it = 0; it < g.iters; ++it) {
        // Consecutive items go to different workgroups, so that a layer with fewer items than wave slots still uses every compute unit.
        const int item = (it * tiles_per_block + tile_in_block) * nb + block_l;
        const bool have = item < g.n_items;
        const int item_c = have ? item : 0;
        const int oc_tile = sk_div(item_c, g.d_n_patches);
        const int patch = item_c - oc_tile * g.n_patches;
        const int imgg = sk_div(patch, g.d_patches_img);
        const int prem_i = patch - imgg * g.patches_img;
        const int py = sk_div(prem_i, g.d_patches_x);
        const int n0 = imgg * g.PI;
        const int oh0 = py * g.PR;
        const int ow0 = (prem_i - py * g.patches_x) * g.PC;
        const int ih_lo = oh0 * g.sh - g.ph;
        const int iw_lo = ow0 * g.sw - g.pw;

        const int ocf0 = oc_tile * NF;
        // With K split over waves, every wave finishes a part of the tile's eight quads, which its accumulators hold in the same registers
        // whatever the wave: the upper half of the waves computes the two 32-channel fragments in swapped places, and the lanes
        // read the weight rows of a fragment with the quads exchanged (quad q of the accumulators is quad q ^ quad_x of the fragment).
        const int swap_f = SK && !NARROW ? wk >> (g.wk_log2 - 1) : 0;
        const int quad_x = SK && !NARROW ? (wk << (3 - g.wk_log2)) & 3 : 0;      // (eight waves: wk & 3, four: 2 (wk & 1), two: 0)
        const int64_t w_frag0 = min(ocf0 + swap_f, g.nocf - 1);
        const int64_t w_frag1 = min(ocf0 + 1 - swap_f, g.nocf - 1);

        for (int t0 = 0; t0 < nsteps_t; t0 += TT) {
            // (Defined here, as anything: what is first written under a condition inside a loop is otherwise carried around all loops by the compiler,
            // 128 registers that are never read again through the whole epilogue.)
            sk_f32x16 acc[TT][NF];
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int f = 0; f < NF; ++f) asm("" : "=v"(acc[t][f]));
            // One LDS stage: G channel groups of the patch's halo for TT timesteps, from global memory into this wave's region.
            // Item e = slot * 64 + lane of a timestep = (group, image, row, column) of the halo; its LDS address is 16 e. Items
            // are decoded on the fly (nothing about them is kept in registers across the matrix loop) and move in batches of 4
            // slots x TT timesteps: all loads of a batch are in flight together.
            // PRE (bit-packed inputs, lean epilogue): the first batch of the NEXT stage is requested before the matrix steps of the
            // current one and sits in registers meanwhile, so that its latency hides behind them.
            constexpr bool PRE = FAST && IN == SNNF_LAYOUT_BITS;
            int nstages_all = SC ? g.nstages + g.sc_stages : g.nstages;
            uint64_t low_groups = 0;             // SPLIT: which stages of low terms run (below)
            // The first stage of low terms; of dense frames a wave's own follow its own, so that what it found decides.
            const int low_first = SPLIT && IN == kSpkSteps && SK ? ((g.nstages + (1 << g.wk_log2) - 1) >> g.wk_log2) << g.wk_log2 : g.nstages;
            uint32_t pre_raw[TT][4];
            uint32_t pre_ok = 0;
            // Decodes the 4 items of batch jb of stage s from the workgroup's descriptors: their global index (0 when they are
            // padding) and a flag nibble (bit j: real data).
            // A stage at or beyond g.nstages (SC only) is one of the shortcut's: same halo items, taken from the second input at
            // the sampled positions.
            auto batch_decode = [&](int s, int jb, int lane_s, uint32_t (&idx)[4]) __attribute__((always_inline)) -> uint32_t {
                const bool second = SC && s >= g.nstages;
                const int gg0 = ((SC || SPLIT) && s >= g.nstages ? s - g.nstages : s) * g.G;
                const int c8 = second ? g.sc_C8 : g.C8in;
                const int base_u = second ? ((n0 * g.sc_C8 + gg0) * g.sc_H + ih_lo * g.sc_sh) * g.sc_W + iw_lo * g.sc_sw
                                   : IN == SNNF_LAYOUT_NCHW ? ((n0 * g.Cin + gg0 * 8) * g.H + ih_lo) * g.W + iw_lo
                                          : ((n0 * g.C8in + gg0) * g.H + ih_lo) * g.W + iw_lo;   // may be negative; only added to in-image items
                uint32_t ok_bits = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const Pack<uint32_t, 2> d = desc[(jb + j) * 64 + lane_s];
                    const int r = static_cast<int>(d.v[1] & 255u), c = static_cast<int>((d.v[1] >> 8) & 255u);
                    const int ii = static_cast<int>((d.v[1] >> 16) & 255u), gq = static_cast<int>(d.v[1] >> 24);
                    // (& and not &&: a branch around each comparison waits for each descriptor in turn)
                    const bool ok = static_cast<bool>(static_cast<int>(n0 + ii < g.N) & static_cast<int>(gg0 + gq < c8) &
                                                      static_cast<int>(static_cast<unsigned>(ih_lo + r) < static_cast<unsigned>(g.H)) &
                                                      static_cast<int>(static_cast<unsigned>(iw_lo + c) < static_cast<unsigned>(g.W)));
                    int off = static_cast<int>(d.v[0]);
                    if constexpr (SC) {
                        if (second) off = ((ii * g.sc_C8 + gq) * g.sc_H + r * g.sc_sh) * g.sc_W + c * g.sc_sw;
                    }
                    idx[j] = ok ? static_cast<uint32_t>(base_u + off) : 0u;
                    ok_bits |= ok ? (1u << j) : 0u;
                }
                return ok_bits;
            };
            auto batch_load_bits = [&](int s, const uint32_t (&idx)[4], uint32_t (&raw)[TT][4]) __attribute__((always_inline)) {
                const int ptr_table = SC && s >= g.nstages ? kResTable : 0;
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const int ts = t0 + t < nsteps_t ? t0 + t : t0;   // steps beyond T repeat the window's first and are never stored
                    const sk_global_bytes src = (sk_global_bytes)sk_kernarg_ptr(ptr_table, ts);
#pragma unroll
                    for (int j = 0; j < 4; ++j) raw[t][j] = src[idx[j]];
                }
            };
            auto batch_put_bits = [&](int jb, int lane_s, uint32_t ok_bits, const uint32_t (&raw)[TT][4]) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t keep = ((ok_bits >> j) & 1u) ? 0x0c000c00u : 0x0c0c0c0cu;   // v_perm: byte 0 at bytes 0 and 2, or zeros
                    // every slot writes: an item beyond the stage goes to the timestep's dummy item
                    unsigned char* const item = wlds + min((jb + j) * 64 + lane_s, g.IT) * 16;
#pragma unroll
                    for (int t = 0; t < TT; ++t) *reinterpret_cast<sk_u32x4*>(item + t * tile_t) = sk_expand_bits<ONE>(__builtin_amdgcn_perm(raw[t][j], raw[t][j], keep));
                }
            };
            // Requests the first batch of stage s (PRE only).
            auto stage_req = [&](int s) __attribute__((always_inline)) {
                int lane_s = lane;
                asm volatile("" : "+v"(lane_s));
                uint32_t idx[4];
                pre_ok = batch_decode(s, 0, lane_s, idx);
                batch_load_bits(s, idx, pre_raw);
            };
            // One LDS stage: G channel groups of the patch's halo for TT timesteps, from global memory into this wave's region.
            // Item e = slot * 64 + lane of a timestep = (group, image, row, column) of the halo; its LDS address is 16 e. Items
            // are decoded on the fly (nothing about them is kept in registers across the matrix loop) and move in batches of 4
            // slots x TT timesteps: all loads of a batch are in flight together.
            // ... of dense frames: all timesteps of 64 pairs of items together.
            // (fp32: the high bf16 terms, or the low ones; whether any item has one is the answer.)
            auto stage_pairs = [&](int gg0, bool low_terms, int lane_s) __attribute__((always_inline)) -> bool {
                const int plane = g.H * g.W;
                uint32_t any = 0;
                const int base_u = ((n0 * g.Cin + gg0 * 8) * g.H + ih_lo) * g.W + iw_lo;
#pragma unroll
                for (int jb = 0; jb < kSpkSlots / 2; ++jb) {
                    if (jb < sk_here(g.JT)) {
                        const Pack<uint32_t, 2> d = desc[jb * 64 + lane_s];
                        const int r = static_cast<int>(d.v[1] & 255u), c = iw_lo + static_cast<int>((d.v[1] >> 8) & 255u);
                        const int ii = static_cast<int>((d.v[1] >> 16) & 255u), gq = static_cast<int>(d.v[1] >> 24);
                        const bool ok = static_cast<bool>(static_cast<int>(n0 + ii < g.N) & static_cast<int>(gg0 + gq < g.C8in) &
                                                          static_cast<int>(static_cast<unsigned>(ih_lo + r) < static_cast<unsigned>(g.H)));
                        const bool in0 = ok & (static_cast<unsigned>(c) < static_cast<unsigned>(g.W)), in1 = ok & (static_cast<unsigned>(c + 1) < static_cast<unsigned>(g.W));
                        // A pair of which one pixel lies in the image is read with that pixel's other neighbour (rows have at least two).
                        const uint32_t off = in0 || in1 ? static_cast<uint32_t>(base_u + static_cast<int>(d.v[0]) + (in0 ? (in1 ? 0 : -1) : 1)) : 0u;
                        constexpr uint32_t kLow = 0x05040100u, kHigh = 0x07060302u, kNone = 0x0c0c0c0cu;     // v_perm: the low or the high halves of two words
                        const uint32_t sel0 = in0 ? (in1 ? kLow : kHigh) : kNone, sel1 = in1 ? (in0 ? kHigh : kLow) : kNone;
                        const int left = in0 || in1 ? g.Cin - (gg0 + gq) * 8 : g.Cin;    // channels of this group, and beyond (of the first one where there is no pixel)
                        unsigned char* const item = wlds + min((jb * 64 + lane_s) * 2, g.IT) * 16;
                        if constexpr (SPLIT) {
                            struct __attribute__((packed, aligned(4))) Two { float v[2]; };
                            const bool take0 = in0 && !in1, take1 = in0 && in1;      // which of the two values is the first pixel's second, and the second one's
                            Two raw[TT][8];
#pragma unroll
                            for (int t = 0; t < TT; ++t) {
                                const float* __restrict__ src = static_cast<const float*>(sk_kernarg_ptr(0, t0 + t < nsteps_t ? t0 + t : t0));
#pragma unroll
                                for (int k = 0; k < 8; ++k) raw[t][k] = *reinterpret_cast<const Two*>(src + (off + static_cast<uint32_t>(min(k, left - 1) * plane)));
                            }
#pragma unroll
                            for (int t = 0; t < TT; ++t) {
                                sk_u32x4 a, b;
#pragma unroll
                                for (int k = 0; k < 4; ++k) {
                                    float f0[2], f1[2];
#pragma unroll
                                    for (int i = 0; i < 2; ++i) {
                                        const Two& two = raw[t][2 * k + i];
                                        const bool here = 2 * k + i < left;
                                        f0[i] = in0 && here ? (take0 ? two.v[1] : two.v[0]) : 0.0f;
                                        f1[i] = in1 && here ? (take1 ? two.v[1] : two.v[0]) : 0.0f;
                                    }
                                    uint32_t hi0, lo0, hi1, lo1;
                                    split_bf16_pair(f0[0], f0[1], hi0, lo0);
                                    split_bf16_pair(f1[0], f1[1], hi1, lo1);
                                    any |= (lo0 | lo1) & 0x7fff7fffu;
                                    a[k] = low_terms ? lo0 : hi0;
                                    b[k] = low_terms ? lo1 : hi1;
                                }
                                *reinterpret_cast<sk_u32x4*>(item + t * tile_t) = a;
                                *reinterpret_cast<sk_u32x4*>(item + t * tile_t + 16) = b;
                            }
                            continue;
                        }
                        struct __attribute__((packed, aligned(2))) Word { uint32_t v; };
                        uint32_t raw[TT][8];
                        if (g.Cin & 7) {
#pragma unroll
                            for (int t = 0; t < TT; ++t) {
                                const uint16_t* __restrict__ src = static_cast<const uint16_t*>(sk_kernarg_ptr(0, t0 + t < nsteps_t ? t0 + t : t0));
#pragma unroll
                                for (int k = 0; k < 8; ++k) raw[t][k] = reinterpret_cast<const Word*>(src + (off + static_cast<uint32_t>(min(k, left - 1) * plane)))->v;
                            }
#pragma unroll
                            for (int t = 0; t < TT; ++t)
#pragma unroll
                                for (int k = 0; k < 8; ++k) raw[t][k] = k < left ? raw[t][k] : 0u;
                        } else {
#pragma unroll
                            for (int t = 0; t < TT; ++t) {
                                const uint16_t* __restrict__ src = static_cast<const uint16_t*>(sk_kernarg_ptr(0, t0 + t < nsteps_t ? t0 + t : t0));
#pragma unroll
                                for (int k = 0; k < 8; ++k) raw[t][k] = reinterpret_cast<const Word*>(src + (off + static_cast<uint32_t>(k * plane)))->v;
                            }
                        }
#pragma unroll
                        for (int t = 0; t < TT; ++t) {
                            sk_u32x4 a, b;
#pragma unroll
                            for (int k = 0; k < 4; ++k) {
                                a[k] = __builtin_amdgcn_perm(raw[t][2 * k + 1], raw[t][2 * k], sel0);
                                b[k] = __builtin_amdgcn_perm(raw[t][2 * k + 1], raw[t][2 * k], sel1);
                            }
                            *reinterpret_cast<sk_u32x4*>(item + t * tile_t) = a;
                            *reinterpret_cast<sk_u32x4*>(item + t * tile_t + 16) = b;
                        }
                    }
                }
                return __ballot(any != 0u) != 0ull;
            };
            auto stage_in = [&](int s) __attribute__((always_inline)) {
                __builtin_amdgcn_wave_barrier();   // the matrix steps of the previous stage have read their operands
                int lane_s = lane;                 // opaque: the decode below stays here instead of being hoisted out of every loop
                asm volatile("" : "+v"(lane_s));   // (its results would sit in registers, or in scratch memory, across the matrix loop)
                if constexpr (IN == kSpkSteps) {
                    const bool low_terms = SPLIT && s >= low_first;
                    const int at = low_terms ? s - low_first : s;
                    if (stage_pairs(at * g.G, low_terms, lane_s) && !low_terms) {
                        low_groups |= 1ull << (at & 63);
                        nstages_all = 2 * low_first;
                    }
                } else {
#pragma unroll
                for (int jb = 0; jb < kSpkSlots; jb += 4) {
                    if (jb < sk_here(g.JT)) {
                        if constexpr (PRE) {
                            if (jb == 0) {
                                batch_put_bits(0, lane_s, pre_ok, pre_raw);
                                continue;
                            }
                        }
                        uint32_t idx[4];
                        const uint32_t ok_bits = batch_decode(s, jb, lane_s, idx);
                        if constexpr (IN == SNNF_LAYOUT_BITS) {
                            uint32_t raw[TT][4];
                            batch_load_bits(s, idx, raw);
                            batch_put_bits(jb, lane_s, ok_bits, raw);
                        } else if constexpr (IN == SNNF_LAYOUT_NCHW) {
                            // A dense frame of at most 8 channels (the network's input): one 16-bit load per channel and item.
                            const int plane = g.H * g.W;
#pragma unroll
                            for (int t = 0; t < TT; ++t) {
                                const int ts = t0 + t < nsteps_t ? t0 + t : t0;
                                const uint16_t* __restrict__ src = static_cast<const uint16_t*>(sk_kernarg_ptr(0, ts));
                                uint32_t h[4][8];
#pragma unroll
                                for (int k = 0; k < 8; ++k) {
                                    if (k < g.Cin) {
#pragma unroll
                                        for (int j = 0; j < 4; ++j) h[j][k] = src[idx[j] + static_cast<uint32_t>(k * plane)];
                                    } else {
#pragma unroll
                                        for (int j = 0; j < 4; ++j) h[j][k] = 0u;
                                    }
                                }
#pragma unroll
                                for (int j = 0; j < 4; ++j) {
                                    sk_u32x4 d;
#pragma unroll
                                    for (int k = 0; k < 4; ++k) d[k] = ((ok_bits >> j) & 1u) ? (h[j][2 * k] | (h[j][2 * k + 1] << 16)) : 0u;
                                    *reinterpret_cast<sk_u32x4*>(wlds + t * tile_t + min((jb + j) * 64 + lane_s, g.IT) * 16) = d;
                                }
                            }
                        } else {
#pragma unroll
                            for (int t = 0; t < TT; ++t) {
                                const int ts = t0 + t < nsteps_t ? t0 + t : t0;
                                const unsigned char* __restrict__ src = static_cast<const unsigned char*>(sk_kernarg_ptr(0, ts));
                                uint32_t ok_t = ok_bits;
                                if constexpr (SPLIT) {
                                    if (s >= g.nstages) {   // low terms: items without any were not written
                                        src += g.lo_offset;
                                        const unsigned char* __restrict__ flags_t = lo_flags + static_cast<int64_t>(ts) * g.flag_stride;
#pragma unroll
                                        for (int j = 0; j < 4; ++j)
                                            if (flags_t[idx[j] >> 6] == 0) ok_t &= ~(1u << j);
                                    }
                                }
                                sk_u32x4 raw[4];
#pragma unroll
                                for (int j = 0; j < 4; ++j) raw[j] = *reinterpret_cast<const sk_u32x4*>(src + idx[j] * 16u);
#pragma unroll
                                for (int j = 0; j < 4; ++j) {
                                    sk_u32x4 d;
#pragma unroll
                                    for (int k = 0; k < 4; ++k) d[k] = ((ok_t >> j) & 1u) ? raw[j][k] : 0u;
                                    *reinterpret_cast<sk_u32x4*>(wlds + t * tile_t + min((jb + j) * 64 + lane_s, g.IT) * 16) = d;
                                }
                            }
                        }
                    }
                }
                }
                __builtin_amdgcn_wave_barrier();   // LDS serves a wave's accesses in order: the reads below see these writes
            };

            // ---- matrix loop over this wave's stages. Step = one pair of k-slots = one matrix instruction per (timestep,
            // 32-channel fragment). Per stage: the first weight fragments are requested from L2, the stage is brought into LDS,
            // then the steps run four at a time without a branch: weight fragments three steps ahead through four register
            // sets, activation fragments one step ahead through two.
            const int s_first = SK ? wk : 0;
            const int s_step = SK ? WK : 1;
            // SPLIT: stages of low terms only where the tile's halo has any in this window: bit c8 & 63 of `low_groups` says that channel group
            // c8 has one in the rows of the halo. A lane reads the flags of one group, RR W / 64 of them and one more; the groups of whole
            // images (tiles of several, at most 32 pixels a group) are one short range of flags and run all their low stages or none.
            // Reading whole images for every tile, and running all low stages of an image for one low term in it, took 64 -> 64 at 224^2 114 us
            // without low terms (here 69) and 147 with a single one (76), 512 -> 512 at 112^2 722 (575) and 1231 (579), 64 -> 8 as 1x1 at
            // 640^2, one timestep, 156 (54); 64 -> 64 at 32^2 x 8 is the same, 20 us.
            // Of dense frames a wave finds the low terms of a stage as it brings in the high ones, and runs those of its own stages behind them: bit s & 63 is stage s.
            if constexpr (SPLIT && IN != kSpkSteps) {
                const int plane = g.H * g.W;
                const bool images = g.PI > 1;
                const int r0 = images ? 0 : max(ih_lo, 0);
                const int items = images ? min(g.PI, g.N - n0) * g.C8in * plane : (min(ih_lo + g.RR, g.H) - r0) * g.W;
                const int dwords = ((items - 1) >> 8) + 2;                       // of four flags, 256 items; that many at most
                for (int c0 = 0; c0 < (images ? 1 : g.C8in); c0 += 64) {
                    const bool mine = images || c0 + lane < g.C8in;
                    const int first = ((n0 * g.C8in + (!images && mine ? c0 + lane : 0)) * g.H + r0) * g.W, last = first + items - 1;
                    const int w0 = first >> 8, w1 = last >> 8;
                    uint32_t any = 0;
                    for (int d = images ? lane : 0; d < dwords; d += images ? 64 : 1) {
                        const int w = min(w0 + d, w1);
                        const uint32_t mask = (w == w0 ? ~0u << ((first >> 6 & 3) * 8) : ~0u) & (w == w1 ? ~0u >> ((3 - (last >> 6 & 3)) * 8) : ~0u);
#pragma unroll
                        for (int t = 0; t < TT; ++t)
                            any |= reinterpret_cast<const uint32_t*>(lo_flags + static_cast<int64_t>(min(t0 + t, nsteps_t - 1)) * g.flag_stride)[w] & mask;
                    }
                    low_groups |= __ballot(mine && any != 0u);
                }
                if (images && low_groups != 0) low_groups = ~0ull;
                if (low_groups != 0) nstages_all = 2 * g.nstages;
            }
            if constexpr (PRE) {
                stage_req(s_first);      // (there is one for every wave; one without a tile reads the first tile's)
            }
            // The accumulators start from the bias: register 4 q + k of fragment f is channel 64 oc_tile + 32 f + 8 q + 4 half + k. With K
            // split over waves only the first one adds it; the others read the zeros behind it. One value per lane is requested here, right
            // behind the first stage's activations, and goes through the wave's region of LDS ahead of that stage.
            const int first_bias = ((!SK || wk == 0) ? oc_tile * (32 * NF) : ((g.nocf + 1) >> 1) * 64) + (NARROW ? l32 : lane);
            float bias_lane = bias[first_bias];
            float bias2_lane = 0.0f;
            if constexpr (SC) bias2_lane = bias2[first_bias];
            // ---- this lane's output pixel, and where its top-left input sits in the staged halo.
            int lane_l = l32;
            asm volatile("" : "+v"(lane_l));
            const Pack<uint32_t, 2> lane_pos = reinterpret_cast<const Pack<uint32_t, 2>*>(lds + kSpkTableBytes + kSpkDescBytes)[lane_l];
            const uint32_t lane_b = lane_pos.v[1];
            // The epilogue's view of the tile's channel block, opaque from here on: the scalar arithmetic that depends on it
            // (per-quad base addresses and store predicates, several hundred scalar instructions that the compiler computes
            // ahead of time) then runs after the tile's first loads have been requested, under their latency, instead of in
            // front of them.
            int oc_e = oc_tile;
            asm volatile("" : "+s"(oc_e));
            auto park_bias = [&]() __attribute__((always_inline)) {
                if constexpr (LATE_BIAS) {
#pragma unroll
                    for (int f = 0; f < NF; ++f)
#pragma unroll
                        for (int k = 0; k < 16; ++k) acc[0][f][k] = 0.0f;
                    return;
                }
                if constexpr (SC) bias_lane += bias2_lane;
                reinterpret_cast<float*>(wlds)[lane] = bias_lane;
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int f = 0; f < NF; ++f)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const sk_f32x4 b4 = *reinterpret_cast<const sk_f32x4*>(wlds + (f * 32 + q * 8 + 4 * half) * 4);
#pragma unroll
                        for (int k = 0; k < 4; ++k) acc[0][f][4 * q + k] = b4[k];
                    }
            };
            auto start_sums = [&]() __attribute__((always_inline)) {
#pragma unroll
                for (int t = 1; t < TT; ++t)
#pragma unroll
                    for (int f = 0; f < NF; ++f) acc[t][f] = acc[0][f];
            };
            // Waves of several tiles take turns of one tile each: half a tile out of step, one's epilogue runs under the other's matrix instructions, and
            // both end together (the older wave ahead all the way, the other one's last tile ran alone: 256 -> 256 at 14^2 x 128 97.1 -> 95.9 us,
            // 128 -> 128 at 28^2 x 128 101.1 -> 98.0, 64 -> 64 at 56^2 x 128 96.0 -> 95.7; turns of a stage each kept the two in step and lost 2 % there).
            if (!SK && g.iters > 1) {
                if (wave >= 4) __builtin_amdgcn_s_setprio(2);
                else if (it & 1) __builtin_amdgcn_s_setprio(1);
                else __builtin_amdgcn_s_setprio(3);
            }
            if (have) {
                const uint32_t lane16 = static_cast<uint32_t>(lane ^ (quad_x * 8)) * 16u;
                const unsigned char* __restrict__ bl = wlds + lane_b;
#pragma clang loop unroll(disable)
                for (int stage = s_first; stage < nstages_all; stage += s_step) {
                    const bool second = SC && stage >= g.nstages;     // a stage of the shortcut
                    const bool low = SPLIT && stage >= low_first;     // a stage of low activation terms: against the high weight terms alone
                    const int gg0 = (second ? stage - g.nstages : low ? stage - low_first : stage) * g.G;
                    if constexpr (SPLIT && IN == kSpkSteps) {
                        // (The waves' shares are of one length here: the last round of stages may have none for a wave.)
                        if (gg0 >= g.nstages * g.G || (low && (low_groups >> ((stage - low_first) & 63) & 1ull) == 0)) continue;
                    } else if (SPLIT && low && (low_groups >> (gg0 & 63) & ((1ull << g.G) - 1)) == 0) {
                        continue;
                    }
                    const int gpc_l2 = second ? g.sc_gpc_log2 : g.gpc_log2;
                    const int chunk = gg0 >> gpc_l2;
                    const int pbase = chunk * (second ? g.sc_npairs : g.npairs) + ((gg0 - (chunk << gpc_l2)) >> 1);   // pair of (tap 0, the stage's first two groups)
                    const uint16_t* __restrict__ wp = second ? wpacked2 : wpacked;
                    const int64_t fs = second ? g.sc_frag_stride : g.frag_stride;
                    const unsigned char* __restrict__ pa0 = reinterpret_cast<const unsigned char*>(wp + w_frag0 * fs + static_cast<int64_t>(pbase) * (kFragBytes / 2));
                    const unsigned char* __restrict__ pa1 = reinterpret_cast<const unsigned char*>(wp + (SPLIT ? w_frag0 * fs + g.w_lo_offset : w_frag1 * fs) + static_cast<int64_t>(pbase) * (kFragBytes / 2));
                    const Pack<uint32_t, 2>* __restrict__ tb = second ? table + 2 * (nst + 4) : table;
                    const int nst_s = second ? hg : nst;
                    constexpr int WF = SPLIT ? 2 : NF;    // weight fragments of a step: two of 32 channels, or the two terms of one
                    sk_u32x4 wa[4][WF];
                    sk_u32x4 wb[2][TL];
                    uint32_t bo[4];
                    // Requests the weight fragments of the step described by table entry `e` and notes where its activations are.
                    auto req_a = [&](int slot, const Pack<uint32_t, 2>& e) __attribute__((always_inline)) {
                        const uint32_t voff = lane16 + e.v[0];
                        wa[slot][0] = *reinterpret_cast<const sk_u32x4*>(pa0 + voff);
                        if constexpr (WF == 2) wa[slot][1] = *reinterpret_cast<const sk_u32x4*>(pa1 + voff);
                        bo[slot] = e.v[1];
                    };
                    auto read_b = [&](int slot, uint32_t boff) __attribute__((always_inline)) {
#pragma unroll
                        for (int t = 0; t < TL; ++t) wb[slot][t] = *reinterpret_cast<const sk_u32x4*>(bl + boff + t * tile_t);
                    };
                    auto mma = [&](int sa, int sb) __attribute__((always_inline)) {
#pragma unroll
                        for (int t = 0; t < TL; ++t) {
                            acc[t][0] = sk_mfma<F16>(wa[sa][0], wb[sb][t], acc[t][0]);
                            if constexpr (!NARROW) acc[t][1] = sk_mfma<F16>(wa[sa][1], wb[sb][t], acc[t][1]);
                        }
                        if constexpr (SPLIT) {
                            if (!low) {
#pragma unroll
                                for (int t = 0; t < TT; ++t) acc[t][0] = sk_mfma<F16>(wa[sa][1], wb[sb][t], acc[t][0]);
                            }
                        }
                    };
                    // The timesteps from the fifth on (TT > 4): a matrix step's second half, against the same weights.
                    auto read_b_late = [&](int slot, uint32_t boff) __attribute__((always_inline)) {
#pragma unroll
                        for (int t = TL; t < TT; ++t) wb[slot][t - TL] = *reinterpret_cast<const sk_u32x4*>(bl + boff + t * tile_t);
                    };
                    auto mma_late = [&](int sa, int sb) __attribute__((always_inline)) {
#pragma unroll
                        for (int t = TL; t < TT; ++t) acc[t][0] = sk_mfma<F16>(wa[sa][0], wb[sb][t - TL], acc[t][0]);
                    };
                    req_a(0, tb[0]);
                    req_a(1, tb[2]);
                    req_a(2, tb[4]);
                    Pack<uint32_t, 2> ent = tb[6];       // entry of the step whose weights are requested next
                    if (stage == s_first) park_bias();
                    stage_in(stage);
                    if (stage == s_first) start_sums();
                    if constexpr (PRE) {
                        if (stage + s_step < nstages_all) stage_req(stage + s_step);
                    }
                    read_b(0, bo[0]);
                    // The two waves of a SIMD (w and w + 4) share its matrix cores, and at equal priority the older one wins every instruction: it ran
                    // through all its stages, and then the other one through its own, with nothing under either's staging. So a wave on its last stage
                    // gives way to one that is not (128 -> 128 at 28^2 x 16, two stages per wave, 18.1 -> 17.6 us, 512 -> 512 at 7^2 x 16 18.7 -> 18.3, 64 -> 128 stride 2 at
                    // 56^2 x 16 16.1 -> 15.5; 72 -> 104 at 28^2 x 5 with a residual, one or two stages, 11.0 either way).
                    if (SK || g.iters == 1) {
                        if (stage + s_step < nstages_all) __builtin_amdgcn_s_setprio(2);
                        else __builtin_amdgcn_s_setprio(1);
                    }
                    int st = 0;
                    // Four steps per trip, no branch inside: weights three steps ahead (4 register sets), activations one step
                    // ahead (2 sets). A wave issues in order and a matrix instruction occupies the matrix pipe for 32 cycles: the
                    // requests of the coming steps are therefore spread between the matrix instructions of the current one (each
                    // gap takes a few of them for free) instead of standing in a block in front of them, where the matrix pipe
                    // would run dry while they issue.
                    auto step_order = [&]() __attribute__((always_inline)) {
                        constexpr int kMfma = 0x008, kValu = 0x002, kVmemRead = 0x020, kDsRead = 0x100;
                        if constexpr (SPLIT) return;
                        if constexpr (TT > 4) {      // (the first half of a step: four matrix instructions, the second half's activations)
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kVmemRead, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kDsRead, 2, 0);
                            __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kDsRead, 3, 0);
                            __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            __builtin_amdgcn_sched_barrier(0);
                            return;
                        }
                        if constexpr (NARROW) {
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kVmemRead, 1, 0);
                            if constexpr (TT >= 2) {
                                __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                                __builtin_amdgcn_sched_group_barrier(kDsRead, 2, 0);
                                __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                            }
                            if constexpr (TT == 3) {
                                __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                                __builtin_amdgcn_sched_group_barrier(kDsRead, 2, 0);
                            }
                            if constexpr (TT >= 4) {
                                __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                                __builtin_amdgcn_sched_group_barrier(kDsRead, 2, 0);
                                __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                                __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            }
                            __builtin_amdgcn_sched_barrier(0);
                            return;
                        }
                        __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(kVmemRead, 2, 0);
                        __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                        if constexpr (TT >= 2) {
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                        }
                        if constexpr (TT == 3) {
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                        }
                        if constexpr (TT >= 4) {
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kValu, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(kMfma, 2, 0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    };
                    auto late_order = [&]() __attribute__((always_inline)) {   // the second half: TT - 4 matrix instructions, the next step's first activations
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                        if constexpr (TT > 6) __builtin_amdgcn_sched_group_barrier(0x008, TT - 6, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    };
                    if constexpr (TT > 4) {
                        // Weights as below; the activations one half step ahead.
                        auto step = [&](int cur, int next, int far, int i) __attribute__((always_inline)) {
                            req_a(far, ent);
                            ent = tb[2 * (st + i)];
                            read_b_late(1, bo[cur]);
                            mma(cur, 0);
                            step_order();
                            read_b(0, bo[next]);
                            mma_late(cur, 1);
                            late_order();
                        };
                        for (; st + 4 <= nst_s; st += 4) {
                            step(0, 1, 3, 4);
                            step(1, 2, 0, 5);
                            step(2, 3, 1, 6);
                            step(3, 0, 2, 7);
                        }
                        if (st < nst_s) {
                            read_b_late(1, bo[0]);
                            mma(0, 0);
                            if (st + 1 < nst_s) read_b(0, bo[1]);
                            mma_late(0, 1);
                            if (st + 1 < nst_s) {
                                read_b_late(1, bo[1]);
                                mma(1, 0);
                                if (st + 2 < nst_s) read_b(0, bo[2]);
                                mma_late(1, 1);
                                if (st + 2 < nst_s) {
                                    read_b_late(1, bo[2]);
                                    mma(2, 0);
                                    mma_late(2, 1);
                                }
                            }
                        }
                        continue;
                    }
                    for (; st + 4 <= nst_s; st += 4) {
                        req_a(3, ent);
                        ent = tb[2 * (st + 4)];
                        read_b(1, bo[1]);
                        mma(0, 0);
                        step_order();
                        req_a(0, ent);
                        ent = tb[2 * (st + 5)];
                        read_b(0, bo[2]);
                        mma(1, 1);
                        step_order();
                        req_a(1, ent);
                        ent = tb[2 * (st + 6)];
                        read_b(1, bo[3]);
                        mma(2, 0);
                        step_order();
                        req_a(2, ent);
                        ent = tb[2 * (st + 7)];
                        read_b(0, bo[0]);
                        mma(3, 1);
                        step_order();
                    }
                    // The last nst % 4 steps: wa[0..2] hold their weight fragments, wb[0] the first one's activations.
                    if (st < nst_s) {
                        if (st + 1 < nst_s) read_b(1, bo[1]);
                        mma(0, 0);
                        if (st + 1 < nst_s) {
                            if (st + 2 < nst_s) read_b(0, bo[2]);
                            mma(1, 1);
                            if (st + 2 < nst_s) mma(2, 0);
                        }
                    }
                }
            }

            else {   // (a wave without a tile: never stored)
                park_bias();
                start_sums();
            }

            // The epilogue reads the geometry and the neuron again, from the (cached) kernel arguments: see sk_here.
            const auto& args = sk_kernarg_spk();
            const auto& g = args.g;
            const LifParams lif = {args.lif.v_threshold, args.lif.v_reset, args.lif.tau, args.lif.inv_tau, args.lif.charge_mode, args.lif.soft_reset};
            const int po = g.Ho * g.Wo;
            const int wave_all = wave;
            const int wave = sk_here(wave_all);
            const int WK = SK ? (1 << g.wk_log2) : 1;
            const int wk = SK ? sk_share(wave, WK) : 0;
            const int swap_f = SK && !NARROW ? wk >> (g.wk_log2 - 1) : 0;
            const int quad_x = SK && !NARROW ? (wk << (3 - g.wk_log2)) & 3 : 0;
            const bool common_lif = lif.charge_mode == CHARGE_SCALE && !lif.soft_reset;
            const bool half_tau = lif.inv_tau == 0.5f;

            // ---- epilogue. Accumulator register 4 q + k of fragment f holds channel 32 f + 8 q + 4 half + k of the lane's
            // pixel: a "quad" (f, q) is the lane's half of channel group j8 = TG oc_tile + 4 f + q. One quad at a time: its bias
            // and membrane (4 + 4 registers) live across its timesteps; a lane's addresses are 32-bit offsets from uniform bases.
            if constexpr (!SK) __builtin_amdgcn_s_setprio(0);
            const bool first_window = t0 == 0, last_window = t0 + TT >= nsteps_t;
            const void* v_src = first_window ? v_init : v_carry;          // later windows continue from the stored membrane
            void* const v_dst = last_window ? v_store : v_carry;
            constexpr bool V16 = !SPLIT && IN != SNNF_LAYOUT_NCHW;     // a frame's membrane is fp32 (takes_frame; the internal layouts know no other)
            const bool v_src16 = V16 && g.v16 && first_window, v_dst16 = V16 && g.v16 && last_window;
            const int t_count = g.shared_x ? g.T : min(TT, g.T - t0);      // LIF steps of this window
            // (Made opaque here: everything derived from the lane's pixel is then computed after the matrix loop instead of
            // before it, where the compiler would otherwise park two dozen store addresses in registers or scratch memory.)
            int half_e = half;
            uint32_t pos_e = lane_pos.v[0];
            asm volatile("" : "+v"(pos_e), "+v"(half_e));
            const int pi = static_cast<int>(pos_e & 255u);
            const int n = n0 + pi;
            const int oh = oh0 + static_cast<int>((pos_e >> 8) & 255u);
            const int ow = ow0 + static_cast<int>(pos_e >> 16);
            const bool px_ok = static_cast<bool>(static_cast<int>(have) & static_cast<int>(pi < g.PI) & static_cast<int>(n < g.N) & static_cast<int>(oh < g.Ho) &
                                                 static_cast<int>(ow < g.Wo));
            const int pxo_e = px_ok ? oh * g.Wo + ow : 0;
            const int n_e = px_ok ? n : 0;
            const uint32_t lane_nchw = static_cast<uint32_t>((n_e * g.Cout + 4 * half_e) * po + pxo_e);        // elements
            const uint32_t lane_c8 = static_cast<uint32_t>(((n_e * g.C8out) * po + pxo_e) * 8 + 4 * half_e);   // elements
            const uint32_t lane_bits = static_cast<uint32_t>((n_e * g.C8out) * po + pxo_e);                  // bytes

            // Valid-channel mask and initial membrane of the quad of channel group j8.
            auto quad_begin = [&](int j8, float (&v)[4], uint32_t& chm) __attribute__((always_inline)) {
                const int ch0 = j8 * 8 + 4 * half_e;
                chm = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    chm |= ch0 + k < g.Cout ? (1u << k) : 0u;
                    v[k] = 0.0f;
                }
                if (v_src != nullptr && !g.analog_out && px_ok) {
                    if (v_src16) {
                        const XT* vp = static_cast<const XT*>(v_src) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if ((chm >> k) & 1u) v[k] = to_float(vp[lane_nchw + static_cast<uint32_t>(k * po)]);
                    } else {
                        const float* vp = static_cast<const float*>(v_src) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if ((chm >> k) & 1u) v[k] = vp[lane_nchw + static_cast<uint32_t>(k * po)];
                    }
                }
            };
            // The residual of a quad at timestep `ta`, raw (two registers in any layout), and its addition to the quad's sums.
            constexpr int RW = SPLIT ? 4 : 2;     // registers of a residual quad
            auto res_load = [&](int ta, int j8, uint32_t (&raw)[RW]) __attribute__((always_inline)) {
#pragma unroll
                for (int k = 0; k < RW; ++k) raw[k] = 0u;
                if (g.res_layout < 0 || !(j8 < g.C8out && px_ok)) return;
                const unsigned char* __restrict__ res_t = static_cast<const unsigned char*>(sk_kernarg_ptr(kResTable, ta));
                if constexpr (SPLIT) {
                    const float* __restrict__ rp = reinterpret_cast<const float*>(res_t) + static_cast<int64_t>(j8) * 8 * po;
                    const int ch0 = j8 * 8 + 4 * half_e;
#pragma unroll
                    for (int k = 0; k < 4; ++k) raw[k] = ch0 + k < g.Cout ? __float_as_uint(rp[lane_nchw + static_cast<uint32_t>(k * po)]) : 0u;
                } else if (g.res_layout == SNNF_LAYOUT_BITS) {
                    raw[0] = (res_t + static_cast<int64_t>(j8) * po)[lane_bits];
                } else if (g.res_layout == SNNF_LAYOUT_C8) {
                    const Pack<uint32_t, 2> r2 = *reinterpret_cast<const Pack<uint32_t, 2>*>(reinterpret_cast<const XT*>(res_t) + static_cast<int64_t>(j8) * po * 8 + lane_c8);
                    raw[0] = r2.v[0];
                    raw[1] = r2.v[1];
                } else {
                    const uint16_t* __restrict__ rp = reinterpret_cast<const uint16_t*>(res_t) + static_cast<int64_t>(j8) * 8 * po;
                    const int ch0 = j8 * 8 + 4 * half_e;
                    uint32_t e[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) e[k] = ch0 + k < g.Cout ? rp[lane_nchw + static_cast<uint32_t>(k * po)] : 0u;
                    raw[0] = e[0] | (e[1] << 16);
                    raw[1] = e[2] | (e[3] << 16);
                }
            };
            auto res_add = [&](const uint32_t (&raw)[RW], float (&x)[4]) __attribute__((always_inline)) {
                if (g.res_layout < 0) return;
                if constexpr (SPLIT) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) x[k] += __uint_as_float(raw[k]);
                } else if (g.res_layout == SNNF_LAYOUT_BITS) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) x[k] += ((raw[0] >> (4 * half_e + k)) & 1u) ? 1.0f : 0.0f;
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const uint32_t bits = (raw[k >> 1] >> (16 * (k & 1))) & 0xffffu;
                        if constexpr (!SPLIT) x[k] += to_float(XT{static_cast<uint16_t>(bits)});
                    }
                }
            };
            // Store of 4 channel values of the lane's pixel at timestep `ta` in a dense layout (C8: one 8-byte store).
            auto quad_store_dense = [&](int ta, int j8, const Pack<XT, 4>& o, uint32_t chm) __attribute__((always_inline)) {
                unsigned char* __restrict__ out_t = out + static_cast<int64_t>(ta) * g.out_step_stride;
                if (!SPLIT && g.out_layout == SNNF_LAYOUT_C8) {
                    *reinterpret_cast<Pack<XT, 4>*>(reinterpret_cast<XT*>(out_t) + static_cast<int64_t>(j8) * po * 8 + lane_c8) = o;
                } else {
                    XT* __restrict__ op = reinterpret_cast<XT*>(out_t) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if ((chm >> k) & 1u) op[lane_nchw + static_cast<uint32_t>(k * po)] = o.v[k];
                }
            };
            // One step of a quad at absolute timestep `ta`: x = sums (bias included) (+ residual), then the neuron (its spikes are the
            // returned nibble) or, without a neuron, x itself written to the dense output.
            auto quad_step = [&](int ta, int j8, const float (&x_in)[4], const uint32_t (&res_raw)[RW], float (&v)[4], uint32_t chm) __attribute__((always_inline)) -> uint32_t {
                const bool grp_ok = j8 < g.C8out && px_ok;
                float x[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] = x_in[k];
                res_add(res_raw, x);
                uint32_t nib = 0;
                if (!g.analog_out) {
                    if (common_lif) {   // power-of-two tau, hard reset: one test per quad step instead of two per neuron step
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            // tau = 2: (v + x) / 2, one rounding, the form the straight-line epilogue computes.
                            const float h = half_tau ? (v[k] + x[k]) * 0.5f : v[k] + (x[k] - v[k]) * lif.inv_tau;
                            const bool fired = h >= lif.v_threshold;
                            v[k] = fired ? lif.v_reset : h;
                            nib |= fired ? (1u << k) : 0u;
                        }
                    } else {
#pragma unroll
                        for (int k = 0; k < 4; ++k) nib |= lif_step(x[k], v[k], lif) ? (1u << k) : 0u;
                    }
                    nib &= chm;
                } else if (grp_ok) {
                    Pack<XT, 4> o;
#pragma unroll
                    for (int k = 0; k < 4; ++k) o.v[k] = from_float<XT>(((chm >> k) & 1u) ? x[k] : 0.0f);
                    quad_store_dense(ta, j8, o, chm);
                }
                return nib;
            };
            // Dense spike output of up to 8 consecutive steps [ta0, ta0 + cnt) of a quad from their nibbles, one step at a time
            // (a loop: dense spikes only leave at the network's boundary, and unrolled stores would cost the common path registers).
            auto quad_store_spikes = [&](int ta0, int cnt, int j8, uint32_t nibw, uint32_t chm) __attribute__((always_inline)) {
                if (j8 < g.C8out && px_ok) {
                    for (int i = 0; i < cnt; ++i) {
                        Pack<XT, 4> o;
#pragma unroll
                        for (int k = 0; k < 4; ++k) o.v[k] = spike_value<XT>((nibw >> (4 * i + k)) & 1u);
                        quad_store_dense(ta0 + i, j8, o, chm);
                    }
                }
            };
            // Bit-packed output of up to 8 consecutive steps [ta0, ta0 + cnt) of a quad: nibble i of `nibw` = step ta0 + i. The
            // other half of the wave holds the other nibble of every byte (lanes l and l + 32 own the same pixel); even
            // steps are stored by the lower half, odd steps by the upper half.
            auto quad_store_bits = [&](int ta0, int cnt, int j8, uint32_t nibw) __attribute__((always_inline)) {
                const auto both = __builtin_amdgcn_permlane32_swap(nibw, nibw, false, false);   // [0]: lanes 0..31's word, [1]: lanes 32..63's
                const uint32_t lo = both[0];
                const uint32_t hi = both[1];
                if (j8 < g.C8out && px_ok) {
                    unsigned char* __restrict__ ob = out + static_cast<int64_t>(j8) * po;
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const int i = 2 * m + half_e;
                        if (i < cnt) {
                            const uint32_t byte = ((lo >> (4 * i)) & 15u) | (((hi >> (4 * i)) & 15u) << 4);
                            ob[static_cast<uint32_t>(ta0 + i) * static_cast<uint32_t>(g.out_step_stride) + lane_bits] = static_cast<unsigned char>(byte);
                        }
                    }
                }
            };
            auto quad_end = [&](int j8, const float (&v)[4], uint32_t chm) __attribute__((always_inline)) {
                if (v_dst != nullptr && !g.analog_out && px_ok) {
                    if (v_dst16) {
                        XT* vp = static_cast<XT*>(v_dst) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if ((chm >> k) & 1u) vp[lane_nchw + static_cast<uint32_t>(k * po)] = from_float<XT>(v[k]);
                    } else {
                        float* vp = static_cast<float*>(v_dst) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if ((chm >> k) & 1u) vp[lane_nchw + static_cast<uint32_t>(k * po)] = v[k];
                    }
                }
            };

            const int tb = MULTI ? t0 : 0;   // the straight-line epilogue's first step
            // FAST: the layer as it runs inside a network - bit-packed output, no or a bit-packed residual, the usual neuron
            // (tau = 2, hard reset to 0, a threshold whose power-of-two multiples are normal numbers), zero initial membrane,
            // whole channel groups. Straight-line code.
            // The membrane is kept scaled, S_t = 2^t v_t: a step is then S += 2^(t-1) x (every scaling is exact, so S_t / 2^t
            // is bit for bit the (v + x) / 2 of the general path), a comparison against 2^t v_th and a select, and the carry of
            // the comparison is shifted into the quad's word of quiet (not fired) bits: four instructions per neuron step.
            // After n steps the word holds step i's nibble at bits [4 (n - 1 - i), +4), bit k of a nibble = neuron k.
            auto fast_step4 = [&](const float (&x)[4], int t, float (&S)[4], uint32_t& quiet) __attribute__((always_inline)) {
                const float c = __uint_as_float(static_cast<uint32_t>(127 + t) << 23);                                   // 2^t
                const float th2 = __uint_as_float(__float_as_uint(lif.v_threshold) + (static_cast<uint32_t>(t + 1) << 23));   // 2^(t+1) v_th
                // Neuron 3 first: the last bit shifted in (neuron 0) lands at the nibble's bit 0. The four comparisons write four
                // mask registers and every instruction that reads a mask stands at least two instructions behind the one that
                // wrote it (a vector instruction may not read a scalar register that the previous two vector instructions wrote).
                uint64_t m0, m1, m2, m3;
                asm("v_fmac_f32 %0, %9, %13\n\t"
                    "v_fmac_f32 %1, %9, %12\n\t"
                    "v_fmac_f32 %2, %9, %11\n\t"
                    "v_fmac_f32 %3, %9, %10\n\t"
                    "v_cmp_nle_f32_e64 %5, %14, %0\n\t"
                    "v_cmp_nle_f32_e64 %6, %14, %1\n\t"
                    "v_cmp_nle_f32_e64 %7, %14, %2\n\t"
                    "v_cmp_nle_f32_e64 %8, %14, %3\n\t"
                    "v_cndmask_b32_e64 %0, 0, %0, %5\n\t"
                    "v_cndmask_b32_e64 %1, 0, %1, %6\n\t"
                    "v_cndmask_b32_e64 %2, 0, %2, %7\n\t"
                    "v_cndmask_b32_e64 %3, 0, %3, %8\n\t"
                    "v_addc_co_u32_e64 %4, vcc, %4, %4, %5\n\t"
                    "v_addc_co_u32_e64 %4, vcc, %4, %4, %6\n\t"
                    "v_addc_co_u32_e64 %4, vcc, %4, %4, %7\n\t"
                    "v_addc_co_u32_e64 %4, vcc, %4, %4, %8"
                    : "+v"(S[3]), "+v"(S[2]), "+v"(S[1]), "+v"(S[0]), "+v"(quiet), "=&s"(m3), "=&s"(m2), "=&s"(m1), "=&s"(m0)
                    : "s"(c), "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "s"(th2)
                    : "vcc");
            };
            // x += the residual spikes of this half of the byte (bit k of the nibble -> 0.0 / 1.0 through one byte each).
            auto fast_add_res = [&](uint32_t res_byte, float (&x)[4]) __attribute__((always_inline)) {
                const uint32_t nib = (res_byte >> (4 * half_e)) & 15u;
                const uint32_t spread = __umul24(nib, 0x00204081u) & 0x01010101u;
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] += static_cast<float>((spread >> (8 * k)) & 0xffu);
            };
            // Residual byte of channel group j8 at timestep ta for this lane's pixel (this half's nibble is picked at the use,
            // so that nothing waits on the load where it is issued). Lanes without a pixel read pixel 0 of image 0 (their
            // result is never stored).
            auto fast_res = [&](int ta, int j8) __attribute__((always_inline)) -> uint32_t {
                const unsigned char* __restrict__ res_t = static_cast<const unsigned char*>(sk_kernarg_ptr(kResTable, ta));
                return (res_t + static_cast<int64_t>(min(j8, g.C8out - 1)) * po)[lane_bits];
            };
            // Bit-packed store of the n <= 8 steps [ta0, ta0 + n) of a quad from its word of quiet bits. Lanes l and l + 32 own
            // the two nibbles of every byte of a pixel and swap their words in registers; even steps are stored by the lower
            // half of the wave, odd steps by the upper half.
            auto fast_store = [&](int ta0, int n, int j8, uint32_t quiet) __attribute__((always_inline)) {
                const uint32_t fired = ~quiet;
                const auto both = __builtin_amdgcn_permlane32_swap(fired, fired, false, false);   // [0]: lanes 0..31's word, [1]: lanes 32..63's
                if (j8 < g.C8out && px_ok) {
                    unsigned char* __restrict__ ob = out + static_cast<int64_t>(j8) * po;
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const int i = 2 * m + half_e;
                        if (i < n) {
                            const uint32_t sh = 4u * static_cast<uint32_t>(n - 1 - i);
                            const uint32_t byte = ((both[0] >> sh) & 15u) | (((both[1] >> sh) & 15u) << 4);
                            ob[static_cast<uint32_t>(ta0 + i) * static_cast<uint32_t>(g.out_step_stride) + lane_bits] = static_cast<unsigned char>(byte);
                        }
                    }
                }
            };
            // The same for exactly the four steps of a whole window, of two quads (or of one, with j8b < 0) at once: step i of a word is its nibble
            // 3 - i, so that masked nibbles of both halves' words are whole bytes. The lower half stores steps 0 and 2, the upper half steps 1 and 3.
            const uint32_t step_stride = static_cast<uint32_t>(g.out_step_stride);
            const uint32_t store_first = lane_bits + (half_e ? step_stride : 0u), store_second = store_first + 2u * step_stride;
            const uint32_t nib_down = half_e ? 0u : 4u;
            unsigned char* __restrict__ const out_w = out + static_cast<int64_t>(tb) * g.out_step_stride;
            auto fast_store4 = [&](int j8a, uint32_t quiet_a, int j8b, uint32_t quiet_b) __attribute__((always_inline)) {
                const uint32_t word = quiet_a | (quiet_b << 16);
                const auto both = __builtin_amdgcn_permlane32_swap(word, word, false, false);
                const uint32_t lo = (both[0] >> nib_down) & 0x0f0f0f0fu, hi = (both[1] << (4u - nib_down)) & 0xf0f0f0f0u;
                const uint32_t bytes = ~(lo | hi);               // quad a: steps 2 / 3 and 0 / 1 of this half, then quad b's
                if (px_ok) {
                    if (j8a < g.C8out) {
                        unsigned char* __restrict__ ob = out_w + static_cast<int64_t>(j8a) * po;
                        ob[store_first] = static_cast<unsigned char>(bytes >> 8);
                        ob[store_second] = static_cast<unsigned char>(bytes);
                    }
                    if (j8b >= 0 && j8b < g.C8out) {
                        unsigned char* __restrict__ ob = out_w + static_cast<int64_t>(j8b) * po;
                        ob[store_first] = static_cast<unsigned char>(bytes >> 24);
                        ob[store_second] = static_cast<unsigned char>(bytes >> 16);
                    }
                }
            };
            // The four steps 0..3 as 2x2 average pools of the spikes (POOL): the four lanes of a window (patches have even
            // extents, so a window lies inside one wave half) hold one byte-wide count per channel and step, add them in a
            // reduce-scatter of two exchanges (first with the horizontal neighbour, two steps each way; then with the vertical
            // one, one step each way), and the lane at window position (row r, column c) ends up with step 2 c + r, whose
            // four quarters it stores as 16-bit values of the pooled, channel-blocked tensor. (The caller's steps may lie any distance apart, in
            // either direction: the step's base has 64 bits, the place inside its frame 32.)
            bool odd_col = false, odd_row = false;
            int side = 0, along = 0;
            unsigned char* pool_out = nullptr;
            if constexpr (POOL) {
                const int prow_e = static_cast<int>((pos_e >> 8) & 255u), pcol_e = static_cast<int>(pos_e >> 16);
                odd_col = (pcol_e & 1) != 0;
                odd_row = (prow_e & 1) != 0;
                side = (lane ^ 1) * 4;
                along = (lane + (odd_row ? -g.PC : g.PC)) * 4;
                const int hp = g.Ho >> 1, wp = g.Wo >> 1;
                const int step = (odd_col ? 2 : 0) + (odd_row ? 1 : 0);
                pool_out = out + static_cast<int64_t>(step) * g.out_step_stride + static_cast<uint32_t>(((n_e * g.C8out * hp + (oh >> 1)) * wp + (ow >> 1)) * 8 + 4 * half_e) * 2u;
            }
            auto fast_store4_pooled = [&](int j8, uint32_t quiet) __attribute__((always_inline)) {
                const uint32_t fired = ~quiet;
                uint32_t w[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) w[t] = __umul24((fired >> (4 * (3 - t))) & 15u, 0x00204081u) & 0x01010101u;
                uint32_t keep0 = odd_col ? w[2] : w[0], keep1 = odd_col ? w[3] : w[1];
                const uint32_t give0 = odd_col ? w[0] : w[2], give1 = odd_col ? w[1] : w[3];
                keep0 += static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(side, static_cast<int>(give0)));
                keep1 += static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(side, static_cast<int>(give1)));
                uint32_t keep = odd_row ? keep1 : keep0;
                const uint32_t give = odd_row ? keep0 : keep1;
                keep += static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(along, static_cast<int>(give)));
                if (j8 < g.C8out && px_ok) {
                    Pack<XT, 4> q4;
#pragma unroll
                    for (int k = 0; k < 4; ++k) q4.v[k] = from_float<XT>(static_cast<float>((keep >> (8 * k)) & 255u) * 0.25f);
                    *reinterpret_cast<Pack<XT, 4>*>(pool_out + static_cast<int64_t>(j8) * ((g.Ho >> 1) * (g.Wo >> 1)) * 16) = q4;
                }
            };
            // A quad's membrane from the window before.
            auto fast_v0 = [&](int j8, float (&v0)[4]) __attribute__((always_inline)) {
                if (MULTI && t0 > 0) {
                    const float* vp = v_out + static_cast<int64_t>(min(j8, g.C8out - 1)) * 8 * po;
#pragma unroll
                    for (int k = 0; k < 4; ++k) v0[k] = vp[lane_nchw + static_cast<uint32_t>(k * po)];
                }
            };
            // All steps of one quad whose sums are xq[tw][k]: residual, LIF, bit-packed store, optional membrane store.
            // `v0`: the membrane the window starts from (a later window's is what the one before stored, zero in the first).
            auto fast_quad = [&](int j8, const float (&xq)[TT][4], const uint32_t (&rb)[TT], bool with_res, const float (&v0)[4]) __attribute__((always_inline)) {
                float S[4] = {v0[0], v0[1], v0[2], v0[3]};
                if constexpr (TT == 1) {
                    if (t_count == 4 && !with_res) {
                        // The usual stem: one frame, four steps, no residual. Straight-line.
                        uint32_t quiet = 0;
#pragma unroll
                        for (int i = 0; i < 4; ++i) fast_step4(xq[0], i, S, quiet);
                        if constexpr (POOL) fast_store4_pooled(j8, quiet);
                        else fast_store4(j8, quiet, -1, 0u);
                    } else {
                        for (int ta0 = 0; ta0 < t_count; ta0 += 8) {
                            const int cnt = min(8, t_count - ta0);
                            uint32_t quiet = 0;
                            for (int i = 0; i < cnt; ++i) {
                                float x[4];
#pragma unroll
                                for (int k = 0; k < 4; ++k) x[k] = xq[0][k];
                                if (with_res) fast_add_res(fast_res(tb + ta0 + i, j8), x);
                                fast_step4(x, ta0 + i, S, quiet);
                            }
                            fast_store(tb + ta0, cnt, j8, quiet);
                        }
                    }
                } else {
                    uint32_t quiet = 0;
                    if (t_count == TT) {
                        // Every step of the window is real (the usual case): no condition per step.
                        if (with_res) {
#pragma unroll
                            for (int tw = 0; tw < TT; ++tw) {
                                float x[4];
#pragma unroll
                                for (int k = 0; k < 4; ++k) x[k] = xq[tw][k];
                                fast_add_res(rb[tw], x);
                                fast_step4(x, tw, S, quiet);
                            }
                        } else {
#pragma unroll
                            for (int tw = 0; tw < TT; ++tw) fast_step4(xq[tw], tw, S, quiet);
                        }
                        if constexpr (TT == 4) {
                            if constexpr (POOL) fast_store4_pooled(j8, quiet);
                            else fast_store4(j8, quiet, -1, 0u);
                        } else {
                            fast_store(tb, TT, j8, quiet);
                        }
                    } else {
#pragma unroll
                        for (int tw = 0; tw < TT; ++tw) {
                            if (tw < t_count) {
                                float x[4];
#pragma unroll
                                for (int k = 0; k < 4; ++k) x[k] = xq[tw][k];
                                if (with_res) fast_add_res(rb[tw], x);
                                fast_step4(x, tw, S, quiet);
                            }
                        }
                        fast_store(tb, t_count, j8, quiet);
                    }
                }
                if (v_out != nullptr && px_ok && j8 < g.C8out) {
                    float* __restrict__ vp = v_out + static_cast<int64_t>(j8) * 8 * po;
                    const float unscale = __uint_as_float(static_cast<uint32_t>(127 - t_count) << 23);   // 2^-t_count
#pragma unroll
                    for (int k = 0; k < 4; ++k) vp[lane_nchw + static_cast<uint32_t>(k * po)] = S[k] * unscale;
                }
            };
            // The quads of a usual tile - four steps from a zero membrane that is not asked for - two at a time, without a condition per quad: 8.4 k -> 5.2 k
            // cycles for a wave's eight quads, 11.5 k -> 7.9 k with a residual (64 -> 64 at 56^2 x 16 19.5 -> 18.4 us and 20.7 -> 19.8).
            constexpr bool LEAN = TT == 4 || TT == 3 || TT == 1;
            constexpr int LT = TT == 3 ? 3 : 4;      // (of three steps where the window has three)
            const bool lean = LEAN && !MULTI && t_count == LT && v_out == nullptr;
            auto lean_quad = [&](const float (&xq)[TT][4], const uint32_t (&rb)[TT], auto res_tag) __attribute__((always_inline)) -> uint32_t {
                float S[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                uint32_t quiet = 0;
#pragma unroll
                for (int i = 0; i < LT; ++i) {
                    if constexpr (decltype(res_tag)::value) {
                        float x[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) x[k] = xq[i % TT][k];
                        fast_add_res(rb[i % TT], x);
                        fast_step4(x, i, S, quiet);
                    } else {
                        fast_step4(xq[i % TT], i, S, quiet);
                    }
                }
                return quiet;
            };
            // Quad FQ, and FQ + 1 with TWO, of the sums `sum(timestep, quad, k)`, as the channel groups j8a and j8b.
            auto lean_pair = [&](const auto& sum, auto fq_tag, auto two_tag, auto res_tag, int j8a, int j8b, const uint32_t (&ra)[TT], const uint32_t (&rb)[TT]) __attribute__((always_inline)) {
                constexpr int FQ = decltype(fq_tag)::value;
                constexpr bool TWO = decltype(two_tag)::value;
                uint32_t qa, qb = 0;
                float xq[TT][4];
#pragma unroll
                for (int tw = 0; tw < TT; ++tw)
#pragma unroll
                    for (int k = 0; k < 4; ++k) xq[tw][k] = sum(tw, FQ, k);
                qa = lean_quad(xq, ra, res_tag);
                if constexpr (POOL) fast_store4_pooled(j8a, qa);
                if constexpr (TWO) {
#pragma unroll
                    for (int tw = 0; tw < TT; ++tw)
#pragma unroll
                        for (int k = 0; k < 4; ++k) xq[tw][k] = sum(tw, FQ + 1, k);
                    qb = lean_quad(xq, rb, res_tag);
                    if constexpr (POOL) fast_store4_pooled(j8b, qb);
                }
                if constexpr (TT == 3) {
                    fast_store(tb, 3, j8a, qa);
                    if constexpr (TWO) fast_store(tb, 3, j8b, qb);
                } else if constexpr (!POOL) {
                    fast_store4(j8a, qa, TWO ? j8b : -1, qb);
                }
            };
            // DENSE: dense spikes (and residual) around the usual neuron (tau 2, hard reset), any number of windows and channels. A lane's
            // pixel is one element of a channel plane, so spikes, residual and membrane move as single elements, 32 lanes side by side.
            // What that costs is the segments of a patch's rows, not the instructions: 25.7 MB of spikes in patches of 4 x 8 pixels take
            // 12 us in single elements and in runs of 16 bytes alike. The residual (and the membrane of a previous window) of a
            // quad is requested one quad ahead: waited for in turn it cost 28 us on 64 -> 64 at 56^2 x 16 (67 -> 39 us without).
            using DT = typename std::conditional<SPLIT, uint32_t, uint16_t>::type;     // an element's bits
            constexpr bool FRAME = LATE_BIAS;                   // one sum for all steps, no residual
            struct DenseIn { uint32_t res[TT][4]; uint32_t v[4]; sk_f32x4 bias; };
            auto dense_request = [&](int j8_any, DenseIn& in) __attribute__((always_inline)) {
                const int j8 = min(j8_any, g.C8out - 1);
                const int left = g.Cout - (j8 * 8 + 4 * half_e);     // channels of this lane's quad, and beyond
                if constexpr (FRAME) in.bias = *reinterpret_cast<const sk_f32x4*>(bias + j8 * 8 + 4 * half_e);     // (zeros beyond the last)
                auto get = [&](auto ragged_tag) __attribute__((always_inline)) {
                    constexpr bool RAGGED = decltype(ragged_tag)::value;
                    // Lanes without a pixel read pixel 0 of image 0; channels beyond the last are not read.
                    if (RAGGED || left > 0) {
                        if (g.res_layout >= 0) {
#pragma unroll
                            for (int tw = 0; tw < TT; ++tw) {
                                const DT* __restrict__ rp = static_cast<const DT*>(sk_kernarg_ptr(kResTable, min(t0 + tw, g.T - 1))) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                                for (int k = 0; k < 4; ++k)
                                    if (!RAGGED || k < left) in.res[tw][k] = rp[lane_nchw + static_cast<uint32_t>(k * po)];
                            }
                        }
                        if (v_src != nullptr) {
                            if (v_src16) {
                                const uint16_t* vp = static_cast<const uint16_t*>(v_src) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                                for (int k = 0; k < 4; ++k)
                                    if (!RAGGED || k < left) in.v[k] = vp[lane_nchw + static_cast<uint32_t>(k * po)];
                            } else {
                                const uint32_t* vp = static_cast<const uint32_t*>(v_src) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                                for (int k = 0; k < 4; ++k)
                                    if (!RAGGED || k < left) in.v[k] = vp[lane_nchw + static_cast<uint32_t>(k * po)];
                            }
                        }
                    }
                };
                if (g.res_layout >= 0 || v_src != nullptr) {
                    if (g.Cout & 3) get(std::true_type{});
                    else get(std::false_type{});
                }
            };
            auto dense_quad = [&](int j8, const float (&xq)[TT][4], const DenseIn& in) __attribute__((always_inline)) {
                if (j8 >= g.C8out) return;
                const int left = g.Cout - (j8 * 8 + 4 * half_e);
                float v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = 0.0f;
                if (v_src != nullptr) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        if constexpr (SPLIT) v[k] = __uint_as_float(in.v[k]);
                        else v[k] = v_src16 ? to_float(XT{static_cast<uint16_t>(in.v[k])}) : __uint_as_float(in.v[k]);
                    }
                }
                auto run = [&](auto ragged_tag) __attribute__((always_inline)) {
                    constexpr bool RAGGED = decltype(ragged_tag)::value;
                    if (px_ok && left > 0) {
                        auto step = [&](int t, int tw) __attribute__((always_inline)) {
                            DT* __restrict__ op = reinterpret_cast<DT*>(out + static_cast<int64_t>(t) * g.out_step_stride) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                            for (int k = 0; k < 4; ++k) {
                                float x = xq[tw][k];
                                if constexpr (FRAME) x += in.bias[k];
                                if (!FRAME && g.res_layout >= 0) {
                                    if constexpr (SPLIT) x += __uint_as_float(in.res[tw][k]);
                                    else x += to_float(XT{static_cast<uint16_t>(in.res[tw][k])});
                                }
                                const float h = FRAME ? v[k] + (x - v[k]) * 0.5f : (v[k] + x) * 0.5f;
                                const bool fired = h >= lif.v_threshold;
                                v[k] = fired ? lif.v_reset : h;
                                const DT spike = fired ? static_cast<DT>(SPLIT ? 0x3f800000u : ONE) : DT{0};
                                if (!RAGGED || k < left) op[lane_nchw + static_cast<uint32_t>(k * po)] = spike;
                            }
                        };
                        if constexpr (FRAME) {
                            for (int t = 0; t < t_count; ++t) step(t, 0);
                        } else {
#pragma unroll
                            for (int tw = 0; tw < TT; ++tw)
                                if (tw < t_count) step(t0 + tw, tw);
                        }
                        if (v_dst16) {
                            if constexpr (!SPLIT) {
                                XT* vp = static_cast<XT*>(v_dst) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                                for (int k = 0; k < 4; ++k)
                                    if (!RAGGED || k < left) vp[lane_nchw + static_cast<uint32_t>(k * po)] = from_float<XT>(v[k]);
                            }
                        } else if (!FRAME || v_dst != nullptr) {      // (a network's own layers keep no membrane)
                            float* vp = static_cast<float*>(v_dst) + static_cast<int64_t>(j8) * 8 * po;
#pragma unroll
                            for (int k = 0; k < 4; ++k)
                                if (!RAGGED || k < left) vp[lane_nchw + static_cast<uint32_t>(k * po)] = v[k];
                        }
                    }
                };
                if (g.Cout & 3) run(std::true_type{});
                else run(std::false_type{});
            };
            // All steps of one quad, any layouts and neuron (the general path).
            auto general_quad = [&](int j8, const float (&xq)[TT][4]) __attribute__((always_inline)) {
                float v[4];
                uint32_t chm;
                quad_begin(j8, v, chm);
                if constexpr (TT == 1) {
                    // One convolution result, t_count LIF steps on it (one step, or one frame shared by all T timesteps).
                    for (int ta0 = 0; ta0 < t_count; ta0 += 8) {
                        const int cnt = min(8, t_count - ta0);
                        uint32_t nibw = 0;
                        for (int i = 0; i < cnt; ++i) {
                            uint32_t rr[RW];
                            res_load(t0 + ta0 + i, j8, rr);
                            nibw |= quad_step(t0 + ta0 + i, j8, xq[0], rr, v, chm) << (4 * i);
                        }
                        if (g.out_layout == SNNF_LAYOUT_BITS) quad_store_bits(t0 + ta0, cnt, j8, nibw);
                        else if (!g.analog_out) quad_store_spikes(t0 + ta0, cnt, j8, nibw, chm);
                    }
                } else {
                    uint32_t rr[TT][RW];
#pragma unroll
                    for (int tw = 0; tw < TT; ++tw) res_load(min(t0 + tw, g.T - 1), j8, rr[tw]);
                    uint32_t nibw = 0;
#pragma unroll
                    for (int tw = 0; tw < TT; ++tw)
                        if (tw < t_count) nibw |= quad_step(t0 + tw, j8, xq[tw], rr[tw], v, chm) << (4 * tw);
                    if (g.out_layout == SNNF_LAYOUT_BITS) quad_store_bits(t0, t_count, j8, nibw);
                    else if (!g.analog_out) quad_store_spikes(t0, t_count, j8, nibw, chm);
                }
                quad_end(j8, v, chm);
            };

            if constexpr (!SK) {
                if constexpr (FAST) {
                    const bool with_res = g.res_layout >= 0;
                    // The residual bytes of all 8 quads are requested up front (the matrix loop's operand registers are free now):
                    // one round trip to memory for the whole epilogue. The fence keeps the compiler from sinking each request
                    // to its use, where every one of them would be waited for in turn.
                    uint32_t rb[8][TT];
                    float v0[8][4];
#pragma unroll
                    for (int fq = 0; fq < 8; ++fq) {
#pragma unroll
                        for (int tw = 0; tw < TT; ++tw) rb[fq][tw] = 0u;
#pragma unroll
                        for (int k = 0; k < 4; ++k) v0[fq][k] = 0.0f;
                    }
                    if (MULTI && t0 > 0) {
#pragma unroll
                        for (int fq = 0; fq < TG; ++fq) fast_v0(oc_e * TG + fq, v0[fq]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if (with_res && TT > 1) {
                        const unsigned char* res_ptr[TT];
#pragma unroll
                        for (int tw = 0; tw < TT; ++tw)
                            res_ptr[tw] = static_cast<const unsigned char*>(sk_kernarg_ptr(kResTable, tb + min(tw, t_count - 1))) + static_cast<int64_t>(oc_e) * TG * po;
                        auto req_res = [&](auto fq_tag) __attribute__((always_inline)) {
                            constexpr int fq = decltype(fq_tag)::value;
                            if constexpr (fq >= TG) return;
                            const uint32_t off = lane_bits + static_cast<uint32_t>(min(fq, g.C8out - 1 - oc_e * TG) * po);
#pragma unroll
                            for (int tw = 0; tw < TT; ++tw) rb[fq][tw] = res_ptr[tw][off];
                        };
                        req_res(std::integral_constant<int, 0>{});
                        req_res(std::integral_constant<int, 1>{});
                        req_res(std::integral_constant<int, 2>{});
                        req_res(std::integral_constant<int, 3>{});
                        req_res(std::integral_constant<int, 4>{});
                        req_res(std::integral_constant<int, 5>{});
                        req_res(std::integral_constant<int, 6>{});
                        req_res(std::integral_constant<int, 7>{});
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    auto lean_all = [&](auto res_tag) __attribute__((always_inline)) {
                        const int j0 = oc_e * TG;
                        const std::true_type two;
                        const auto sum = [&](int tw, int fq, int k) __attribute__((always_inline)) { return acc[tw][(fq >> 2) % NF][4 * (fq & 3) + k]; };
                        lean_pair(sum, std::integral_constant<int, 0>{}, two, res_tag, j0, j0 + 1, rb[0], rb[1]);
                        lean_pair(sum, std::integral_constant<int, 2>{}, two, res_tag, j0 + 2, j0 + 3, rb[2], rb[3]);
                        if constexpr (TG == 8) {
                            lean_pair(sum, std::integral_constant<int, 4>{}, two, res_tag, j0 + 4, j0 + 5, rb[4], rb[5]);
                            lean_pair(sum, std::integral_constant<int, 6>{}, two, res_tag, j0 + 6, j0 + 7, rb[6], rb[7]);
                        }
                    };
                    if constexpr (MULTI) {
                        auto do_quad = [&](auto fq_tag) __attribute__((always_inline)) {
                            constexpr int fq = decltype(fq_tag)::value;
                            if constexpr (fq < TG) {
                                float xq[TT][4];
#pragma unroll
                                for (int tw = 0; tw < TT; ++tw)
#pragma unroll
                                    for (int k = 0; k < 4; ++k) xq[tw][k] = acc[tw][(fq >> 2) % NF][4 * (fq & 3) + k];
                                fast_quad(oc_e * TG + fq, xq, rb[fq], with_res, v0[fq]);
                            }
                        };
                        do_quad(std::integral_constant<int, 0>{});
                        do_quad(std::integral_constant<int, 1>{});
                        do_quad(std::integral_constant<int, 2>{});
                        do_quad(std::integral_constant<int, 3>{});
                        do_quad(std::integral_constant<int, 4>{});
                        do_quad(std::integral_constant<int, 5>{});
                        do_quad(std::integral_constant<int, 6>{});
                        do_quad(std::integral_constant<int, 7>{});
                    } else if (lean && !with_res) {
                        lean_all(std::false_type{});
                    } else if (lean && TT >= 3) {
                        lean_all(std::true_type{});
                    } else {
                        // A loop: a quad's sums are copied out of the accumulators by a switch (constant register indices).
                        for (int fq = 0; fq < TG; ++fq) {
                            float xq[TT][4];
                            uint32_t rq[TT];
#define SNNF_SPK_COPY_QUAD(F, Q)                                                                                          \
    _Pragma("unroll") for (int tw = 0; tw < TT; ++tw) {                                                                   \
        _Pragma("unroll") for (int k = 0; k < 4; ++k) xq[tw][k] = acc[tw][(F) % NF][4 * (Q) + k];                         \
        rq[tw] = rb[4 * (F) + (Q)][tw];                                                                                   \
    }
                            switch (fq) {
                                case 0: SNNF_SPK_COPY_QUAD(0, 0); break;
                                case 1: SNNF_SPK_COPY_QUAD(0, 1); break;
                                case 2: SNNF_SPK_COPY_QUAD(0, 2); break;
                                case 3: SNNF_SPK_COPY_QUAD(0, 3); break;
                                case 4: SNNF_SPK_COPY_QUAD(1, 0); break;
                                case 5: SNNF_SPK_COPY_QUAD(1, 1); break;
                                case 6: SNNF_SPK_COPY_QUAD(1, 2); break;
                                default: SNNF_SPK_COPY_QUAD(1, 3); break;
                            }
#undef SNNF_SPK_COPY_QUAD
                            fast_quad(oc_e * TG + fq, xq, rq, with_res, v0[0]);
                        }
                    }
                } else if constexpr (DENSE) {
                    DenseIn in[2] = {};
                    dense_request(oc_e * TG, in[0]);
                    auto do_quad = [&](auto fq_tag) __attribute__((always_inline)) {
                        constexpr int fq = decltype(fq_tag)::value;
                        if constexpr (fq < TG) {
                            if constexpr (fq + 1 < TG) dense_request(oc_e * TG + fq + 1, in[(fq + 1) & 1]);
                            float xq[TT][4];
#pragma unroll
                            for (int tw = 0; tw < TT; ++tw)
#pragma unroll
                                for (int k = 0; k < 4; ++k) xq[tw][k] = acc[tw][(fq >> 2) % NF][4 * (fq & 3) + k];
                            dense_quad(oc_e * TG + fq, xq, in[fq & 1]);
                        }
                    };
                    do_quad(std::integral_constant<int, 0>{});
                    do_quad(std::integral_constant<int, 1>{});
                    do_quad(std::integral_constant<int, 2>{});
                    do_quad(std::integral_constant<int, 3>{});
                    do_quad(std::integral_constant<int, 4>{});
                    do_quad(std::integral_constant<int, 5>{});
                    do_quad(std::integral_constant<int, 6>{});
                    do_quad(std::integral_constant<int, 7>{});
                } else {
                    // A runtime loop over the wave's 8 quads keeps the code small; a quad's sums are copied out of the accumulators
                    // by a switch (constant register indices), so the accumulators stay in registers.
                    for (int fq = 0; fq < TG; ++fq) {
                        float xq[TT][4];
#define SNNF_SPK_COPY_QUAD(F, Q)                                          \
    _Pragma("unroll") for (int tw = 0; tw < TT; ++tw)                     \
        _Pragma("unroll") for (int k = 0; k < 4; ++k) xq[tw][k] = acc[tw][(F) % NF][4 * (Q) + k]
                        switch (fq) {
                            case 0: SNNF_SPK_COPY_QUAD(0, 0); break;
                            case 1: SNNF_SPK_COPY_QUAD(0, 1); break;
                            case 2: SNNF_SPK_COPY_QUAD(0, 2); break;
                            case 3: SNNF_SPK_COPY_QUAD(0, 3); break;
                            case 4: SNNF_SPK_COPY_QUAD(1, 0); break;
                            case 5: SNNF_SPK_COPY_QUAD(1, 1); break;
                            case 6: SNNF_SPK_COPY_QUAD(1, 2); break;
                            default: SNNF_SPK_COPY_QUAD(1, 3); break;
                        }
#undef SNNF_SPK_COPY_QUAD
                        general_quad(oc_e * TG + fq, xq);
                    }
                }
            } else {
                // Split K: the WK waves of a tile add their partial sums through LDS. A wave's slot is its own staging region, which it has read when it
                // parks its sums there: the waves that are done first park while the others still multiply, and the workgroup meets once before the first
                // sums are read. With that, reads that are all requested before the first is waited for (in turn, 16 latencies of 130 cycles), one round
                // instead of two between the last four waves, the residual bytes of all quads under way from the start, and the lean quads above, a wave
                // of 128 -> 128 at 28^2 x 16 has its sums 3.4 k cycles after its last product instead of 4.4 k and is done 2.3 k later instead of 4.5 k, at
                // 512 -> 512, 7^2 x 16 5.1 k instead of 7.0 k (20.2 -> 19.3 us, 18.9 -> 18.5; 64 -> 128 stride 2 16.9 -> 16.1, 72 -> 104 at 28^2 x 5 with a residual 11.9 -> 11.1).
                unsigned char* __restrict__ part = lds + kSpkHeaderBytes;      // [wave][place 0..3][tw][lane][4 floats]
                const int slot_bytes = g.lds_wave_bytes;
                int lane_p = lane;                       // opaque: the addresses below are computed here, not ahead of the matrix loop
                asm volatile("" : "+v"(lane_p));
                // Quad Q of fragment F goes to place P of slot S.
#define SNNF_SPK_PARK_QUAD(S, P, F, Q)                                                                                           \
    _Pragma("unroll") for (int tw = 0; tw < TT; ++tw) {                                                                          \
        const sk_f32x4 four = {acc[tw][(F) % NF][4 * (Q)], acc[tw][(F) % NF][4 * (Q) + 1], acc[tw][(F) % NF][4 * (Q) + 2], acc[tw][(F) % NF][4 * (Q) + 3]};  \
        *reinterpret_cast<sk_f32x4*>(part + (S) * slot_bytes + (((P) * TT + tw) * 64 + lane_p) * 16) = four;                      \
    }
                if constexpr (!NARROW) {
                    // Halves are exchanged until every wave owns 8 / WK quads: first the fragment that a wave does not finish, then two
                    // quads of its own (three of eight waves). All waves add and finish at the same time; a slot that a wave has read takes what it
                    // gives away next. (Quads parked by all waves and summed by one each, in two rounds of which half of eight waves
                    // took no part, took 23.4 us at 512 -> 512, 7^2 x 16 against 22.4, 21.8 against 21.2 at 256 -> 256, 14^2 x 16, and in two windows 25.7
                    // against 22.3 at 128 -> 256 stride 2, 40^2 x 3, T = 8; 1.04 over 60 such layers.)
                    SNNF_SPK_PARK_QUAD(wave, 0, 1, 0) SNNF_SPK_PARK_QUAD(wave, 1, 1, 1) SNNF_SPK_PARK_QUAD(wave, 2, 1, 2) SNNF_SPK_PARK_QUAD(wave, 3, 1, 3)
                    const int jq = oc_e * TG + 4 * swap_f;
                    const int quads = 8 >> g.wk_log2;
                    // The residual bytes (and membranes of the window before) of all of the wave's quads travel while the workgroup meets: a second round
                    // trip for the second quad and on, after the sums had met, was 0.8 k cycles each.
                    uint32_t rb[4][TT];
                    float v0[4][4];
                    DenseIn in = {};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
#pragma unroll
                        for (int tw = 0; tw < TT; ++tw) rb[e][tw] = 0u;
#pragma unroll
                        for (int k = 0; k < 4; ++k) v0[e][k] = 0.0f;
                    }
                    if constexpr (FAST) {
                        if (g.res_layout >= 0 && TT > 1) {
                            const unsigned char* res_t[TT];
#pragma unroll
                            for (int tw = 0; tw < TT; ++tw) res_t[tw] = static_cast<const unsigned char*>(sk_kernarg_ptr(kResTable, tb + min(tw, t_count - 1)));
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                if (e < quads) {
                                    const uint32_t off = lane_bits + static_cast<uint32_t>(min(jq + (e ^ quad_x), g.C8out - 1) * po);
#pragma unroll
                                    for (int tw = 0; tw < TT; ++tw) rb[e][tw] = res_t[tw][off];
                                }
                        }
                        if constexpr (MULTI) {
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                if (e < quads) fast_v0(jq + (e ^ quad_x), v0[e]);
                        }
                    }
                    if constexpr (DENSE) dense_request(jq + quad_x, in);
                    __syncthreads();
                    const int across = wave ^ (WK >> 1);
                    unsigned char* const mine = part + across * slot_bytes + lane_p * 16;      // the slot that this wave reads, and takes for its own from then on
                    // Place `place` of slot `slot`: a quad of all timesteps.
                    auto take = [&](int slot, int place, sk_f32x4 (&four)[TT]) __attribute__((always_inline)) {
#pragma unroll
                        for (int tw = 0; tw < TT; ++tw) four[tw] = *reinterpret_cast<const sk_f32x4*>(part + slot * slot_bytes + ((place * TT + tw) * 64 + lane_p) * 16);
                    };
                    auto give = [&](int place, const sk_f32x4 (&four)[TT]) __attribute__((always_inline)) {
#pragma unroll
                        for (int tw = 0; tw < TT; ++tw) *reinterpret_cast<sk_f32x4*>(mine + (place * TT + tw) * 1024) = four[tw];
                    };
                    auto add = [&](sk_f32x4 (&to)[TT], const sk_f32x4 (&four)[TT]) __attribute__((always_inline)) {
#pragma unroll
                        for (int tw = 0; tw < TT; ++tw)
#pragma unroll
                            for (int k = 0; k < 4; ++k) to[tw][k] += four[tw][k];
                    };
                    sk_f32x4 own[4][TT];
                    {
                        sk_f32x4 sums[4][TT];            // (all requested before the first is waited for: one latency instead of sixteen)
#pragma unroll
                        for (int q = 0; q < 4; ++q) take(across, q, sums[q]);
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
#pragma unroll
                            for (int tw = 0; tw < TT; ++tw)
#pragma unroll
                                for (int k = 0; k < 4; ++k) own[q][tw][k] = acc[tw][0][4 * q + k];
                            add(own[q], sums[q]);
                        }
                    }
                    // The wave's finished quads: run at once (FAST, usual tiles), or left in LDS for the loop below.
                    auto finish = [&](auto quads_tag) __attribute__((always_inline)) {
                        constexpr int QUADS = decltype(quads_tag)::value;
                        if constexpr (FAST && LEAN) {
                            const auto sum = [&](int tw, int q, int k) __attribute__((always_inline)) { return own[q][tw][k]; };
                            auto lean_all = [&](auto res_tag) __attribute__((always_inline)) {
                                lean_pair(sum, std::integral_constant<int, 0>{}, std::integral_constant<bool, (QUADS > 1)>{}, res_tag, jq + quad_x, jq + (1 ^ quad_x), rb[0], rb[1]);
                                if constexpr (QUADS == 4) lean_pair(sum, std::integral_constant<int, 2>{}, std::true_type{}, res_tag, jq + 2, jq + 3, rb[2], rb[3]);
                            };
                            if (lean && g.res_layout < 0) {
                                lean_all(std::false_type{});
                                return;
                            }
                            if (lean && TT >= 3) {
                                lean_all(std::true_type{});
                                return;
                            }
                        }
#pragma unroll
                        for (int q = 0; q < QUADS; ++q) give(q, own[q]);
                    };
                    if (WK == 2) {
                        finish(std::integral_constant<int, 4>{});
                    } else if (WK == 4) {
                        give(2, own[2]);
                        give(3, own[3]);
                        __syncthreads();
                        sk_f32x4 sums[2][TT];
                        take(across ^ 1, 2, sums[0]);
                        take(across ^ 1, 3, sums[1]);
                        __builtin_amdgcn_sched_barrier(0);
                        add(own[0], sums[0]);
                        add(own[1], sums[1]);
                        finish(std::integral_constant<int, 2>{});
                    } else {
                        // Of four waves each keeps one quad and gives the others theirs, added as (own + second) + (first + third).
                        give(1, own[1]);
                        give(2, own[2]);
                        give(3, own[3]);
                        __syncthreads();
                        sk_f32x4 first[TT], second[TT], third[TT];
                        take(across ^ 2, 2, second);
                        take(across ^ 1, 1, first);
                        take(across ^ 3, 3, third);
                        __builtin_amdgcn_sched_barrier(0);
                        add(own[0], second);
                        add(first, third);
                        add(own[0], first);
                        finish(std::integral_constant<int, 1>{});
                    }
                    if (!(FAST && lean && (TT >= 3 || (TT == 1 && g.res_layout < 0)))) {
                        for (int e = 0; e < quads; ++e) {
                            const int j8 = jq + (e ^ quad_x);
                            float xq[TT][4];
#pragma unroll
                            for (int tw = 0; tw < TT; ++tw) {
                                const sk_f32x4 four = *reinterpret_cast<const sk_f32x4*>(mine + (e * TT + tw) * 1024);
#pragma unroll
                                for (int k = 0; k < 4; ++k) xq[tw][k] = four[k];
                            }
                            if constexpr (FAST) {
                                float start[4] = {v0[0][0], v0[0][1], v0[0][2], v0[0][3]};
                                uint32_t rq[TT];
#pragma unroll
                                for (int tw = 0; tw < TT; ++tw) rq[tw] = rb[0][tw];
                                if (e > 0) {     // (constant register indices)
#pragma unroll
                                    for (int q = 1; q < 4; ++q)
                                        if (e == q) {
#pragma unroll
                                            for (int tw = 0; tw < TT; ++tw) rq[tw] = rb[q][tw];
#pragma unroll
                                            for (int k = 0; k < 4; ++k) start[k] = v0[q][k];
                                        }
                                }
                                fast_quad(j8, xq, rq, g.res_layout >= 0, start);
                            } else if constexpr (DENSE) {
                                const DenseIn now = in;
                                if (e + 1 < quads) dense_request(jq + ((e + 1) ^ quad_x), in);
                                dense_quad(j8, xq, now);
                            } else {
                                general_quad(j8, xq);
                            }
                        }
                    }
                } else {
                    // A narrow tile's four quads, all TT timesteps: quad e is finished by wave e mod WK of the tile, which adds the WK
                    // partial sums in a fixed order and then runs that quad's timesteps like the unsplit kernel.
                    // (Of more than four timesteps a slot holds four at a time: the first four of all quads, then the others.)
                    auto park = [&](auto from_tag, auto to_tag) __attribute__((always_inline)) {
                        constexpr int FROM = decltype(from_tag)::value, TO = decltype(to_tag)::value;
#pragma unroll
                        for (int q = 0; q < 4; ++q)
#pragma unroll
                            for (int tw = FROM; tw < TO; ++tw) {
                                const sk_f32x4 four = {acc[tw][0][4 * q], acc[tw][0][4 * q + 1], acc[tw][0][4 * q + 2], acc[tw][0][4 * q + 3]};
                                *reinterpret_cast<sk_f32x4*>(part + wave * slot_bytes + ((q * TL + tw - FROM) * 64 + lane_p) * 16) = four;
                            }
                    };
                    park(std::integral_constant<int, 0>{}, std::integral_constant<int, TL>{});
                    const int part0 = wave ^ wk;         // the slot of part k is part0 ^ k
                    const int e_first = wk;      // this wave finishes quads e_first, e_first + WK, ... < 4
                    // The residual bytes of the wave's first quad travel while the workgroup meets.
                    uint32_t rb[TT];
#pragma unroll
                    for (int tw = 0; tw < TT; ++tw) rb[tw] = 0u;
                    if constexpr (FAST) {
                        if (e_first < 4 && g.res_layout >= 0 && TT > 1) {
#pragma unroll
                            for (int tw = 0; tw < TT; ++tw) rb[tw] = fast_res(tb + min(tw, t_count - 1), oc_e * TG + e_first);
                        }
                    }
                    float v0[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                    if constexpr (FAST) {
                        if (e_first < 4) fast_v0(oc_e * TG + e_first, v0);
                    }
                    DenseIn in = {};
                    if constexpr (DENSE) {
                        if (e_first < 4) dense_request(oc_e * TG + e_first, in);
                    }
                    __syncthreads();
                    // The partial sums of the tile's waves for the N timesteps that are parked, of two or four waves in flight together (WK is a power of two
                    // >= 2); added in the order of the parts.
                    auto gather = [&](auto n_tag, int e_own, sk_f32x4* __restrict__ sum) __attribute__((always_inline)) {
                        constexpr int N = decltype(n_tag)::value;
#pragma unroll
                        for (int tw = 0; tw < N; ++tw) sum[tw] = sk_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                        auto add_parts = [&](auto parts_tag, int k) __attribute__((always_inline)) {
                            constexpr int PARTS = decltype(parts_tag)::value;
                            sk_f32x4 p[PARTS][N];
#pragma unroll
                            for (int i = 0; i < PARTS; ++i)
#pragma unroll
                                for (int tw = 0; tw < N; ++tw) p[i][tw] = *reinterpret_cast<const sk_f32x4*>(part + (part0 ^ (k + i)) * slot_bytes + ((e_own * TL + tw) * 64 + lane_p) * 16);
                            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                            for (int i = 0; i < PARTS; ++i)
#pragma unroll
                                for (int tw = 0; tw < N; ++tw)
#pragma unroll
                                    for (int c = 0; c < 4; ++c) sum[tw][c] += p[i][tw][c];
                        };
                        if constexpr (FAST || DENSE) {
                            if (WK == 2) add_parts(std::integral_constant<int, 2>{}, 0);
                            else
                                for (int k = 0; k < WK; k += 4) add_parts(std::integral_constant<int, 4>{}, k);
                        } else {   // the general epilogue has no registers to spare: one wave's sums at a time
                            for (int k = 0; k < WK; ++k) {
#pragma unroll
                                for (int tw = 0; tw < N; ++tw)
                                    sum[tw] += *reinterpret_cast<const sk_f32x4*>(part + (part0 ^ k) * slot_bytes + ((e_own * TL + tw) * 64 + lane_p) * 16);
                            }
                        }
                    };
                    // One of the wave's quads, with its sums.
                    auto run_quad = [&](int e_own, const sk_f32x4 (&sum)[TT]) __attribute__((always_inline)) {
                        const int j8 = oc_e * TG + e_own;
                        float xq[TT][4];
#pragma unroll
                        for (int tw = 0; tw < TT; ++tw)
#pragma unroll
                            for (int k = 0; k < 4; ++k) xq[tw][k] = sum[tw][k];
                        if constexpr (FAST) {
                            if (e_own != e_first && g.res_layout >= 0 && TT > 1) {
#pragma unroll
                                for (int tw = 0; tw < TT; ++tw) rb[tw] = fast_res(tb + min(tw, t_count - 1), j8);
                            }
                            const float start[4] = {v0[0], v0[1], v0[2], v0[3]};
                            if (e_own + WK < 4) fast_v0(j8 + WK, v0);
                            if (lean && (g.res_layout < 0 || TT >= 3)) {
                                const uint32_t quiet = g.res_layout < 0 ? lean_quad(xq, rb, std::false_type{}) : lean_quad(xq, rb, std::true_type{});
                                if constexpr (POOL) fast_store4_pooled(j8, quiet);
                                else if constexpr (TT == 3) fast_store(tb, 3, j8, quiet);
                                else fast_store4(j8, quiet, -1, 0u);
                            } else {
                                fast_quad(j8, xq, rb, g.res_layout >= 0, start);
                            }
                        } else if constexpr (DENSE) {
                            const DenseIn now = in;
                            if (e_own + WK < 4) dense_request(j8 + WK, in);
                            dense_quad(j8, xq, now);
                        } else {
                            general_quad(j8, xq);
                        }
                    };
                    if constexpr (TT > 4) {
                        sk_f32x4 sums[2][TT];    // (a wave of two finishes two quads, one of four or eight at most one)
                        if (e_first < 4) gather(std::integral_constant<int, TL>{}, e_first, sums[0]);
                        if (WK == 2) gather(std::integral_constant<int, TL>{}, e_first + 2, sums[1]);
                        __syncthreads();
                        park(std::integral_constant<int, TL>{}, std::integral_constant<int, TT>{});
                        __syncthreads();
                        if (e_first < 4) {
                            gather(std::integral_constant<int, TT - TL>{}, e_first, sums[0] + TL);
                            run_quad(e_first, sums[0]);
                        }
                        if (WK == 2) {
                            gather(std::integral_constant<int, TT - TL>{}, e_first + 2, sums[1] + TL);
                            run_quad(e_first + 2, sums[1]);
                        }
                    } else {
                        for (int e_own = e_first; e_own < 4; e_own += WK) {
                            sk_f32x4 sum[TT];
                            gather(std::integral_constant<int, TT>{}, e_own, sum);
                            run_quad(e_own, sum);
                        }
                    }
                }
            }
#undef SNNF_SPK_PARK_QUAD
            if constexpr (SK) __syncthreads();   // the partial sums are read before the next window's staging overwrites them
        }
    }
}

template <typename XT, int TT, int IN>
int launch_conv_spk_variant(const SpkLaunch& L) {
    auto run = [&](auto kernel) -> int {
        if (const int rc = reserve_lds(reinterpret_cast<const void*>(kernel), L.lds_bytes, "snnf_conv_lif_blocked"); rc != SNNF_OK) return rc;
        kernel<<<dim3(L.grid), kSpkWaves * 64, L.lds_bytes, L.stream>>>(L.xs, L.residuals, L.g, L.wpacked, L.bias, L.v_start,
                                                                        static_cast<unsigned char*>(L.out), L.v_store, L.lif, L.wpacked2, L.bias2, L.v_scratch, L.lo_flags);
        return check_launch("snnf_conv_lif_blocked");
    };
    if constexpr (IN == SNNF_LAYOUT_C8) {
        if (L.dense_epilogue) {
            if (L.g.narrow) return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, IN, true, false, false, false, true, true>) : run(conv_spk_kernel<XT, TT, IN, false, false, false, false, true, true>);
            return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, IN, true, false, false, false, false, true>) : run(conv_spk_kernel<XT, TT, IN, false, false, false, false, false, true>);
        }
    }
    if constexpr (TT >= 3) {
        if (L.fast_epilogue && L.multi_window) {
            if (L.g.narrow) return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, IN, true, true, false, false, true, false, true>) : run(conv_spk_kernel<XT, TT, IN, false, true, false, false, true, false, true>);
            return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, IN, true, true, false, false, false, false, true>) : run(conv_spk_kernel<XT, TT, IN, false, true, false, false, false, false, true>);
        }
    }
    if (L.g.narrow) {
        if (L.g.wk_log2 == 0) return L.fast_epilogue ? run(conv_spk_kernel<XT, TT, IN, false, true, false, false, true>) : run(conv_spk_kernel<XT, TT, IN, false, false, false, false, true>);
        return L.fast_epilogue ? run(conv_spk_kernel<XT, TT, IN, true, true, false, false, true>) : run(conv_spk_kernel<XT, TT, IN, true, false, false, false, true>);
    }
    if (L.fast_epilogue) return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, IN, true, true>) : run(conv_spk_kernel<XT, TT, IN, false, true>);
    return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, IN, true, false>) : run(conv_spk_kernel<XT, TT, IN, false, false>);
}

// fp32 tensors as two bf16 terms each.
template <int TT>
int launch_conv_spk_split(const SpkLaunch& L) {
    auto run = [&](auto kernel) -> int {
        if (const int rc = reserve_lds(reinterpret_cast<const void*>(kernel), L.lds_bytes, "snnf_conv_lif"); rc != SNNF_OK) return rc;
        kernel<<<dim3(L.grid), kSpkWaves * 64, L.lds_bytes, L.stream>>>(L.xs, L.residuals, L.g, L.wpacked, L.bias, L.v_start,
                                                                        static_cast<unsigned char*>(L.out), L.v_store, L.lif, L.wpacked2, L.bias2, L.v_scratch, L.lo_flags);
        return check_launch("snnf_conv_lif");
    };
    constexpr int C = SNNF_LAYOUT_C8;
    if (L.dense_epilogue) return L.g.wk_log2 > 0 ? run(conv_spk_kernel<float, TT, C, true, false, false, false, true, true>) : run(conv_spk_kernel<float, TT, C, false, false, false, false, true, true>);
    return L.g.wk_log2 > 0 ? run(conv_spk_kernel<float, TT, C, true, false, false, false, true>) : run(conv_spk_kernel<float, TT, C, false, false, false, false, true>);
}

// The variants whose spikes leave as 2x2 average pools: straight-line epilogue, four steps (side by side, or of one frame).
template <typename XT, int IN>
int launch_conv_spk_pooled(const SpkLaunch& L, int tt) {
    auto run = [&](auto kernel) -> int {
        if (const int rc = reserve_lds(reinterpret_cast<const void*>(kernel), L.lds_bytes, "snnf_conv_lif_blocked_avgpool"); rc != SNNF_OK) return rc;
        kernel<<<dim3(L.grid), kSpkWaves * 64, L.lds_bytes, L.stream>>>(L.xs, L.residuals, L.g, L.wpacked, L.bias, L.v_start,
                                                                        static_cast<unsigned char*>(L.out), L.v_store, L.lif, L.wpacked2, L.bias2, L.v_scratch, L.lo_flags);
        return check_launch("snnf_conv_lif_blocked_avgpool");
    };
    if (tt == 4 && L.g.narrow) return run(conv_spk_kernel<XT, 4, IN, true, true, false, true, true>);
    if (tt == 4) return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, 4, IN, true, true, false, true>) : run(conv_spk_kernel<XT, 4, IN, false, true, false, true>);
    return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, 1, IN, true, true, false, true>) : run(conv_spk_kernel<XT, 1, IN, false, true, false, true>);
}

// The variants that read the network's input as it is: one dense frame of at most 8 channels for all timesteps, hence one channel group in one stage, which
// waves can't share.
template <typename XT>
int launch_conv_spk_frame(const SpkLaunch& L, bool pooled) {
    auto run = [&](auto kernel) -> int {
        if (const int rc = reserve_lds(reinterpret_cast<const void*>(kernel), L.lds_bytes, "snnf_conv_lif_blocked"); rc != SNNF_OK) return rc;
        kernel<<<dim3(L.grid), kSpkWaves * 64, L.lds_bytes, L.stream>>>(L.xs, L.residuals, L.g, L.wpacked, L.bias, L.v_start,
                                                                        static_cast<unsigned char*>(L.out), L.v_store, L.lif, L.wpacked2, L.bias2, L.v_scratch, L.lo_flags);
        return check_launch("snnf_conv_lif_blocked");
    };
    constexpr int D = SNNF_LAYOUT_NCHW;
    if (L.dense_epilogue) {
        if (L.g.narrow) return run(conv_spk_kernel<XT, 1, D, false, false, false, false, true, true>);
        return run(conv_spk_kernel<XT, 1, D, false, false, false, false, false, true>);
    }
    if (L.g.narrow) {
        if (pooled) return run(conv_spk_kernel<XT, 1, D, false, true, false, true, true>);
        return L.fast_epilogue ? run(conv_spk_kernel<XT, 1, D, false, true, false, false, true>) : run(conv_spk_kernel<XT, 1, D, false, false, false, false, true>);
    }
    if (pooled) return run(conv_spk_kernel<XT, 1, D, false, true, false, true>);
    return L.fast_epilogue ? run(conv_spk_kernel<XT, 1, D, false, true>) : run(conv_spk_kernel<XT, 1, D, false, false>);
}

// The variants with a projection shortcut in the accumulators: bit-packed inputs, three or four timesteps side by side.
template <typename XT, int TT>
int launch_conv_spk_shortcut(const SpkLaunch& L) {
    auto run = [&](auto kernel) -> int {
        if (const int rc = reserve_lds(reinterpret_cast<const void*>(kernel), L.lds_bytes, "snnf_conv_lif_blocked_shortcut"); rc != SNNF_OK) return rc;
        kernel<<<dim3(L.grid), kSpkWaves * 64, L.lds_bytes, L.stream>>>(L.xs, L.residuals, L.g, L.wpacked, L.bias, L.v_start,
                                                                        static_cast<unsigned char*>(L.out), L.v_store, L.lif, L.wpacked2, L.bias2, L.v_scratch, L.lo_flags);
        return check_launch("snnf_conv_lif_blocked_shortcut");
    };
    constexpr int B = SNNF_LAYOUT_BITS;
    if (L.fast_epilogue && L.multi_window) {
        if (L.g.narrow) return run(conv_spk_kernel<XT, TT, B, true, true, true, false, true, false, true>);
        return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, B, true, true, true, false, false, false, true>) : run(conv_spk_kernel<XT, TT, B, false, true, true, false, false, false, true>);
    }
    if (L.g.narrow) return L.fast_epilogue ? run(conv_spk_kernel<XT, TT, B, true, true, true, false, true>) : run(conv_spk_kernel<XT, TT, B, true, false, true, false, true>);
    if (L.fast_epilogue) return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, B, true, true, true>) : run(conv_spk_kernel<XT, TT, B, false, true, true>);
    return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, B, true, false, true>) : run(conv_spk_kernel<XT, TT, B, false, false, true>);
}

// Five or six timesteps in one window: narrow tiles whose K several waves share.
template <typename XT, int TT, int IN>
int launch_conv_spk_long(const SpkLaunch& L) {
    auto run = [&](auto kernel) -> int {
        if (const int rc = reserve_lds(reinterpret_cast<const void*>(kernel), L.lds_bytes, "snnf_conv_lif_blocked"); rc != SNNF_OK) return rc;
        kernel<<<dim3(L.grid), kSpkWaves * 64, L.lds_bytes, L.stream>>>(L.xs, L.residuals, L.g, L.wpacked, L.bias, L.v_start,
                                                                        static_cast<unsigned char*>(L.out), L.v_store, L.lif, L.wpacked2, L.bias2, L.v_scratch, L.lo_flags);
        return check_launch("snnf_conv_lif_blocked");
    };
    if constexpr (IN == SNNF_LAYOUT_C8) {
        if (L.dense_epilogue) return run(conv_spk_kernel<XT, TT, IN, true, false, false, false, true, true>);
    }
    return L.fast_epilogue ? run(conv_spk_kernel<XT, TT, IN, true, true, false, false, true>) : run(conv_spk_kernel<XT, TT, IN, true, false, false, false, true>);
}

// Dense frames per timestep around the dense epilogue (fp32: narrow tiles alone).
template <typename XT, int TT>
int launch_conv_spk_steps(const SpkLaunch& L) {
    auto run = [&](auto kernel) -> int {
        if (const int rc = reserve_lds(reinterpret_cast<const void*>(kernel), L.lds_bytes, "snnf_conv_lif"); rc != SNNF_OK) return rc;
        kernel<<<dim3(L.grid), kSpkWaves * 64, L.lds_bytes, L.stream>>>(L.xs, L.residuals, L.g, L.wpacked, L.bias, L.v_start,
                                                                        static_cast<unsigned char*>(L.out), L.v_store, L.lif, L.wpacked2, L.bias2, L.v_scratch, L.lo_flags);
        return check_launch("snnf_conv_lif");
    };
    if constexpr (TT > 4) {
        return run(conv_spk_kernel<XT, TT, kSpkSteps, true, false, false, false, true, true>);
    } else {
        if (std::is_same<XT, float>::value || L.g.narrow) return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, kSpkSteps, true, false, false, false, true, true>) : run(conv_spk_kernel<XT, TT, kSpkSteps, false, false, false, false, true, true>);
        if constexpr (!std::is_same<XT, float>::value)
            return L.g.wk_log2 > 0 ? run(conv_spk_kernel<XT, TT, kSpkSteps, true, false, false, false, false, true>) : run(conv_spk_kernel<XT, TT, kSpkSteps, false, false, false, false, false, true>);
    }
}

template <typename XT, int IN>
int launch_conv_spk_tt(const SpkLaunch& L, int tt) {
    if (tt == 4) return launch_conv_spk_variant<XT, 4, IN>(L);
    if (tt == 2) return launch_conv_spk_variant<XT, 2, IN>(L);
    return launch_conv_spk_variant<XT, 1, IN>(L);
}

// One launcher per activation dtype and input layout (each in its own translation unit, so that they compile in parallel).
int launch_conv_spk_bf16_bits(const SpkLaunch& L, int tt);
int launch_conv_spk_bf16_long(const SpkLaunch& L);
int launch_conv_spk_bf16_steps(const SpkLaunch& L, int tt);
int launch_conv_spk_bf16_three(const SpkLaunch& L);
int launch_conv_spk_bf16_three_shortcut(const SpkLaunch& L);
int launch_conv_spk_bf16_c8(const SpkLaunch& L, int tt);
int launch_conv_spk_f16_bits(const SpkLaunch& L, int tt);
int launch_conv_spk_f16_long(const SpkLaunch& L);
int launch_conv_spk_f16_steps(const SpkLaunch& L, int tt);
int launch_conv_spk_f16_three(const SpkLaunch& L);
int launch_conv_spk_f16_three_shortcut(const SpkLaunch& L);
int launch_conv_spk_f16_c8(const SpkLaunch& L, int tt);
int launch_conv_spk_bf16_shortcut(const SpkLaunch& L);
int launch_conv_spk_f16_shortcut(const SpkLaunch& L);
int launch_conv_spk_bf16_pooled(const SpkLaunch& L, int tt);
int launch_conv_spk_f16_pooled(const SpkLaunch& L, int tt);
int launch_conv_spk_bf16_frame(const SpkLaunch& L, bool pooled);
int launch_conv_spk_f16_frame(const SpkLaunch& L, bool pooled);
int launch_conv_spk_f32(const SpkLaunch& L, int tt);
int launch_conv_spk_f32_steps(const SpkLaunch& L, int tt);

}  // namespace snnf
