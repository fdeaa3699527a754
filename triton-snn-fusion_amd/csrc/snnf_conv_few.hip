// Convolution + bias (+ residual) + LIF on the internal layouts for layers of few output pixels (deep layers of small batches): such a launch
// lasts as long as the chain of one of its workgroups, most of the chip has nothing to do, and neither memory nor the matrix cores are busy.
//
// Against conv_spk_kernel's tiles of 32 channels x 32 pixels, whose workgroups run 36 steps of four 32x32 products per wave at 512 -> 512 and read 295 KB of
// weights each, a workgroup here has 16 channels and 4, 8 or 16 pixels: up to sixteen times the workgroups, a half of the weights each, and products of
// 16x16 whose 16 columns are pixels AND timesteps (column = timestep x PX + pixel), so that none is empty when a plane has four pixels.
//   * The workgroup stages the halo of its pixels for all channel groups, meets once, and every wave multiplies an eighth of
//     the (tap, channel pair) list. A matrix step takes two entries of that list, any two: each lane adds its entry's offset to its pixel's.
//   * A wave's weights depend on nothing: up to 18 fragments are requested behind the first activations and travel while those are staged.
//   * Partial sums meet in LDS; then a lane per neuron adds the eight, in the order of the waves, and runs its timesteps with the general neuron, any initial
//     membrane, residual and number of windows (the membrane stays in a register). There are so few neurons that one path does for all.
// What is left of a launch of 256 -> 256 at 8^2, one image (7.4 us, of which an empty launch is about 4): set-up, one trip to memory for spikes and weights, nine steps, the
// exchange. 18 fragments requested where nine are there cost 0.5 us, the weights in front of the spikes as much where both are many.
#include <algorithm>

#include "snnf_conv_few.h"

namespace snnf {
namespace {

constexpr int kFewWaves = 8;
constexpr int kFewThreads = kFewWaves * 64;
constexpr int kFewTableEntries = 2 * 18;                         // (tap, channel pair) entries of a block, at most
constexpr int kFewTableBytes = kFewWaves * kFewTableEntries * 16;
constexpr int kFewBitsBytes = 4 * 4 * 8;                         // spikes of a window: four steps x 256 neurons
constexpr uint32_t kFewOutside = 0x80000000u;                    // offset of a weight that is not there: the range check answers zero
constexpr int kFewResTable = static_cast<int>(sizeof(StepPtrs));

typedef float fw_f32x4 __attribute__((ext_vector_type(4)));

struct FewArgs {      // the kernel's arguments as they lie in the kernel-argument segment
    StepPtrs xs, residuals;
    FewGeom g;
    const void *wpacked, *bias, *v_start, *out, *v_store;
    LifParams lif;
};

template <bool F16>
__device__ __forceinline__ fw_f32x4 few_mfma(sk_u32x4 a, sk_u32x4 b, fw_f32x4 c) {
    if constexpr (F16) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(sk_f16x8, a), __builtin_bit_cast(sk_f16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sk_bf16x8, a), __builtin_bit_cast(sk_bf16x8, b), c, 0, 0, 0);
}

// NF: column fragments of 16 (timesteps x pixels of a workgroup / 16). BLOCK: weight fragments of a wave in flight, all of which are
// requested: those beyond its last cost no traffic, but their addresses (18 for the 9 of 256 channels 0.5 us a launch).
// The two pointer tables MUST be the first two kernel parameters.
template <typename XT, int IN, int NF, int BLOCK>
__global__ __launch_bounds__(kFewThreads, 2) void conv_few_kernel(const StepPtrs xs, const StepPtrs residuals, const FewGeom g, const void* wpacked,
                                                                  const float* __restrict__ bias, const void* v_start, unsigned char* out, void* v_store,
                                                                  const LifParams lif) {
    extern __shared__ __align__(16) unsigned char lds[];
    // Every cache line of the arguments is touched once, in one round trip (as in conv_spk_kernel).
    {
        auto ka = __builtin_amdgcn_kernarg_segment_ptr();
        static_assert(sizeof(FewArgs) >= 0x200 + 4 && sizeof(FewArgs) <= 0x240, "the lines below are those of the explicit arguments");
        uint32_t d0, d1, d2, d3, d4, d5, d6, d7;
        asm volatile(
            "s_load_dword %0, %8, 0x40\n\ts_load_dword %1, %8, 0x80\n\ts_load_dword %2, %8, 0xc0\n\ts_load_dword %3, %8, 0x100\n\t"
            "s_load_dword %4, %8, 0x140\n\ts_load_dword %5, %8, 0x180\n\ts_load_dword %6, %8, 0x1c0\n\ts_load_dword %7, %8, 0x200\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&s"(d0), "=&s"(d1), "=&s"(d2), "=&s"(d3), "=&s"(d4), "=&s"(d5), "=&s"(d6), "=&s"(d7)
            : "s"(ka));
    }
    __builtin_amdgcn_sched_barrier(0);
    constexpr bool F16 = dtype_of<XT>::value == SNNF_F16;
    constexpr uint32_t ONE = F16 ? 0x3c00u : 0x3f80u;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int quarter = lane >> 4, col = lane & 15;
    unsigned char* const table = lds + wave * (kFewTableEntries * 16);
    uint64_t* const bits = reinterpret_cast<uint64_t*>(lds + kFewTableBytes);
    unsigned char* const part = lds + kFewTableBytes + kFewBitsBytes;
    constexpr int kStage = kFewTableBytes + kFewBitsBytes + kFewWaves * NF * 1024;
    const int PX = 1 << g.px_log2;
    const int TT = NF * 16 >> g.px_log2;

    // Workgroups of one channel tile have the same remainder modulo eight where the tiles are a multiple of that: one XCD reads their weights.
    const int patch = sk_div(static_cast<int>(blockIdx.x), g.d_oc_tiles);
    const int oc0 = (static_cast<int>(blockIdx.x) - patch * g.oc_tiles) * 16;
    const int imgg = sk_div(patch, g.d_patches_img);
    const int in_img = patch - imgg * g.patches_img;
    const int py = sk_div(in_img, g.d_patches_x);
    const int n0 = imgg * g.PI, oh0 = py * g.PR, ow0 = (in_img - py * g.patches_x) * g.PC;
    const int ih_lo = oh0 * g.sh - g.ph, iw_lo = ow0 * g.sw - g.pw;

    // Where a pixel of the workgroup lies: image, row and column inside the patch.
    auto pixel_at = [&](int p, int& pi, int& pr, int& pc) __attribute__((always_inline)) {
        pi = sk_div(p, g.d_ppx);
        const int rem = p - pi * (g.PR * g.PC);
        pr = sk_div(rem, g.d_PC);
        pc = rem - pr * g.PC;
        return pi < g.PI;
    };

    // ---- matrix view: this lane's columns, as offsets into the staged halo.
    const int tile_t = g.Gs * g.region * 16;
    uint32_t col_off[NF];
    {
        int pi, pr, pc;
        const bool live = pixel_at(col & (PX - 1), pi, pr, pc);      // (columns without a pixel read pixel 0 and are never stored)
        const int at = live ? ((pi * g.RR + pr * g.sh) * g.RC + pc * g.sw) * 16 : 0;
#pragma unroll
        for (int f = 0; f < NF; ++f) col_off[f] = static_cast<uint32_t>(kStage + at + ((f * 16 + col) >> g.px_log2) * tile_t);
    }
    const auto wrsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(wpacked), 0, g.weight_bytes, 0x00027000);
    // Two 16-row halves of a packed fragment: this workgroup's rows, the k-slot of the lane's quarter.
    const uint32_t w_lane = static_cast<uint32_t>((oc0 >> 5) * g.frag_bytes + (((quarter & 1) * 32) + (oc0 & 16) + col) * 16);

    // ---- neuron view: channel oc0 + 4 cq + ci of pixel p.
    const int ci = tid & 3, np = (tid >> 2) & (PX - 1), cq = tid >> (2 + g.px_log2);
    const int ch = oc0 + 4 * cq + ci;
    int ni, nr, nc;
    const bool np_live = pixel_at(np, ni, nr, nc);
    const int nn = n0 + ni, noh = oh0 + nr, now = ow0 + nc;
    const bool neuron = cq < 4 && np_live && ch < g.Cout && nn < g.N && noh < g.Ho && now < g.Wo;
    const uint32_t at_nchw = neuron ? static_cast<uint32_t>(((nn * g.Cout + ch) * g.Ho + noh) * g.Wo + now) : 0u;
    const uint32_t at_bits = neuron ? static_cast<uint32_t>(((nn * g.C8out + (ch >> 3)) * g.Ho + noh) * g.Wo + now) : 0u;
    const bool half_tau = lif.charge_mode == CHARGE_SCALE && lif.inv_tau == 0.5f && !lif.soft_reset;
    float v = 0.0f, b = 0.0f;
    if (neuron) {
        b = bias[ch];
        const void* const vp = g.v_in_place ? v_store : v_start;
        if (vp != nullptr) v = g.v16 ? to_float(static_cast<const XT*>(vp)[at_nchw]) : static_cast<const float*>(vp)[at_nchw];
    }

    for (int t0 = 0; t0 < g.T; t0 += TT) {
        const int steps = min(TT, g.T - t0);
        fw_f32x4 acc[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[f] = fw_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        uint32_t res[4] = {0u, 0u, 0u, 0u};
        const int pairs = (g.Gs >> 1) * g.taps;
        const int share = (pairs + kFewWaves - 1) / kFewWaves;
        const int first = wave * share;
        const int mine = max(0, min(share, pairs - first));           // entries of this wave

        // Entries from `base` on of this wave: lane i writes entry i. No barrier: a wave's LDS accesses are in order.
        auto make_table = [&](int base) __attribute__((always_inline)) {
            if (lane < 2 * BLOCK) {
                const bool in = base + lane < mine;
                const int e = in ? first + base + lane : 0;
                const int gp = sk_div(e, g.d_taps);
                const int tap = e - gp * g.taps;
                const int kh = (tap * g.kw_mul) >> 16;
                const uint32_t w = in ? static_cast<uint32_t>(((gp >> g.gph_log2) * g.npairs + (tap << g.gph_log2) + (gp & ((1 << g.gph_log2) - 1))) * kFragBytes) : kFewOutside;
                const uint32_t at = static_cast<uint32_t>((2 * gp * g.region + kh * g.RC + (tap - kh * g.KW)) * 16);
                const sk_u32x4 entry = {w, at, w, at + static_cast<uint32_t>(g.region * 16)};
                *reinterpret_cast<sk_u32x4*>(table + lane * 16) = entry;
            }
            __builtin_amdgcn_wave_barrier();
        };
        // What step s of a block means to this lane: its weight's offset and its operand's.
        auto entry_of = [&](int s) __attribute__((always_inline)) {
            return *reinterpret_cast<const Pack<uint32_t, 2>*>(table + (2 * s + (quarter >> 1)) * 16 + (quarter & 1) * 8);
        };
        sk_u32x4 w[BLOCK];
        auto load_weights = [&](int base) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < BLOCK; ++s)          // (all of them, also beyond the last, which cost no traffic: the number in flight is known at every wait)
                w[s] = __builtin_bit_cast(sk_u32x4, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, w_lane + entry_of(s).v[0], 0, 0));
        };
        if (g.res_layout >= 0 && neuron) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i < steps) {
                    const void* const rp = sk_kernarg_ptr(kFewResTable, t0 + i);
                    res[i] = g.res_layout == SNNF_LAYOUT_BITS ? static_cast<const unsigned char*>(rp)[at_bits] : static_cast<const uint16_t*>(rp)[at_nchw];
                }
            }
        }

        // ---- the halo of the patch: all channel groups x all steps of the window, four items of a thread in flight. The first ones are requested in front
        // of the weights, so that nothing is waited for behind those.
        const int items = g.Gs * g.region;
        // (Of dense frames one item, from eight loads of a channel each.)
        constexpr int BATCH = IN == SNNF_LAYOUT_BITS ? 4 : (IN == kSpkSteps ? 1 : 2);
        uint32_t okb = 0;
        typename std::conditional<IN == SNNF_LAYOUT_C8, sk_u32x4, uint32_t>::type raw[4][IN == kSpkSteps ? 8 : BATCH];
        const int in_stride = IN == kSpkSteps ? g.Cin : g.C8in, in_group = IN == kSpkSteps ? 8 : 1;
        int left = 8;                                  // channels of a dense item's group, and beyond
        auto request = [&](int e0) __attribute__((always_inline)) {
            uint32_t idx[BATCH];
            okb = 0;
#pragma unroll
            for (int j = 0; j < BATCH; ++j) {
                const int e = min(e0 + j * kFewThreads, items - 1);
                const int gq = sk_div(e, g.d_region);
                const int rem = e - gq * g.region;
                const int ii = sk_div(rem, g.d_rrrc);
                const int rem2 = rem - ii * (g.RR * g.RC);
                const int r = sk_div(rem2, g.d_RC);
                const int ih = ih_lo + r, iw = iw_lo + rem2 - r * g.RC;
                const bool ok = static_cast<bool>(static_cast<int>(n0 + ii < g.N) & static_cast<int>(gq < g.C8in) & static_cast<int>(static_cast<unsigned>(ih) < static_cast<unsigned>(g.H)) &
                                                  static_cast<int>(static_cast<unsigned>(iw) < static_cast<unsigned>(g.W)));
                idx[j] = ok ? static_cast<uint32_t>((((n0 + ii) * in_stride + gq * in_group) * g.H + ih) * g.W + iw) : 0u;
                okb |= ok ? 1u << j : 0u;
                if constexpr (IN == kSpkSteps) left = g.Cin - (ok ? gq * 8 : 0);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (t < steps) {
                    if constexpr (IN == SNNF_LAYOUT_BITS) {
                        const sk_global_bytes src = (sk_global_bytes)sk_kernarg_ptr(0, t0 + t);
#pragma unroll
                        for (int j = 0; j < BATCH; ++j) raw[t][j] = src[idx[j]];
                    } else if constexpr (IN == kSpkSteps) {
                        const uint16_t* const src = static_cast<const uint16_t*>(sk_kernarg_ptr(0, t0 + t));
#pragma unroll
                        for (int k = 0; k < 8; ++k) raw[t][k] = src[idx[0] + static_cast<uint32_t>(min(k, left - 1) * (g.H * g.W))];
                    } else {
                        const sk_u32x4* const src = static_cast<const sk_u32x4*>(sk_kernarg_ptr(0, t0 + t));
#pragma unroll
                        for (int j = 0; j < BATCH; ++j) raw[t][j] = src[idx[j]];
                    }
                }
            }
        };
        auto put = [&](int e0) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (t < steps) {
#pragma unroll
                    for (int j = 0; j < BATCH; ++j) {
                        const bool ok = ((okb >> j) & 1u) != 0u;
                        sk_u32x4 d;
                        if constexpr (IN == SNNF_LAYOUT_BITS) {
                            const uint32_t keep = ok ? 0x0c000c00u : 0x0c0c0c0cu;   // byte 0 at bytes 0 and 2, or zeros
                            d = sk_expand_bits<ONE>(__builtin_amdgcn_perm(raw[t][j], raw[t][j], keep));
                        } else if constexpr (IN == kSpkSteps) {
#pragma unroll
                            for (int k = 0; k < 4; ++k)
                                d[k] = (ok && 2 * k < left ? raw[t][2 * k] : 0u) | (ok && 2 * k + 1 < left ? raw[t][2 * k + 1] << 16 : 0u);
                        } else {
#pragma unroll
                            for (int k = 0; k < 4; ++k) d[k] = ok ? raw[t][j][k] : 0u;
                        }
                        if (e0 + j * kFewThreads < items) *reinterpret_cast<sk_u32x4*>(lds + kStage + t * tile_t + (e0 + j * kFewThreads) * 16) = d;
                    }
                }
            }
        };
        request(tid);
        __builtin_amdgcn_sched_barrier(0);
        make_table(0);
        load_weights(0);
        __builtin_amdgcn_sched_barrier(0);
        if (t0 > 0) __syncthreads();                   // the operands and sums of the window before have been read
        for (int e0 = tid; e0 < items; e0 += BATCH * kFewThreads) {
            if (e0 != tid) request(e0);
            put(e0);
        }
        __syncthreads();

        // ---- this wave's entries, two a step.
        for (int base = 0; base < mine; base += 2 * BLOCK) {
            if (base > 0) {
                __builtin_amdgcn_wave_barrier();
                make_table(base);
                load_weights(base);
            }
            const int n = (mine - base + 1) >> 1;
            const bool odd = ((mine - base) & 1) != 0;
#pragma unroll
            for (int s = 0; s < BLOCK; ++s) {
                if (s < n) {
                    const uint32_t at = entry_of(s).v[1];
                    sk_u32x4 x[NF];
#pragma unroll
                    for (int f = 0; f < NF; ++f) x[f] = *reinterpret_cast<const sk_u32x4*>(lds + col_off[f] + at);
                    if (odd && s == n - 1) {                     // the second entry of the last step is not there: zeros, whatever lies in LDS
#pragma unroll
                        for (int f = 0; f < NF; ++f)
#pragma unroll
                            for (int k = 0; k < 4; ++k) x[f][k] = quarter >= 2 ? 0u : x[f][k];
                    }
#pragma unroll
                    for (int f = 0; f < NF; ++f) acc[f] = few_mfma<F16>(w[s], x[f], acc[f]);
                }
            }
        }

        // ---- partial sums: [wave][fragment][lane] x 4 channels.
#pragma unroll
        for (int f = 0; f < NF; ++f) *reinterpret_cast<fw_f32x4*>(part + ((wave * NF + f) * 64 + lane) * 16) = acc[f];
        __syncthreads();
        if (wave * 64 < 16 * PX) {
            float x[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int c = i * PX + np;                            // column
                const unsigned char* const at = part + min(((c >> 4) * 64 + cq * 16 + (c & 15)) * 16, NF * 1024 - 16) + ci * 4;
                x[i] = b;
                if (i < TT) {
                    float p[kFewWaves];
#pragma unroll
                    for (int k = 0; k < kFewWaves; ++k) p[k] = *reinterpret_cast<const float*>(at + k * NF * 1024);
#pragma unroll
                    for (int k = 0; k < kFewWaves; ++k) x[i] += p[k];
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (i < steps) {
                    if (g.res_layout == SNNF_LAYOUT_BITS) x[i] += static_cast<float>((res[i] >> (ch & 7)) & 1u);
                    else if (g.res_layout >= 0) x[i] += to_float(XT{static_cast<uint16_t>(res[i])});
                    bool fired;
                    if (half_tau) {                                   // (as in conv_spk_kernel: one rounding, with a hard reset)
                        const float h = (v + x[i]) * 0.5f;
                        fired = h >= lif.v_threshold;
                        v = fired ? lif.v_reset : h;
                    } else {
                        fired = lif_step(x[i], v, lif);
                    }
                    fired = fired && neuron;
                    if (g.out_layout == SNNF_LAYOUT_NCHW) {
                        if (neuron) reinterpret_cast<XT*>(out + static_cast<int64_t>(t0 + i) * g.out_step_stride)[at_nchw] = spike_value<XT>(fired);
                    } else {
                        const uint64_t m = __builtin_amdgcn_ballot_w64(fired);
                        if (lane == 0) bits[i * 4 + wave] = m;
                    }
                }
            }
        }
        if (g.out_layout != SNNF_LAYOUT_NCHW) {
            __syncthreads();
            // The window's spikes as a string of bits, 4 channels of a pixel side by side: bit 4 (cq * PX + p) + ci of step i.
            const unsigned char* const string = reinterpret_cast<const unsigned char*>(bits);
            auto group_byte = [&](int i, int half, int p) __attribute__((always_inline)) -> uint32_t {
                const int lo = 2 * half * PX + p, hi = lo + PX;       // nibbles
                return ((string[i * 32 + (lo >> 1)] >> (4 * (lo & 1))) & 15u) | (((string[i * 32 + (hi >> 1)] >> (4 * (hi & 1))) & 15u) << 4);
            };
            const int p = tid & (PX - 1), half = (tid >> g.px_log2) & 1, i = tid >> (1 + g.px_log2);
            int pi, pr, pc;
            const bool live = pixel_at(p, pi, pr, pc);
            const int n = n0 + pi, oh = oh0 + pr, ow = ow0 + pc, j8 = (oc0 >> 3) + half;
            if (i < steps && live && n < g.N && oh < g.Ho && ow < g.Wo && j8 < g.C8out) {
                unsigned char* const to = out + static_cast<int64_t>(t0 + i) * g.out_step_stride;
                if (g.pool == 0) {
                    to[((n * g.C8out + j8) * g.Ho + oh) * g.Wo + ow] = static_cast<unsigned char>(group_byte(i, half, p));
                } else if (((pr | pc) & 1) == 0) {                    // the upper left pixel of a window of four
                    const uint32_t a0 = group_byte(i, half, p), a1 = group_byte(i, half, p + 1), a2 = group_byte(i, half, p + g.PC), a3 = group_byte(i, half, p + g.PC + 1);
                    Pack<XT, 8> o;
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        o.v[k] = from_float<XT>(0.25f * static_cast<float>(((a0 >> k) & 1u) + ((a1 >> k) & 1u) + ((a2 >> k) & 1u) + ((a3 >> k) & 1u)));
                    *reinterpret_cast<Pack<XT, 8>*>(to + (static_cast<int64_t>((n * g.C8out + j8) * (g.Ho >> 1) + (oh >> 1)) * (g.Wo >> 1) + (ow >> 1)) * 16) = o;
                }
            }
        }
    }
    if (neuron && v_store != nullptr) {
        if (g.v16) static_cast<XT*>(v_store)[at_nchw] = from_float<XT>(v);
        else static_cast<float*>(v_store)[at_nchw] = v;
    }
}

template <typename XT, int IN>
int launch(const FewLaunch& L) {
    auto run = [&](auto kernel) -> int {
        if (const int rc = reserve_lds(reinterpret_cast<const void*>(kernel), L.lds_bytes, "snnf_conv_lif_blocked"); rc != SNNF_OK) return rc;
        kernel<<<dim3(L.g.grid), kFewThreads, L.lds_bytes, L.stream>>>(L.xs, L.residuals, L.g, L.wpacked, L.bias, L.v_start, static_cast<unsigned char*>(L.out), L.v_store, L.lif);
        return check_launch("snnf_conv_lif_blocked");
    };
    const int share = ((L.g.Gs >> 1) * L.g.taps + kFewWaves - 1) / kFewWaves;      // entries of a wave
    auto block = [&](auto frags) -> int {
        constexpr int NF = decltype(frags)::value;
        return share <= 10 ? run(conv_few_kernel<XT, IN, NF, 5>) : (share <= 18 ? run(conv_few_kernel<XT, IN, NF, 9>) : run(conv_few_kernel<XT, IN, NF, 18>));
    };
    return L.g.frags == 4 ? block(std::integral_constant<int, 4>{}) : (L.g.frags == 2 ? block(std::integral_constant<int, 2>{}) : block(std::integral_constant<int, 1>{}));
}

}  // namespace

// Where the kernel is the faster one (us, conv_spk_kernel / here, on bit-packed spikes with a residual unless said; launches replayed in a graph):
// * As long as every workgroup has a compute unit to itself: then the smallest number of pixels for which that holds is the best or within 3 % of it (256 -> 256
//   at 8^2, one image, 4, 8, 16 pixels 7.4, 7.2, 8.6; 128 -> 256 6.4, 6.5, 7.3; 512 -> 512 at 2^2 x 8, 4 and 8 pixels 9.3, 10.0). A second round of workgroups
//   doubles the time (256 -> 256 at 8^2 x 8 10.2 / 16.9).
// * Four steps side by side: 512 -> 512 at 4^2 12.0 / 8.8, x 4 12.6 / 9.2, at 7^2 12.6 / 9.5, 256 -> 256 at 8^2 9.9 / 7.4, x 4 10.0 / 8.7, 128 -> 256 at 8^2 8.0 / 6.4,
//   stride 2 from 28^2 9.4 / 7.4, 64 -> 128 at 16^2 6.9 / 6.1, 32 -> 64 at 12^2 7.1 / 6.1, 512 -> 512 1x1 at 4^2 6.9 / 6.0, 512 -> 100 at 7^2 13.9 / 9.1; T = 8
//   256 -> 256 at 8^2 17.5 / 11.6, 64 -> 128 at 16^2 11.7 / 9.2. Sixteen pixels and one window pay from 128 channels of 3x3 on (8.2 / 7.4; 64 -> 128 at 16^2 x 2
//   6.9 / 7.0).
// * Two steps gain little (256 -> 256 at 8^2 6.8 / 6.4, 128 -> 256 x 2 5.9 / 5.9) and less on sixteen pixels; of one step the tiles of 32 are faster (512 -> 512
//   at 4^2 7.1 / 7.6, 64 -> 128 at 16^2 4.7 / 5.3).
// All channel groups of the halo have to fit LDS.
bool plan_few(FewGeom& g, const PackGeom& pg, size_t& lds_bytes) {
    const int64_t K = static_cast<int64_t>(g.taps) * pg.Cin;
    const int cus = compute_units();
    g.oc_tiles = (g.Cout + 15) / 16;
    if (g.T < 2 || (g.T == 2 && K < 1152) || pg.CK < 16 || static_cast<int64_t>(g.N) * g.Ho * g.Wo * g.oc_tiles > 16 * static_cast<int64_t>(cus)) return false;
    const size_t weight = packed_weight_elems(pg) * 2;
    if (weight >= kFewOutside) return false;
    g.weight_bytes = static_cast<uint32_t>(weight);
    g.frag_bytes = pg.nchunks * pg.npairs * kFragBytes;
    g.npairs = pg.npairs;
    g.gph_log2 = 0;
    while ((2 << g.gph_log2) < pg.CK / 8) ++g.gph_log2;
    g.C8e = (g.C8in + 1) / 2 * 2;
    const int tt = g.T == 2 ? 2 : 4;
    for (int px = 16 / tt; px <= (tt == 2 || (g.T <= 4 && K < 1152) ? 8 : 16); px <<= 1) {
        // The patch of up to `px` pixels with the fewest workgroups, then the smallest halo.
        int64_t best = -1;
        FewGeom found = g;
        for (int pc = 1; pc <= px && pc <= g.Wo; ++pc) {
            const int pr = std::min(px / pc, g.Ho);
            if (g.pool && ((pc | pr) & 1)) continue;
            const int pi = pr == g.Ho && pc == g.Wo ? std::max(1, std::min(g.N, px / (pr * pc))) : 1;
            const int rr = (pr - 1) * g.sh + g.KH, rc = (pc - 1) * g.sw + g.KW;
            const int px_n = (g.Wo + pc - 1) / pc, py_n = (g.Ho + pr - 1) / pr, in = (g.N + pi - 1) / pi;
            const int64_t patches = static_cast<int64_t>(px_n) * py_n * in;
            const int64_t cost = patches * 65536 + static_cast<int64_t>(pi) * rr * rc;
            if (best >= 0 && cost >= best) continue;
            best = cost;
            found.PI = pi; found.PR = pr; found.PC = pc; found.RR = rr; found.RC = rc;
            found.region = pi * rr * rc;
            found.patches_x = px_n;
            found.patches_img = px_n * py_n;
            found.patches = patches;
        }
        const int64_t grid = found.patches * g.oc_tiles;
        if (best < 0 || grid > cus) continue;
        found.frags = px * tt / 16;
        found.px_log2 = px == 16 ? 4 : (px == 8 ? 3 : 2);
        const int fixed = kFewTableBytes + kFewBitsBytes + kFewWaves * found.frags * 1024;
        const int group_bytes = tt * found.region * 16;
        if (static_cast<int64_t>(fixed) + static_cast<int64_t>(g.C8e) * group_bytes <= static_cast<int64_t>(kMaxLds)) {
            found.Gs = g.C8e;
            found.grid = static_cast<int>(grid);
            g = found;
            lds_bytes = static_cast<size_t>(fixed) + static_cast<size_t>(g.Gs) * group_bytes;
            g.d_oc_tiles = make_spk_div(g.oc_tiles);
            g.d_patches_img = make_spk_div(g.patches_img);
            g.d_patches_x = make_spk_div(g.patches_x);
            g.d_ppx = make_spk_div(g.PR * g.PC);
            g.d_PC = make_spk_div(g.PC);
            g.d_region = make_spk_div(g.region);
            g.d_rrrc = make_spk_div(g.RR * g.RC);
            g.d_RC = make_spk_div(g.RC);
            g.d_taps = make_spk_div(g.taps);
            return true;
        }
    }
    return false;
}

int launch_conv_few(const FewLaunch& L, bool f16, int in_layout) {
    if (in_layout == kSpkSteps) return f16 ? launch<f16_t, kSpkSteps>(L) : launch<bf16_t, kSpkSteps>(L);
    if (in_layout == SNNF_LAYOUT_BITS) return f16 ? launch<f16_t, SNNF_LAYOUT_BITS>(L) : launch<bf16_t, SNNF_LAYOUT_BITS>(L);
    return f16 ? launch<f16_t, SNNF_LAYOUT_C8>(L) : launch<bf16_t, SNNF_LAYOUT_C8>(L);
}

}  // namespace snnf
