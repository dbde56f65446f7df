// Stand-alone convolution kernels, the configuration table and the launchers.  Device code: conv_body.h.
#include "conv_kernel.h"
#include "conv_mixed.h"
#include "conv_window.h"
#include "launch_internal.h"

#include <algorithm>
#include <climits>
#include <cstring>
#include <stdexcept>
#include <string>

namespace ios {

__global__ void splitk_reduce_kernel(ReduceArgs a) { splitk_reduce_body(a, blockIdx.x, gridDim.x, blockDim.x); }

// ---- variant table --------------------------------------------------------------------------------------------
typedef void (*ConvKernelFn)(ConvKernelArgs);

struct VariantEntry {
    ConvVariant v;
    KernelPair any;
    int smem_floats;
    KernelPair special[4] = {};   // staged kernels for the filters that kernel_of() names
};

#define IOS_TILED_ENTRY(IDX, NAME, BM, BN, BK, WM, WN, WK, MT, PD)                                        \
    {{NAME, BM, BN, BK, WM, WN, WK, MT, false, ConvTiled<BM, BN, BK, WM, WN, WK, MT, PD>::CPAD, false, \
      ConvTiled<BM, BN, BK, WM, WN, WK, MT, PD>::FUSABLE, false},    \
     kTiledKernels[IDX], \
     ConvTiled<BM, BN, BK, WM, WN, WK, MT, PD>::SMEM_FLOATS},
#define IOS_WSPLIT_ENTRY(IDX, NAME, MT, TM, TN, NW, U, QUAD, D, BF16)                                                                  \
    {{NAME, TM * MT, TN * MT, U *(MT == 32 ? 2 : 4), 1, 1, NW, MT, true, ConvWsplit<MT, TM, TN, NW, U, QUAD, D, BF16>::CPAD, QUAD, \
      ConvWsplit<MT, TM, TN, NW, U, QUAD, D, BF16>::FUSABLE, BF16},      \
     {conv_kernel<ConvWsplit<MT, TM, TN, NW, U, QUAD, D, BF16>>, conv_kernel<ConvWsplit<MT, TM, TN, NW, U, QUAD, D, BF16>, true>}, \
     ConvWsplit<MT, TM, TN, NW, U, QUAD, D, BF16>::SMEM_FLOATS},
#define IOS_WSPLIT_C4_ENTRY(IDX, NAME, MT, TM, TN, NW, U, QUAD, D, BF16)                                                                  \
    {{NAME, TM * MT, TN * MT, U *(MT == 32 ? 2 : 4), 1, 1, NW, MT, true, ConvWsplit<MT, TM, TN, NW, U, QUAD, D, BF16, 4>::CPAD, QUAD, \
      ConvWsplit<MT, TM, TN, NW, U, QUAD, D, BF16, 4>::FUSABLE, BF16},                                                                 \
     {conv_kernel<ConvWsplit<MT, TM, TN, NW, U, QUAD, D, BF16, 4>>, conv_kernel<ConvWsplit<MT, TM, TN, NW, U, QUAD, D, BF16, 4>, true>}, \
     ConvWsplit<MT, TM, TN, NW, U, QUAD, D, BF16, 4>::SMEM_FLOATS},

#define IOS_SPLIT3_ENTRY(IDX, NAME, TMW, TNW, WM, WN, PD)                                                                              \
    {{NAME, ConvSplit3<TMW, TNW, WM, WN, PD>::BM, ConvSplit3<TMW, TNW, WM, WN, PD>::BN, 16, WM, WN, 1, 32, false,                         \
      ConvSplit3<TMW, TNW, WM, WN, PD>::CPAD, false, false, PREC_FP32, 3},                                                                \
     kSplit3Kernels[IDX - kFirstSplit3Variant], \
     ConvSplit3<TMW, TNW, WM, WN, PD>::SMEM_FLOATS},

#define IOS_WSPLIT_X3_ENTRY(IDX, NAME, TM, TN, NW, D)                                                                        \
    {{NAME, TM * 32, TN * 32, 16, 1, 1, NW, 32, true, ConvWsplit<32, TM, TN, NW, 8, true, D, 3>::CPAD, true, false, PREC_FP32, 2, \
      ConvWsplit<32, TM, TN, NW, 8, true, D, 3>::FUSABLE_WIDE},      \
     {conv_kernel<ConvWsplit<32, TM, TN, NW, 8, true, D, 3>>, conv_kernel<ConvWsplit<32, TM, TN, NW, 8, true, D, 3>, true>}, \
     ConvWsplit<32, TM, TN, NW, 8, true, D, 3>::SMEM_FLOATS},

#define IOS_WSPLIT_HALF_ENTRY(KERNEL, BK, MT, RP, PRECISION, PLANES, NAME, TM, TN, NW, D)                                               \
    {{NAME, TM * MT, TN * MT, BK, 1, 1, NW, MT, true, ConvWsplit<MT, TM, TN, NW, 8, true, D, RP>::CPAD, true,                            \
      ConvWsplit<MT, TM, TN, NW, 8, true, D, RP>::FUSABLE, PRECISION, PLANES, ConvWsplit<MT, TM, TN, NW, 8, true, D, RP>::FUSABLE_WIDE},  \
     KERNEL, ConvWsplit<MT, TM, TN, NW, 8, true, D, RP>::SMEM_FLOATS},
#define IOS_WSPLIT_X3S_ENTRY(IDX, ...) IOS_WSPLIT_HALF_ENTRY(kWsplitX3sKernels[IDX - kFirstWsplitX3sVariant], 32, 16, 3, PREC_FP32, 2, __VA_ARGS__)
#define IOS_WSPLIT_XH_ENTRY(IDX, ...) IOS_WSPLIT_HALF_ENTRY(kWsplitXhKernels[IDX - kFirstWsplitXhVariant], 16, 32, 5, PREC_FP16, 1, __VA_ARGS__)

#define IOS_SPLIT1_ENTRY(IDX, NAME, TMW, TNW, WM, WN, PD)                                                                              \
    {{NAME, ConvSplit3<TMW, TNW, WM, WN, PD, 1>::BM, ConvSplit3<TMW, TNW, WM, WN, PD, 1>::BN, 16, WM, WN, 1, 32, false,                   \
      ConvSplit3<TMW, TNW, WM, WN, PD, 1>::CPAD, false, false, PREC_BF16, 1},                                                             \
     kSplit1Kernels[IDX - kFirstSplit1Variant], \
     ConvSplit3<TMW, TNW, WM, WN, PD, 1>::SMEM_FLOATS},

#define IOS_WSPLIT_X1_ENTRY(IDX, NAME, TM, TN, NW, D)                                                                        \
    {{NAME, TM * 32, TN * 32, 16, 1, 1, NW, 32, true, ConvWsplit<32, TM, TN, NW, 8, true, D, 4>::CPAD, true, false, PREC_BF16, 1},      \
     {conv_kernel<ConvWsplit<32, TM, TN, NW, 8, true, D, 4>>, conv_kernel<ConvWsplit<32, TM, TN, NW, 8, true, D, 4>, true>}, \
     ConvWsplit<32, TM, TN, NW, 8, true, D, 4>::SMEM_FLOATS},

#define IOS_PIPE_ENTRY(TERMS, HALF, PRECISION, IDX, NAME, KU, PD, TMW, TNW, WM, WN)                                                       \
    {{NAME, ConvPipe<TERMS, HALF, KU, PD, TMW, TNW, WM, WN>::BM, ConvPipe<TERMS, HALF, KU, PD, TMW, TNW, WM, WN>::BN, 16 * KU, WM, WN, 1, 32, \
      false, 16, false, false, PRECISION, TERMS},                                                                                     \
     kPipeKernels[IDX - kFirstPipeVariant][0], \
     ConvPipe<TERMS, HALF, KU, PD, TMW, TNW, WM, WN>::SMEM_FLOATS,                                                                   \
     {kPipeKernels[IDX - kFirstPipeVariant][1], kPipePlainKernels[IDX - kFirstPipeVariant][0], kPipePlainKernels[IDX - kFirstPipeVariant][1]}},
#define IOS_PIPE3_ENTRY(...) IOS_PIPE_ENTRY(2, true, PREC_FP32, __VA_ARGS__)
#define IOS_PIPE_BF16_ENTRY(...) IOS_PIPE_ENTRY(1, false, PREC_BF16, __VA_ARGS__)
#define IOS_PIPE_FP16_ENTRY(...) IOS_PIPE_ENTRY(1, true, PREC_FP16, __VA_ARGS__)

#define IOS_WINDOW_ENTRY(TERMS, HALF, PRECISION, IDX, NAME, TMW, TNW, WM, WN, P_IT, NBUF)                                                 \
    {{NAME, 32 * TMW * WM, 32 * TNW * WN, 16, WM, WN, 1, 32, false, 16, false, false, PRECISION, TERMS, false,                            \
      ConvWindow<TERMS, HALF, TMW, TNW, WM, WN, P_IT, NBUF>::SPAN},                                                                     \
     kWindowKernels[IDX - kFirstWindowVariant], \
     ConvWindow<TERMS, HALF, TMW, TNW, WM, WN, P_IT, NBUF>::SMEM_FLOATS, \
     {kWindow7Kernels[IDX - kFirstWindowVariant], kWindow9Kernels[IDX - kFirstWindowVariant], \
      kWindow7ShortKernels[IDX - kFirstWindowVariant], kWindow9ShortKernels[IDX - kFirstWindowVariant]}},
#define IOS_WINDOW3_ENTRY(...) IOS_WINDOW_ENTRY(2, true, PREC_FP32, __VA_ARGS__)
#define IOS_WINDOW_BF16_ENTRY(...) IOS_WINDOW_ENTRY(1, false, PREC_BF16, __VA_ARGS__)
#define IOS_WINDOW_FP16_ENTRY(...) IOS_WINDOW_ENTRY(1, true, PREC_FP16, __VA_ARGS__)

static const VariantEntry kVariants[] = {IOS_TILED_VARIANTS(IOS_TILED_ENTRY) IOS_WSPLIT_VARIANTS(IOS_WSPLIT_ENTRY)
                                             IOS_WSPLIT_C4_VARIANTS(IOS_WSPLIT_C4_ENTRY)
                                             IOS_WSPLIT_T32_VARIANTS(IOS_WSPLIT_ENTRY) IOS_WSPLIT_F16_VARIANTS(IOS_WSPLIT_ENTRY)
                                             IOS_WSPLIT_LONGK_VARIANTS(IOS_WSPLIT_ENTRY) IOS_SPLIT3_VARIANTS(IOS_SPLIT3_ENTRY) IOS_WSPLIT_X3_VARIANTS(IOS_WSPLIT_X3_ENTRY)
                                             IOS_SPLIT1_VARIANTS(IOS_SPLIT1_ENTRY) IOS_WSPLIT_X1_VARIANTS(IOS_WSPLIT_X1_ENTRY)
                                             IOS_PIPE3_VARIANTS(IOS_PIPE3_ENTRY) IOS_PIPE_BF16_VARIANTS(IOS_PIPE_BF16_ENTRY)
                                             IOS_PIPE_FP16_VARIANTS(IOS_PIPE_FP16_ENTRY) IOS_WINDOW3_VARIANTS(IOS_WINDOW3_ENTRY)
                                             IOS_WINDOW_BF16_VARIANTS(IOS_WINDOW_BF16_ENTRY) IOS_WINDOW_FP16_VARIANTS(IOS_WINDOW_FP16_ENTRY)
                                             IOS_WSPLIT_X3S_VARIANTS(IOS_WSPLIT_X3S_ENTRY) IOS_WSPLIT_XH_VARIANTS(IOS_WSPLIT_XH_ENTRY)};
constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);
static_assert(kNumVariants == kNumConvVariants, "variant lists and count disagree");

int conv_num_variants() { return kNumVariants; }

const ConvVariant &conv_variant(int index) {
    if (index < 0 || index >= kNumVariants) throw std::runtime_error("conv variant index out of range");
    return kVariants[index].v;
}

static int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

static int variant_by_name(const char *name) {
    for (int i = 0; i < kNumVariants; i++)
        if (std::string(kVariants[i].v.name) == name) return i;
    throw std::runtime_error(std::string("conv: no kernel configuration named ") + name);
}

// Input pixels that a block of `outputs` outputs reads at stride 1, as one run: to the last output's place, over the pixels that
// every row of outputs leaves out, and the rows and columns the filter reaches over.
static long long window_span(const ConvProblem &p, int outputs) {
    return outputs - 1 + (long long)ceil_div(outputs - 1, p.OW) * (p.W - p.OW) + (long long)(p.KH - 1) * p.W + p.KW;
}

bool conv_variant_takes(const ConvProblem &p, int variant) {
    const ConvVariant &v = conv_variant(variant);
    if (v.window == 0) return true;
    const int taps = p.KH * p.KW;   // odd, and a bit each
    return p.sh == 1 && p.sw == 1 && taps % 2 == 1 && taps >= 3 && taps < 32 && p.OH <= p.H && p.OW <= p.W && window_span(p, v.BN) <= v.window;
}

// Configurations that the tuner leaves out.  None of them was the fastest in any share class over 3030 problems: the convolutions of
// nine networks (Inception-v3, SqueezeNet, ResNet-18 / 50, RandWire, NASNet, VGG-16, AlexNet, the sample network) at batch 1 to 64 and
// of multi-branch blocks on odd sizes, in each precision, with three bfloat16 terms where two of half are now.  Against the kernels of
// now, each pinned in turn on 30 fp32 layers (K from 4 to 4608, those below 64 that the two-term kernels do not serve among them) at batch
// 1, 16 and 64: the best of them takes 1.0 to 2.5 times the time of the best measured one, but for 60 -> 60 1 x 1 on 33 x 33 (5.6 against
// 5.7 us at batch 16, 11.0 against 11.3 at 64) and 64 -> 16 on 55 x 55 at batch 16 (5.8 against 6.1).  They serve the closed-form choice, which knows none of the others, and the option that pins a configuration.
static const char *const kNotMeasured[] = {
    "m64n64k32_w2x2x1_t32", "m128n128k16_w2x2x1_t32", "m32n32k64_w1x1x4_t32", "m64n32k32_w2x1x2_t32", "m32n64k32_w1x2x2_t32",
    "m128n64k16_w2x2x1_t32", "m64n16k64_w4x1x1_t16", "m32n16k64_w2x1x2_t16", "m16n16k128_w1x1x4_t16", "m64n128k16_w2x2x1_t32",
    "m64n64k16_w2x2x1_t32", "m32n128k16_w1x4x1_t32", "m192n64k16_w2x2x1_t32", "m96n128k16_w1x4x1_t32", "m192n128k16_w2x2x1_t32",
    "m160n128k16_w1x4x1_t32", "ws_m32n16_w16_t16", "ws_m16n16_w16_t16", "ws_m32n32_w16_t16", "ws_m64n16_w16_t16",
    "ws_m32n16_w8_t16", "ws_m32n16_w4_t16", "ws_m32n32_w16_t32", "ws_m16n32_w16_t16", "wq_m32n32_w16_t16", "wq_m64n32_w8_t16",
    "wq_m64n64_w4_t16", "wq_m32n32_w8_t16", "wq_m64n64_w4_t32", "wq_m16n16_w16_t16_d4",
    "wq_m32n16_w16_t16_d4", "wq_m32n32_w2_t16_d4", "wq_m64n32_w2_t16", "wq_m64n32_w4_t16_d4", "wb_m64n64_w4",
    "ws_m32n64_w1_t16_c4", "wq_m32n32_w8_t32", "wq_m32n32_w16_t32", "wq_m64n32_w8_t32", "wq_m64n32_w4_t32", "wq_m32n64_w8_t32",
    "wq_m32n64_w4_t32", "wq_m64n64_w8_t32", "wq_m64n32_w2_t32", "wq_m64n32_w1_t32", "wq_m32n64_w2_t32", "wq_m32n32_w2_t32_d4",
    "wq_m32n32_w1_t16_d4", "wq_m64n64_w2_t32", "x3_m64n64_w2x2", "x3_m64n64_w1x1", "x3_m64n128_w1x2", "x3_m192n128_w6x2",
    "wb_x1_m64n128_w2x2", "wb_x1_m128n256_w2x4", "wb_x1_m64n128_w1x2", "wb_x1_m64n256_w2x4",
};

static bool precise_only(const ConvProblem &p) { return p.K() < 64; }

bool conv_variant_precise(const ConvProblem &p, int variant) { return !(precise_only(p) && kVariants[variant].v.koct == 2); }

bool conv_variant_measured(const ConvProblem &p, int variant) {
    static const std::vector<char> measured = [] {
        std::vector<char> flags(kNumVariants, 1);
        for (const char *name : kNotMeasured) flags[variant_by_name(name)] = 0;
        return flags;
    }();
    // Two terms of half against three of bfloat16: half the matrix work, and half the roundings of the sum, but operands that are off in
    // the last bit.  Below a K of 64 the second shows (errors 8.3e-8 against 7.1e-8 at K = 16), and nothing there is bound by matrix work
    // (16 -> 64 channels on 55 x 55 at batch 50: 13.1 us by fp32 instructions, 15.2 by two terms); from 64 on the first (2.7e-7 against
    // 3.6e-7 at K = 576), and the three-term kernels are slower or within 1 %.
    const int planes = kVariants[variant].v.koct;
    if (!conv_variant_precise(p, variant) || (planes == 3 && !precise_only(p))) return false;
    return measured.at(variant) != 0;
}

// The entry that serves the problem: where a window kernel is asked for and does not take it, one that reads the same packed filters.
static int variant_for(const ConvProblem &p, const ConvLaunch &l) {
    if (l.variant < 0 || l.variant >= kNumVariants) throw std::runtime_error("conv: bad variant");
    if (conv_variant_takes(p, l.variant)) return l.variant;
    const int precision = kVariants[l.variant].v.precision;
    static const int plain[] = {variant_by_name("x3p_m64n128_w1x4"), variant_by_name("wb_p_m64n128_w1x4"), variant_by_name("wh_p_m64n128_w1x4")};
    return plain[precision == PREC_FP32 ? 0 : precision == PREC_BF16 ? 1 : 2];
}

// tiles of output pixels; a window kernel takes its tiles from one image at a time where the maps shrink (see ConvWindow)
static int tiles_of_pixels(const ConvProblem &p, const ConvVariant &v) {
    return v.window != 0 && p.OH != p.H ? p.B * ceil_div((long long)p.OH * p.OW, v.BN) : ceil_div(p.Npix(), v.BN);
}

static int k_chunk_of(const ConvProblem &p, const ConvLaunch &l) {
    const ConvVariant &v = kVariants[variant_for(p, l)].v;
    if (v.window != 0) return ceil_div(p.ICgP(v.cpad) / 16, std::max(1, l.split_k)) * 16 * p.KH * p.KW;   // chunks of channels, all taps of each
    const int kq = p.Kq(v.cpad);
    // for the wave-split kernels BK is the K extent of one register batch, which may not divide kq
    const int tiles_k = ceil_div(kq, v.BK);
    return ceil_div(tiles_k, std::max(1, l.split_k)) * v.BK;
}

// split_k may ask for more slices than there are K tiles; the effective count leaves no slice empty
static int effective_split(const ConvProblem &p, const ConvLaunch &l) {
    return std::max(1, ceil_div(p.Kq(kVariants[variant_for(p, l)].v.cpad), k_chunk_of(p, l)));
}

int conv_effective_split(const ConvProblem &p, const ConvLaunch &l) { return effective_split(p, l); }

size_t conv_workspace_floats(const ConvProblem &p, const ConvLaunch &l) {
    const int s = effective_split(p, l);
    if (s <= 1) return 0;
    // two-kernel form: [slice][OC][pixels]; one-kernel forms: [group][tile][slice][BM * BN] with the tile count rounded up
    // to a multiple of 8 (the numbering of the XCD-local form, see XcdSlot)
    const ConvVariant &v = kVariants[variant_for(p, l)].v;
    const size_t tiles = (size_t)xcd_padded_tiles(ceil_div(p.OCg(), v.BM) * tiles_of_pixels(p, v));
    const size_t padded = (size_t)p.groups * tiles * v.BM * v.BN;
    return (size_t)s * std::max((size_t)p.OC * (size_t)p.Npix(), padded);
}

size_t conv_counter_count(const ConvProblem &p, const ConvLaunch &l) {
    if (effective_split(p, l) <= 1) return 0;
    const ConvVariant &v = kVariants[variant_for(p, l)].v;
    return (size_t)p.groups * (size_t)xcd_padded_tiles(ceil_div(p.OCg(), v.BM) * tiles_of_pixels(p, v));
}

ConvLaunch conv_pick_launch(const ConvProblem &p, int num_cus, bool fusable_only, int precision) {
    // Closed-form model distilled from measured choices on Inception-v3 at batch 1, 16 and 64: problems that fill
    // the device several times over with 64 x 64 tiles take the LDS-tiled kernel (the largest tile that still
    // offers two blocks per compute unit); smaller ones take the wave-split kernel with the largest tile that
    // still offers a block per compute unit; the smallest split K over the grid as well.
    const long long M = p.OCg(), N = p.Npix();
    auto blocks_of = [&](int idx) {
        const ConvVariant &v = kVariants[idx].v;
        return (long long)ceil_div(M, v.BM) * ceil_div(N, v.BN) * p.groups;
    };
    ConvLaunch best;
    if (precision != PREC_FP32) {
        // reduced precision: wave-split configurations only, the largest tile that offers two blocks per compute unit
        static const int bf16_large_to_small[] = {variant_by_name("wb_m64n64_w4"), variant_by_name("wb_m64n32_w8"),
                                                  variant_by_name("wb_m32n32_w8"), variant_by_name("wb_m32n16_w8"),
                                                  variant_by_name("wb_m16n16_w16")};
        static const int fp16_large_to_small[] = {variant_by_name("wh_m64n64_w4"), variant_by_name("wh_m64n32_w8"),
                                                  variant_by_name("wh_m32n32_w8"), variant_by_name("wh_m32n16_w8"),
                                                  variant_by_name("wh_m16n16_w16")};
        const int *large_to_small = precision == PREC_BF16 ? bf16_large_to_small : fp16_large_to_small;
        for (int i = 0; i < 4; i++) {
            const int idx = large_to_small[i];
            if ((!fusable_only || kVariants[idx].v.fusable()) && blocks_of(idx) >= 2LL * num_cus) {
                best.variant = idx;
                return best;
            }
        }
        best.variant = large_to_small[4];
        const ConvVariant &v = kVariants[best.variant].v;
        const long long blocks = blocks_of(best.variant);
        const int batches = ceil_div(p.Kq(v.cpad), v.BK);
        const long long split = std::min<long long>((num_cus + blocks - 1) / blocks, std::max(1, batches / (2 * v.WK)));
        best.split_k = (int)std::max<long long>(1, std::min<long long>(split, 16));
        return best;
    }
    static const int tiled_mid = variant_by_name("m64n64k16_w2x2x1_t32");
    if (!fusable_only && blocks_of(tiled_mid) >= 4LL * num_cus) {
        static const int by_size[] = {variant_by_name("m128n128k16_w2x2x1_t32"), variant_by_name("m128n64k16_w2x2x1_t32"),
                                      variant_by_name("m64n128k16_w2x2x1_t32")};
        best.variant = tiled_mid;
        for (int idx : by_size) {
            if (fusable_only && !kVariants[idx].v.fusable()) continue;
            if (blocks_of(idx) >= 2LL * num_cus) {
                best.variant = idx;
                break;
            }
        }
        return best;
    }
    static const int split_large_to_small[] = {variant_by_name("wq_m64n32_w8_t16"), variant_by_name("wq_m32n32_w8_t16"),
                                               variant_by_name("wq_m32n16_w8_t16")};
    for (int idx : split_large_to_small)
        if ((!fusable_only || kVariants[idx].v.fusable()) && blocks_of(idx) >= num_cus) {
            best.variant = idx;
            return best;
        }
    best.variant = variant_by_name("wq_m16n16_w16_t16");
    const ConvVariant &v = kVariants[best.variant].v;
    const long long blocks = blocks_of(best.variant);
    const int batches = ceil_div(p.Kq(v.cpad), v.BK);          // register batches along K
    const int per_slice = 2 * v.WK;                            // leave every wavefront two batches
    const long long split = std::min<long long>((num_cus + blocks - 1) / blocks, std::max(1, batches / per_slice));
    best.split_k = (int)std::max<long long>(1, std::min<long long>(split, 16));
    return best;
}

bool conv_matrix_path_supported(const ConvProblem &p) {
    // packed filter rows are indexed with 16 bits, input and filter byte offsets with 31 bits (an input of less than 2^30 bytes has
    // at most 1.6 * 2^30 with its pixels padded, five channels to eight; a window of a wider tensor is checked where it is known)
    const unsigned long long x_bytes = (unsigned long long)p.B * p.IC * p.H * p.W * 4ull;
    const unsigned long long w_bytes = (unsigned long long)p.groups * p.Kq(128) * p.OCgP() * 4ull;
    // image sides below 2^15 and output planes below 2^23 elements keep the kernels' signed 24-bit index multiplies exact
    return p.Kq(128) < 65536 && p.Npix() < (1LL << 31) && x_bytes < (1ull << 30) && w_bytes < (1ull << 31) && p.H < 32768 && p.W < 32768 &&
           (long long)p.OH * p.OW < (1LL << 23) && p.B < (1 << 23);
}

ConvDispatch make_conv_dispatch(const ConvProblem &p, const ConvLaunch &l, const TensorView &x, const float *packed,
                                const float *filters, const float *bias, const TensorView &y, float *workspace, const SplitKReduce &reduce,
                                const TensorView *residual, bool post_relu) {
    const int variant = variant_for(p, l);
    const VariantEntry &e = kVariants[variant];
    if (x.C != p.IC || x.H != p.H || x.W != p.W || y.C != p.OC || y.H != p.OH || y.W != p.OW)
        throw std::runtime_error("conv: tensor views do not match the problem");
    if (p.IC % p.groups != 0 || p.OC % p.groups != 0) throw std::runtime_error("conv: channels not divisible by groups");
    if (!conv_matrix_path_supported(p)) throw std::runtime_error("conv: problem too large for the matrix path");
    ConvDispatch d;
    ConvKernelArgs &a = d.args;
    a.x = x.ptr;
    a.wp = packed;
    a.w = filters;
    a.bias = bias;
    a.y = y.ptr;
    a.ws = workspace;
    a.counters = reduce.counters;
    a.H = p.H; a.W = p.W; a.OH = p.OH; a.OW = p.OW;
    a.sh = p.sh; a.sw = p.sw; a.ph = p.ph; a.pw = p.pw;
    a.KW = p.KW;
    a.ICg = p.ICg(); a.ICgP = p.ICgP(e.v.cpad); a.OCg = p.OCg(); a.OCgP = p.OCgP(); a.Kq = p.Kq(e.v.cpad);
    a.magic_icgp = (unsigned)((1ULL << 32) / (unsigned)a.ICgP + 1);   // ICgP >= 8
    a.magic_kw = (unsigned)((1ULL << 32) / (unsigned)a.KW + 1);       // unused when KW == 1
    a.OHW = p.OH * p.OW; a.groups = p.groups;
    a.x_ps = x.pstride; a.y_ps = y.pstride;
    const unsigned long long x_bytes = conv_input_extent(p, x.pstride);
    const unsigned long long w_bytes = (unsigned long long)p.groups * p.Kq(e.v.cpad) * p.OCgP() * (e.v.koct ? 2ull * e.v.koct : e.v.precision != PREC_FP32 ? 2ull : 4ull);
    if (x_bytes >= (1ull << 31) || w_bytes >= (1ull << 31)) throw std::runtime_error("conv: tensor too large for 31-bit buffer offsets");
    a.x_bytes = (unsigned)x_bytes;
    a.w_bytes = (unsigned)w_bytes;
    a.Npix = (int)p.Npix();
    a.act = p.act; a.pre_relu = p.pre_relu;
    a.k_chunk = k_chunk_of(p, l);
    a.split_k = effective_split(p, l);
    {
        // the wave-split kernels' division of a grid slice among the wavefronts of a block (BK = U k-steps, WK wavefronts)
        const int kstep = e.v.MT == 32 ? 2 : 4;
        const int u = std::max(1, e.v.BK / kstep);
        a.steps_total = a.Kq / kstep;
        a.steps_chunk = a.k_chunk / kstep;
        a.steps_per_wave = e.v.kquad ? ceil_div(ceil_div(a.steps_chunk, u), e.v.WK) * u : ceil_div(a.steps_chunk, e.v.WK);
    }
    a.tiles_m = ceil_div(p.OCg(), e.v.BM);
    a.tiles_n = tiles_of_pixels(p, e.v);
    a.weights_major = (double)p.OC * p.K() > (double)p.B * p.IC * p.H * p.W ? 1 : 0;
    a.tile_div = a.weights_major ? a.tiles_n : a.tiles_m;
    a.xcd_q = (a.tiles_m * a.tiles_n) >> 3;
    a.xcd_r = (a.tiles_m * a.tiles_n) & 7;
    a.div_tile = make_fast_div((unsigned)a.tile_div);
    a.div_ohw = make_fast_div((unsigned)a.OHW);
    a.div_ow = make_fast_div((unsigned)a.OW);
    a.res = nullptr;
    a.res_ps = 0;
    a.post_relu = post_relu ? 1 : 0;
    if (residual != nullptr) {
        if (residual->C != p.OC || residual->H != p.OH || residual->W != p.OW) throw std::runtime_error("conv: residual view does not match the output");
        a.res = residual->ptr;
        a.res_ps = residual->pstride;
    } else if (post_relu) {
        throw std::runtime_error("conv: activation after a residual that is not there");
    }
    if (a.split_k > 1 && workspace == nullptr) throw std::runtime_error("conv: split-K launch without workspace");
    if (p.groups > 65535 || a.split_k > 65535) throw std::runtime_error("conv: grid too large");
    d.variant = variant;
    d.threads = e.v.threads();
    d.smem_bytes = e.smem_floats * (int)sizeof(float);
    d.tiles = a.tiles_m * a.tiles_n;
    d.groups = p.groups;
    d.slices = a.split_k;
    if (a.split_k <= 1) a.counters = nullptr;
    // K slices that meet inside an XCD: a one-dimensional grid in the numbering of XcdSlot (plain convolutions without
    // groups; the fields share their place with those of the residual form)
    a.xcd_local = a.counters != nullptr && reduce.xcd_local && reduce.fault != nullptr && p.groups == 1 && residual == nullptr &&
                          a.split_k <= 64 && xcd_grid_blocks(d.tiles, a.split_k) / 8 < (1 << 26)
                      ? 1 : 0;
    d.xcd_blocks = 0;
    if (a.xcd_local) {
        a.fault = reduce.fault;
        a.xcd_map = reduce.xcd_map;
        a.magic_split = (unsigned)((1ULL << 32) / (unsigned)a.split_k + 1);
        d.xcd_blocks = xcd_grid_blocks(d.tiles, a.split_k);
    }
    d.has_reduce = a.split_k > 1 && a.counters == nullptr;
    d.reduce_blocks = 0;
    if (d.has_reduce) {
        ReduceArgs &r = d.reduce;
        r.ws = workspace;
        r.bias = bias;
        r.y = y.ptr;
        r.slices = a.split_k;
        r.OC = p.OC;
        r.Npix = a.Npix;
        r.act = p.act;
        r.slice_floats = (long long)p.OC * a.Npix;
        r.y_ps = y.pstride;
        r.res = a.res;
        r.res_ps = a.res_ps;
        r.post_relu = a.post_relu;
        d.reduce_blocks = (int)std::min<long long>((r.slice_floats + 255) / 256, 4096);
    }
    return d;
}

// Pipelined kernels: inputs that need neither a ReLU nor channels masked, for kernels of 1 x 1 filters (`point`) in whole stages, for others in
// whole quads
static bool pipe_plain(const ConvProblem &p, const VariantEntry &e, bool point) { return p.pre_relu == 0 && p.ICg() % (point ? e.v.BK : 4) == 0; }

// Which of an entry's kernels serves the problem: 0 any, else the special ones.  Pipelined kernels: [1] 1 x 1 filters without groups,
// whose addresses stay the same over K (at batch 64 768 -> 192 on 17 x 17 39.7 -> 34.8 us, 2048 -> 320 on 8 x 8 51.2 -> 43.1), [2] and [3] any filter
// and these where pipe_plain holds.  Window kernels:
// [1] seven taps, [2] nine (see known_chunk; other numbers are rare, 1 x 3 and 5 x 5), [3] and [4] the same where the window fits three rounds.
static int kernel_of(const ConvProblem &p, const VariantEntry &e) {
    const int taps = p.KH * p.KW;
    if (e.v.window != 0) {
        const int known = taps == 7 ? 1 : taps == 9 ? 2 : 0;
        return known != 0 && window_span(p, e.v.BN) <= short_rounds(INT_MAX) * (e.v.threads() / 2) ? known + 2 : known;
    }
    if (e.special[0].kernel == nullptr) return 0;
    const int point = taps == 1 && p.groups == 1 ? 1 : 0;
    return pipe_plain(p, e, point != 0) ? 2 + point : point;
}

void launch_conv_mfma(const ConvProblem &p, const ConvLaunch &l, const TensorView &x, const float *packed, const float *filters,
                      const float *bias, const TensorView &y, float *workspace, const SplitKReduce &reduce, hipStream_t stream,
                      const TensorView *residual, bool post_relu) {
    const ConvDispatch d = make_conv_dispatch(p, l, x, packed, filters, bias, y, workspace, reduce, residual, post_relu);
    const VariantEntry &e = kVariants[d.variant];
    const dim3 grid = d.xcd_blocks > 0 ? dim3((unsigned)d.xcd_blocks) : dim3((unsigned)d.tiles, (unsigned)d.groups, (unsigned)d.slices);
    const int which = kernel_of(p, e);
    const KernelPair &pair = which == 0 ? e.any : e.special[which - 1];
    const bool with_residual = !d.args.xcd_local && d.args.res != nullptr;
    const ConvKernelFn kernel = with_residual ? pair.kernel_residual : pair.kernel;
    if (d.smem_bytes > 64 * 1024) {   // beyond the default limit of dynamic LDS: raised once per kernel
        static bool raised[kNumConvVariants][10] = {};
        bool &done = raised[d.variant][2 * which + (with_residual ? 1 : 0)];
        if (!done) {
            if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, d.smem_bytes) != hipSuccess)
                throw std::runtime_error(std::string("conv: cannot reserve LDS for configuration ") + e.v.name);
            done = true;
        }
    }
    hipLaunchKernelGGL(kernel, grid, dim3(d.threads), d.smem_bytes, stream, d.args);
    if (d.has_reduce) hipLaunchKernelGGL(splitk_reduce_kernel, dim3(d.reduce_blocks), dim3(256), 0, stream, d.reduce);
}

// ---- several convolutions in a launch ------------------------------------------------------
bool conv_variant_batches(int variant) { return variant >= kFirstPipeVariant && variant < kFirstWindowVariant; }

bool conv_batchable(const ConvProblem &a, const ConvProblem &b) {
    return a.KH == 1 && a.KW == 1 && b.KH == 1 && b.KW == 1 && a.groups == 1 && b.groups == 1 && a.B == b.B && a.IC == b.IC && a.H == b.H && a.W == b.W &&
           a.sh == b.sh && a.sw == b.sw && a.ph == b.ph && a.pw == b.pw;
}

void launch_conv_batch(const ConvBatchMember *members, int count, int variant, hipStream_t stream) {
    if (count < 1 || count > kMaxConvBatch || !conv_variant_batches(variant)) throw std::runtime_error("conv: no such batch");
    const VariantEntry &e = kVariants[variant];
    ConvLaunch l;
    l.variant = variant;
    ConvBatchArgs b;
    int tiles_m = 0, tiles_n = 0, threads = 0, smem_bytes = 0, plain = 1;
    double filters = 0.0;
    for (int i = 0; i < kMaxConvBatch; i++) {
        const ConvBatchMember &m = members[std::min(i, count - 1)];
        if (!conv_batchable(members[0].p, m.p)) throw std::runtime_error("conv: a batch of convolutions that do not fit each other");
        const ConvDispatch d = make_conv_dispatch(m.p, l, members[0].x, m.packed, m.filters, m.bias, m.y, nullptr, SplitKReduce{});
        b.item[i] = d.args;
        b.item[i].xcd_q = b.item[i].xcd_r = b.item[i].weights_major = 0;
        b.item[i].tile_div = d.args.tiles_m;
        b.item[i].div_tile = make_fast_div((unsigned)d.args.tiles_m);
        b.first[i] = i < count ? tiles_m : INT_MAX;
        if (i >= count) continue;
        tiles_m += d.args.tiles_m;
        tiles_n = d.args.tiles_n;
        threads = d.threads;
        smem_bytes = d.smem_bytes;
        filters += (double)m.p.OC * m.p.K();
        plain &= pipe_plain(m.p, e, true) ? 1 : 0;
    }
    const ConvProblem &p = members[0].p;
    b.weights_major = filters > (double)p.B * p.IC * p.H * p.W ? 1 : 0;
    b.tile_div = b.weights_major ? tiles_n : tiles_m;
    b.div_tile = make_fast_div((unsigned)b.tile_div);
    b.xcd_q = (tiles_m * tiles_n) >> 3;
    b.xcd_r = (tiles_m * tiles_n) & 7;
    const ConvBatchKernelFn kernel = kPipeBatchKernels[variant - kFirstPipeVariant][plain];
    if (smem_bytes > 64 * 1024) {
        static bool raised[kNumConvVariants][2] = {};
        if (!raised[variant][plain]) {
            if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem_bytes) != hipSuccess)
                throw std::runtime_error(std::string("conv: cannot reserve LDS for a batch on configuration ") + e.v.name);
            raised[variant][plain] = true;
        }
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n)), dim3(threads), smem_bytes, stream, b);
}

bool conv_variant_mixes(int variant) { return variant >= kFirstPipeVariant && variant < kFirstWindowVariant + kWindowVariants; }

bool conv_mixable(const ConvProblem &p, int variant) {
    return conv_variant_mixes(variant) && p.groups == 1 && conv_variant_takes(p, variant) && conv_variant_precise(p, variant);
}

void launch_conv_mixed(const ConvBatchMember *members, int count, const MixedPool *pool, int variant, hipStream_t stream) {
    if (count < 1 || count > kMaxConvBatch || !conv_variant_mixes(variant)) throw std::runtime_error("conv: no such launch of mixed convolutions");
    const VariantEntry &e = kVariants[variant];
    ConvLaunch l;
    l.variant = variant;
    ConvMixedArgs b;
    long long blocks = 0;
    int threads = 0, smem_bytes = 0, which = -1, plain = 1;
    for (int i = 0; i < kMaxConvBatch; i++) {
        const ConvBatchMember &m = members[std::min(i, count - 1)];
        if (!conv_mixable(m.p, variant)) throw std::runtime_error(std::string("conv: configuration ") + e.v.name + " does not take a member of a launch");
        const ConvDispatch d = make_conv_dispatch(m.p, l, m.x, m.packed, m.filters, m.bias, m.y, nullptr, SplitKReduce{});
        b.item[i] = d.args;
        b.first[i] = i < count ? (int)blocks : INT_MAX;
        if (i >= count) continue;
        blocks += ((long long)d.tiles + 7) & ~7ll;
        threads = d.threads;
        smem_bytes = d.smem_bytes;
        const int here = e.v.window != 0 ? kernel_of(m.p, e) : 0;
        which = which < 0 || which == here ? here : 0;
        plain &= pipe_plain(m.p, e, false) ? 1 : 0;
    }
    b.pool_first = INT_MAX;
    b.pool_blocks = 0;
    memset(&b.pool, 0, sizeof(b.pool));
    if (pool != nullptr) {
        b.pool = make_pool_args(pool->p, pool->x, pool->y, false, &b.pool_blocks, pool->bias, pool->act);
        b.pool_blocks = std::max(1, (b.pool_blocks * 256 + threads - 1) / threads);   // (counted for 256 threads)
        b.pool_first = (int)std::min<long long>(blocks, INT_MAX);
        blocks += b.pool_blocks;
    }
    if (blocks >= INT_MAX) throw std::runtime_error("conv: grid too large");
    const int index = variant - (e.v.window != 0 ? kFirstWindowVariant : kFirstPipeVariant);
    // (windows of more than three rounds with a known number of taps are rare here: the kernel for any number serves them)
    const ConvMixedKernelFn *windows = which == 3 ? kWindow7MixedKernels : which == 4 ? kWindow9MixedKernels : kWindowMixedKernels;
    const ConvMixedKernelFn kernel = e.v.window != 0 ? windows[index] : kPipeMixedKernels[index][plain];
    if (smem_bytes > 64 * 1024) {
        static bool raised[kNumConvVariants][3] = {};
        bool &done = raised[variant][e.v.window == 0 ? plain : which >= 3 ? which - 2 : 0];
        if (!done) {
            if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem_bytes) != hipSuccess)
                throw std::runtime_error(std::string("conv: cannot reserve LDS for mixed convolutions on configuration ") + e.v.name);
            done = true;
        }
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(threads), smem_bytes, stream, b);
}

// ---- filter packing ------------------------------------------------------------------------
// Filters as two terms of half, [g][k / 8][plane][m][8], and behind the planes what channel_scale_quad and channel_least read: channel m's
// filters are packed times 2^up, which puts the largest of them (infinities and NaN aside) into [2^14, 2^15).  A block reads the
// filters of four channels twice, for the largest and to pack them (from the L2), and writes 64 bytes at a time.  With a launch of its own
// for the factors, which costs the host thread that queues the copies too, Inception-v3 at batch 1 that brings its weights along took
// 2952 us, like this 2588.
__global__ __launch_bounds__(512) void pack_half2_kernel(const float *w, float *packed, float *scales, float *leasts, int OCg, int OCgP, int ICg, int ICgP, int taps) {
    const int quads = OCgP / 4, g = blockIdx.x / quads, m0 = 4 * (blockIdx.x - g * quads);
    const int fan = ICg * taps, octets = taps * ICgP / 8;
    __shared__ unsigned waves[8];
    __shared__ float parts[8][4];
    {
        const int m = m0 + (threadIdx.x >> 7);
        const float *row = w + ((size_t)g * OCg + min(m, OCg - 1)) * fan;
        unsigned most = 0;   // magnitudes compare as integers
#pragma unroll 4
        for (int i = threadIdx.x & 127; i < fan; i += 128) {
            const unsigned v = __float_as_uint(row[i]) & 0x7fffffffu;
            if (v < 0x7f800000u) most = max(most, v);
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) most = max(most, (unsigned)__shfl_xor((int)most, d));
        if ((threadIdx.x & 63) == 0) waves[threadIdx.x >> 6] = most;
    }
    __syncthreads();
    const int m = m0 + (threadIdx.x & 3);
    const unsigned most = max(waves[2 * (threadIdx.x & 3)], waves[2 * (threadIdx.x & 3) + 1]);
    // (2^140 serves the smallest subnormal value and is undone by a subnormal factor; it takes two multiplications)
    const int up = most == 0 ? 0 : min(14 - ((int)(most >> 23) - 127), 140);
    const float first = __uint_as_float((unsigned)(127 + min(up, 100)) << 23), second = __uint_as_float((unsigned)(127 + max(up - 100, 0)) << 23);
    const float *row = w + ((size_t)g * OCg + min(m, OCg - 1)) * fan;
    halfx8 *out = reinterpret_cast<halfx8 *>(packed);
    float least = 0.f;
#pragma unroll 1
    for (int o = threadIdx.x >> 2; o < octets; o += 128) {
        const int tap = o * 8 / ICgP, c = o * 8 - tap * ICgP;
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = m < OCg && c + j < ICg ? row[(c + j) * taps + tap] : 0.f;
        halfx8 hi, lo;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float scaled = v[j] * first * second;
            hi[j] = (_Float16)scaled;
            lo[j] = (_Float16)((scaled - (float)hi[j]) * kFilterLift);
            // what a filter below the window is off by, its upper term times 2^-8 against a lower one (2^-11 of the input, times 2^8), and
            // the product of lower terms that is left out (infinite and NaN filters: all results of the channel are computed again)
            const float upper = (float)hi[j], lower = (float)lo[j] / kFilterLift, down = upper / kInputLift;
            const float off = fabsf(scaled - upper - lower) + (fabsf(down - (float)(_Float16)down) * kInputLift + fabsf(lower)) * 0x1p-11f;
            least += __builtin_isfinite(scaled) ? fabsf(scaled) < kFilterFloor ? off : 0.f : __builtin_inff();
        }
        const size_t at = ((size_t)g * octets + o) * 2 * OCgP + m;
        out[at] = hi;
        out[at + OCgP] = lo;
    }
#pragma unroll
    for (int d = 32; d >= 4; d >>= 1) least += __shfl_xor(least, d);
    if ((threadIdx.x & 63) < 4) parts[threadIdx.x >> 6][threadIdx.x & 3] = least;
    __syncthreads();
    if (threadIdx.x < 4 && m < OCg) {
        float all = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) all += parts[i][threadIdx.x];
        scales[g * OCg + m] = __uint_as_float(up <= 126 ? (unsigned)(127 - up) << 23 : 1u << (149 - up));
        leasts[g * OCg + m] = all * 4200000.f;   // 2^22, and what the sum is rounded by
    }
}

__global__ void pack_filters_kernel(const float *w, float *packed, int OCg, int OCgP, int ICg, int ICgP, int taps, int groups, int kvec,
                                    int precision, int planes) {
    // packed[g][k][m] = w[g * OCg + m][c][tap] with k = tap * ICgP + c;  rows with c >= ICg and columns with m >= OCg are zero.
    // kvec = 4: packed[g][k / 4][m][k % 4] instead (ICgP is a multiple of 4)
    // kvec = 8: planes of 16-bit values, packed[g][k / 8][plane][m][k % 8]: three planes with the exact three-term split of every
    // filter value, or one plane with the value rounded to nearest even (the reduced-precision modes)
    const size_t total = (size_t)groups * taps * ICgP * OCgP;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        int m;
        size_t gk;
        if (kvec > 1) {
            const size_t chunk = i / kvec;                       // (g, k / kvec, m)
            m = (int)(chunk % OCgP);
            gk = (chunk / OCgP) * kvec + (i % kvec);             // (g, k)
        } else {
            m = (int)(i % OCgP);
            gk = i / OCgP;
        }
        const int c = (int)(gk % ICgP);
        const size_t gt = gk / ICgP;
        const int tap = (int)(gt % taps);
        const int g = (int)(gt / taps);
        const float value = (m < OCg && c < ICg) ? w[(((size_t)g * OCg + m) * ICg + c) * taps + tap] : 0.f;
        if (kvec == 8) {
            const size_t octet = gk / 8;                         // (g, k / 8)
            const size_t at = (octet * planes * OCgP + m) * 8 + (gk % 8);
            if (planes == 3) {
                unsigned hi, mid, lo;
                split3(value, hi, mid, lo);
                unsigned short *out = reinterpret_cast<unsigned short *>(packed);
                out[at] = (unsigned short)(hi >> 16);
                out[at + (size_t)OCgP * 8] = (unsigned short)(mid >> 16);
                out[at + (size_t)OCgP * 16] = (unsigned short)(lo >> 16);
            } else if (precision == PREC_FP16) {
                reinterpret_cast<_Float16 *>(packed)[at] = (_Float16)value;   // round to nearest even
            } else {
                reinterpret_cast<__bf16 *>(packed)[at] = (__bf16)value;   // round to nearest even
            }
        } else if (precision == PREC_BF16) reinterpret_cast<__bf16 *>(packed)[i] = (__bf16)value;   // round to nearest even
        else if (precision == PREC_FP16) reinterpret_cast<_Float16 *>(packed)[i] = (_Float16)value;   // round to nearest even
        else packed[i] = value;
    }
}

static size_t packed_floats(const ConvProblem &p, const ConvVariant &v) {
    const size_t elements = (size_t)p.groups * p.Kq(v.cpad) * p.OCgP();
    if (v.koct == 2) return elements + 2 * (p.OC + 3);   // two planes of half, two words per channel (read in quads)
    if (v.koct) return (elements * v.koct + 1) / 2;   // planes of bfloat16
    return v.precision != PREC_FP32 ? (elements + 1) / 2 : elements;
}

size_t conv_packed_floats(const ConvProblem &p, const ConvLaunch &l) {
    if (l.variant < 0 || l.variant >= kNumVariants) throw std::runtime_error("conv: bad variant");
    return packed_floats(p, kVariants[l.variant].v);
}

size_t conv_packed_floats_max(const ConvProblem &p) {
    size_t most = 0;
    for (const VariantEntry &e : kVariants) most = std::max(most, packed_floats(p, e.v));
    return most;
}

void launch_pack_filters(const ConvProblem &p, const ConvLaunch &l, const float *w, float *packed, hipStream_t stream) {
    const int cpad = kVariants[l.variant].v.cpad;
    const size_t total = (size_t)p.groups * p.Kq(cpad) * p.OCgP();   // elements
    const unsigned blocks = (unsigned)std::min<size_t>((total + 255) / 256, 65535);
    if (kVariants[l.variant].v.koct == 2) {   // (two planes of half take the room of the elements)
        hipLaunchKernelGGL(pack_half2_kernel, dim3((unsigned)(p.groups * (p.OCgP() / 4))), dim3(512), 0, stream, w, packed, packed + total, packed + total + p.OC + 3, p.OCg(), p.OCgP(),
                           p.ICg(), p.ICgP(cpad), p.KH * p.KW);
        return;
    }
    hipLaunchKernelGGL(pack_filters_kernel, dim3(blocks), dim3(256), 0, stream, w, packed, p.OCg(), p.OCgP(), p.ICg(), p.ICgP(cpad),
                       p.KH * p.KW, p.groups, kVariants[l.variant].v.kvec(), kVariants[l.variant].v.precision, kVariants[l.variant].v.koct);
}

}  // namespace ios
