// Device kernels of the runtime and their host-side launchers (gfx950 / CDNA4 only).
//
// All tensors are fp32 NHWC *views*: a pointer to element (n=0, h=0, w=0, c=0), the extents C/H/W and the distance of
// neighbouring pixels in elements.  Pixels follow each other in (n, h, w) order without gaps of their own, so a channel slice or
// a window inside a wider concat buffer is again a view; producers write straight into such windows and consumers read
// slices without copies.  The channels of a pixel lie side by side because that is what every kernel reads: four consecutive
// k of an implicit GEMM, four channels of a pool or of a sum are one 16-byte load, where a channel-major tensor takes four.
// Loads and stores assume 4-byte alignment only (a window may start at any channel).  A 16-byte load of a pixel's last channels
// may run up to twelve bytes past them, into the next pixel, a neighbouring window or the padding behind a tensor.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ios {

enum Act : int { ACT_NONE = 0, ACT_RELU = 1, ACT_TANH = 2, ACT_SIGMOID = 3 };
enum Precision : int { PREC_FP32 = 0, PREC_BF16 = 1, PREC_FP16 = 2 };   // operand type of the matrix-path convolutions

constexpr int kMaxNaryInputs = 8;   // views one launch adds (or multiplies)

struct TensorView {
    float *ptr = nullptr;  // element (0, 0, 0, 0)
    int C = 0, H = 0, W = 0;
    int pstride = 0;       // elements between pixels
};

// Division of a 32-bit unsigned by a divisor fixed at launch time (Granlund-Montgomery): exact for every dividend,
// five instructions instead of the ~20 of a hardware-less integer division.
struct FastDiv {
    unsigned m, s1, s2;
};

inline FastDiv make_fast_div(unsigned d) {   // d >= 1
    unsigned l = 0;
    while ((1ull << l) < d) l++;   // ceil(log2(d))
    FastDiv f;
    f.m = (unsigned)((((1ull << l) - d) << 32) / d + 1);
    f.s1 = l < 1 ? l : 1;
    f.s2 = l > 0 ? l - 1 : 0;
    return f;
}

__device__ __forceinline__ unsigned fast_div(unsigned n, const FastDiv &f) {
    const unsigned t = __umulhi(f.m, n);
    return (t + ((n - t) >> f.s1)) >> f.s2;
}

// max(x, 0) or x, chosen by a floor that does not depend on the lane.  NaN gives 0, as in the reference (its descriptors say
// NOT_PROPAGATE_NAN).  For the loaders of convolutions, whose values come from memory, in one instruction: v_med3_f32 of 0, |x| and
// x is x above zero and 0 below it, and the smallest of those that are numbers, 0, where x is not; with a floor that is NaN
// itself it is the smaller of |x| and x: x as it is.  (A floating-point maximum takes a second instruction for a value that may be
// a signalling NaN; an integer maximum keeps a NaN whose sign is clear.)
__device__ __forceinline__ float relu_floor(bool relu) { return relu ? 0.f : __builtin_nanf(""); }
__device__ __forceinline__ float relu_above(float floor, float x) { return __builtin_amdgcn_fmed3f(floor, __builtin_fabsf(x), x); }

// Activation of V values of a lane.  The usual ones (none, ReLU) are one maximum per value; the others go through one copy of
// their code in turn: inlined once per value, tanh and sigmoid put kilobytes of code between a kernel's last load and its store,
// and skipping them cost a batch-1 launch a microsecond of instruction fetches.
template <int V>
__device__ __forceinline__ void apply_activation(float (&v)[V], int act) {
    if (__builtin_expect(act <= ACT_RELU, 1)) {
        const float floor = relu_floor(act == ACT_RELU);
#pragma unroll
        for (int k = 0; k < V; k++) v[k] = fmaxf(v[k], floor);   // (the maximum of a number and NaN is the number)
        return;
    }
#pragma unroll 1
    for (int n = 0; n < V; n++) {
        const float x = v[0];
        const float y = act == ACT_TANH ? tanhf(x) : 1.0f / (1.0f + __expf(-x));
#pragma unroll
        for (int k = 0; k + 1 < V; k++) v[k] = v[k + 1];
        v[V - 1] = y;
    }
}

// ---- convolution ------------------------------------------------------------------------------------
struct ConvProblem {
    int B, IC, H, W, OC, KH, KW, sh, sw, ph, pw, groups;
    int OH, OW;
    int act;       // Act applied after bias
    int pre_relu;  // apply max(x, 0) to the input while loading it
    int ICg() const { return IC / groups; }
    int OCg() const { return OC / groups; }
    int K() const { return ICg() * KH * KW; }
    // rows of the packed filter matrix when the channels of every tap are padded to a multiple of cpad
    int ICgP(int cpad) const { return (ICg() + cpad - 1) / cpad * cpad; }
    int Kq(int cpad) const { return KH * KW * ICgP(cpad); }
    long long Npix() const { return (long long)B * OH * OW; }
    int OCgP() const { return (OCg() + 3) & ~3; }  // row length of the packed filter matrix
    bool is_depthwise() const { return groups > 1 && IC == groups && OC == groups; }
    double flops() const { return 2.0 * (double)Npix() * OC * K(); }
};

// One implicit-GEMM kernel configuration: block tile BM (output channels) x BN (pixels) x BK, a grid of
// WM x WN x WK wavefronts (WK wavefronts split K) built from MT x MT fp32 MFMA tiles.  `wave_split` selects
// the kernel without LDS staging whose WK wavefronts each own a contiguous range of K (of the block's K slice).
struct ConvVariant {
    const char *name;
    int BM, BN, BK, WM, WN, WK, MT;
    bool wave_split;
    int cpad;   // channel padding of the packed filters this configuration reads
    bool kquad; // packed filters are [k / 4][m][4] (16-byte loads along k) instead of [k][m]
    int threads() const { return 64 * WM * WN * WK; }
    bool fusable_;   // light enough on registers to run inside a fused stage launch
    int precision;   // PREC_FP32, or a reduced-precision mode: bfloat16 / IEEE half filters and inputs, fp32 accumulation
    // packed filters as planes of 16-bit values, [k / 8][plane][m][8]: 3 = the exact split of fp32 values into three bfloat16 terms and
    // 2 = their split into two terms of IEEE half, scaled per output channel (fp32 results from the 16-bit matrix pipe), 1 = one plane
    // rounded to nearest even (the reduced-precision mode on the same kernels), 0 = neither
    int koct = 0;
    // fits a fused stage launch of the wide-register kernel family only (the two-term wave-split configurations)
    bool fusable_wide_ = false;
    int window = 0;   // > 0: stages a window of up to this many input pixels (conv_window.h); for the shapes conv_variant_takes allows
    bool fusable() const { return fusable_ || fusable_wide_; }
    bool needs_wide() const { return fusable_wide_ && !fusable_; }
    int kvec() const { return koct ? 8 : kquad ? 4 : 1; }   // consecutive k of one output channel that lie together
};

int conv_num_variants();
const ConvVariant &conv_variant(int index);
bool conv_variant_measured(const ConvProblem &p, int variant);   // the tuner tries it
bool conv_variant_precise(const ConvProblem &p, int variant);   // fp32 configurations: its operands are as good as fp32 ones for this K
bool conv_variant_takes(const ConvProblem &p, int variant);   // (a launch of another shape runs on a configuration that reads the same packed filters)

struct ConvLaunch {
    int variant = 0;
    int split_k = 1;  // number of grid slices along K; > 1 needs workspace
};

// Grid slices along K a launch configuration really uses (split_k may ask for more than there are K tiles).
int conv_effective_split(const ConvProblem &p, const ConvLaunch &l);
// Floats of workspace a launch configuration needs (split_k partial outputs; large enough for both split-K forms).
size_t conv_workspace_floats(const ConvProblem &p, const ConvLaunch &l);
// Ticket counters the one-kernel split-K form needs: one unsigned per (group, output tile), zero before the
// first launch (the kernel leaves them zero); 0 when the configuration does not split K.
size_t conv_counter_count(const ConvProblem &p, const ConvLaunch &l);
// Bytes from a convolution's first input element to the end of the last quad of channels of its last pixel.
inline unsigned long long conv_input_extent(const ConvProblem &p, int pstride) {
    return (((unsigned long long)p.B * p.H * p.W - 1) * (unsigned long long)pstride + (unsigned long long)((p.IC + 3) & ~3)) * 4ull;
}
// The matrix path indexes packed filter rows with 16 bits and pixels / input offsets with 31 bits.
bool conv_matrix_path_supported(const ConvProblem &p);

// Default configuration from a closed-form occupancy model (num_cus = compute units of the device);
// fusable_only restricts the choice to configurations that can run inside a fused stage launch.
// precision selects the family of configurations (fp32, bfloat16 or half operands).
ConvLaunch conv_pick_launch(const ConvProblem &p, int num_cus, bool fusable_only = false, int precision = PREC_FP32);

// Filter packing for a kernel configuration: w[OC][ICg][KH][KW] -> packed[g][k = (kh*KW + kw)*ICgP + c][OCgP]
// (or [g][k / 4][OCgP][k % 4] for kquad configurations, planes of 16-bit values [g][k / 8][plane][OCgP][k % 8] for koct ones, with two
// words per output channel behind two planes: the factor that undoes its scale, and a bound for what its smallest filters are off by), ICgP = ICg rounded up to the configuration's channel
// padding (zero rows), OCgP = OCg rounded up to 4.  16-bit configurations pack bfloat16 or half (round to nearest even), two
// per float of the returned size.
size_t conv_packed_floats(const ConvProblem &p, const ConvLaunch &l);
size_t conv_packed_floats_max(const ConvProblem &p);   // over all configurations
void launch_pack_filters(const ConvProblem &p, const ConvLaunch &l, const float *w, float *packed, hipStream_t stream);

// How the K slices of a split-K launch meet.  Without `counters` a second kernel adds them on the same stream.  With
// counters (conv_counter_count of them, zero before the first launch) the block that finishes a tile last adds the slices
// inside the kernel; `xcd_local` additionally numbers the grid so that the slices of a tile share an XCD and meet in its L2
// (only for convolutions without groups; others silently use the device-wide form).  All forms add in slice order.
struct SplitKReduce {
    unsigned *counters = nullptr;
    bool xcd_local = false;
    unsigned xcd_map = 0;        // XCC id of the blocks with index % 8 == c, four bits per c (DeviceContext measures it)
    unsigned *fault = nullptr;   // device-visible word in host memory, set to 1 by a block that runs on an unexpected XCC
};

// y = act(conv(x, w) + bias).  `packed` comes from launch_pack_filters, `filters` are those it packed.  `workspace` holds the split_k
// partial outputs (conv_workspace_floats).
void launch_conv_mfma(const ConvProblem &p, const ConvLaunch &l, const TensorView &x, const float *packed, const float *filters,
                      const float *bias, const TensorView &y, float *workspace, const SplitKReduce &reduce, hipStream_t stream,
                      const TensorView *residual = nullptr, bool post_relu = false);

// Several convolutions in a launch, without groups or a residual, each with the packed filters, bias and output of its own.
// A batch: they read the same view (the first member's x) through the same 1 x 1 window.  A mixed one: no two need be alike, and a pool may
// run beside them.
struct ConvBatchMember {
    ConvProblem p;
    const float *packed, *filters, *bias;
    TensorView x, y;
};
constexpr int kMaxConvBatch = 4;
bool conv_variant_batches(int variant);                              // there is a batched kernel on this configuration
bool conv_batchable(const ConvProblem &a, const ConvProblem &b);     // two convolutions of one view may share a launch
void launch_conv_batch(const ConvBatchMember *members, int count, int variant, hipStream_t stream);
bool conv_variant_mixes(int variant);                                // there is a kernel for mixed members on this configuration
bool conv_mixable(const ConvProblem &p, int variant);                // and it takes this one

// Filters of a depth-wise convolution: w[C][1][KH][KW] -> packed[tap][C rounded up to 4] (padding zero).
inline size_t dwconv_packed_floats(const ConvProblem &p) { return (size_t)p.KH * p.KW * ((p.OC + 3) & ~3); }
void launch_pack_depthwise(const ConvProblem &p, const float *w, float *packed, hipStream_t stream);
// Depth-wise convolution (groups == IC == OC), filters from launch_pack_depthwise.  With `more`, the input is
// x + more[0] + ... + more[nmore - 1] (at most kMaxNaryInputs views in all, added left to right before the folded ReLU).
void launch_dwconv(const ConvProblem &p, const TensorView &x, const float *w, const float *bias,
                   const TensorView &y, hipStream_t stream, const TensorView *more = nullptr, int nmore = 0);
bool dwconv_sums_inputs(const ConvProblem &p);   // the kernel for this window can add further inputs in its loader (3 x 3, 5 x 5)

// Direct convolution for any geometry (one thread per output element); used for grouped convolutions
// whose groups are too thin for the matrix path.  `thin` selects the form for 3 x 3 convolutions of 3-channel images
// (conv_thin_applies), which is bound by the bytes of its output and serves first layers at large batches.
inline bool conv_thin_applies(const ConvProblem &p) { return p.groups == 1 && p.IC == 3 && p.KH == 3 && p.KW == 3; }
void launch_conv_direct(const ConvProblem &p, const TensorView &x, const float *w, const float *bias,
                        const TensorView &y, hipStream_t stream, bool thin = false);

// ---- pooling ----------------------------------------------------------------------------------------
struct PoolProblem {
    int B, C, H, W, KH, KW, sh, sw, ph, pw, OH, OW;
    int is_max;  // 1: max over in-range elements, 0: sum of in-range elements / (KH*KW)
};
// With `bias` (one value per channel): y = act(pool(x) + bias[c]).
void launch_pool(const PoolProblem &p, const TensorView &x, const TensorView &y, hipStream_t stream, const float *bias = nullptr,
                 int act = ACT_NONE);
// Window == whole map: one wavefront reduces one (n, c) plane.
struct MixedPool {   // a pool beside mixed convolutions
    PoolProblem p;
    TensorView x, y;
    const float *bias;
    int act;
};
void launch_conv_mixed(const ConvBatchMember *members, int count, const MixedPool *pool, int variant, hipStream_t stream);
void launch_global_pool(const PoolProblem &p, const TensorView &x, const TensorView &y, hipStream_t stream);

// ---- element-wise -----------------------------------------------------------------------------------
struct NaryArgs {
    const float *src[kMaxNaryInputs];
    int src_pstride[kMaxNaryInputs];
    int count;
};
// y = act(src0 (+|*) src1 (+|*) ...), left to right; more than kMaxNaryInputs inputs are handled by the
// caller through accumulation (accumulate != 0 also combines the current contents of y first).
void launch_nary(const NaryArgs &a, int multiply, int accumulate, int act, int B, const TensorView &y, hipStream_t stream);
// y = act(x) for views; act == ACT_NONE is a strided copy.
void launch_unary(const TensorView &x, const TensorView &y, int act, int B, hipStream_t stream);
// From a host tensor's layout (NCHW, dense) to a view.  `nchw` may lie in host memory.  plane > 0: elements between the channels
// of `nchw` where the view is a part of its pixels (one image).
void launch_to_view(const float *nchw, const TensorView &y, int B, hipStream_t stream, long long plane = 0);
// Fill n floats with a deterministic pattern in [-1, 1) (seeded), or with a constant.
void launch_fill_pattern(float *dst, size_t n, unsigned seed, hipStream_t stream, float most = 1.f);   // values up to +-most
void launch_fill_u32(unsigned *dst, size_t n, unsigned value, hipStream_t stream);
void launch_delay(int steps, hipStream_t stream);   // keeps the stream waiting about 4 us per step

}  // namespace ios
