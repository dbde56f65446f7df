// Device-side bodies of the convolution kernels; included by the translation units that instantiate them
// (the stand-alone kernels and the fused stage kernel).
//
// Implicit-GEMM convolution on the CDNA4 fp32 matrix cores, in two forms: ConvTiled stages operand tiles in LDS
// (large problems), ConvWsplit feeds the matrix cores straight from global memory and divides K among the
// wavefronts of a block (small and medium problems, and the bfloat16 mode).  This comment describes ConvTiled;
// ConvWsplit is described at its definition.
//
// GEMM view per group:  Y[m][n] = sum_k Wp[k][m] * X_im2col[k][n]
//   m = output channel inside the group (OCg), n = flattened (image, oh, ow) pixel,
//   k = (kh, kw, c) tap-major with the channels of every tap zero-padded to a multiple of the K tile.
// The filter matrix is pre-packed k-major (launch_pack_filters) so that a block's BK x BM slice is read
// with 16-byte loads along m.  The BK x BN input slice is gathered straight from the NHWC input view:
// consecutive lanes take consecutive quads of channels of a pixel, then the next pixel; because a K tile lies inside one
// filter tap, the tap's (kh, kw), its padding test and its base offset are computed once per tile.  Global loads run PD tiles
// ahead of the math in registers (the loop is latency bound at batch 1, where a block sees only a few
// K tiles), tiles are staged in LDS (double buffered, one barrier per K tile) and consumed by
// v_mfma_f32_32x32x2_f32 / v_mfma_f32_16x16x4_f32: lane l supplies A[k = l / MT][m = l % MT] and
// B[k = l / MT][n = l % MT].
//
// Parallelism for small problems comes from three places: WK wavefronts of a block split each K tile
// and add their accumulators through LDS at the end; split_k grid slices along K write partial tiles
// to a workspace, and the block that finishes a tile last (or a second small kernel) sums them in slice
// order (fixed order, so results do not depend on scheduling; no device-scope fences, which would write
// back and invalidate whole L2s); everything else is M x N tiling.
// The epilogue adds the bias, applies the activation and stores through the output view, i.e. directly
// into the consumer's channel window when the output lives inside a concat buffer.
#pragma once

#include "kernels.h"

#include <algorithm>
#include <climits>
#include <type_traits>

namespace ios {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

struct ConvKernelArgs {
    const float *x;
    const float *wp;
    const float *w;                   // the filters as they were given
    const float *bias;
    float *y;
    float *ws;
    unsigned *counters;               // split-K tickets, one per (group, tile), zero between launches; null: two-kernel split-K
    int H, W, OH, OW, sh, sw, ph, pw;
    int KW;
    int xcd_local;                    // split-K inside one XCD, see below
    unsigned magic_icgp, magic_kw;    // floor(2^32 / d) + 1: exact quotients for dividends < 2^16
    int ICg, ICgP, OCg, OCgP, Kq, OHW, groups;   // Kq = taps * ICgP rows of the packed filter matrix
    int x_ps, y_ps;                   // elements between neighbouring pixels of input and output
    unsigned x_bytes, w_bytes;        // extents of the input view and of the packed filters, both < 2^31
    int Npix;
    int act, pre_relu;
    int split_k, k_chunk;
    int steps_total, steps_chunk, steps_per_wave;   // wave-split kernels: MFMA k-steps in K, in a grid slice, in a wavefront's share of a full slice
    int tiles_m, tiles_n;
    int weights_major;   // 1: consecutive tiles share filter rows (filters larger than the input), 0: share pixels
    int xcd_q, xcd_r;    // tiles_m * tiles_n = 8 * xcd_q + xcd_r
    int tile_div;        // tiles_n (weights_major) or tiles_m
    FastDiv div_tile;    // by tile_div
    FastDiv div_ohw, div_ow;
    // Either the residual form (stand-alone kernels only): y = res + act(conv + bias), then max(., 0) when post_relu; res is a
    // view of the output's shape (res_ps elements between pixels), null for a plain convolution.
    // Or split-K inside one XCD (xcd_local != 0; plain convolutions without groups, counters set): the grid is numbered so
    // that all K slices of an output tile run on the same XCD and meet in that XCD's L2 (see XcdSlot).  xcd_map: the XCC id
    // that blocks with index % 8 == c run on, four bits per c, as measured when the device context was created; fault: a
    // word in host memory that a block finding itself elsewhere sets to 1 (the host then stops using this form);
    // magic_split = floor(2^32 / split_k) + 1: exact quotients by split_k for dividends below 2^26.
    union {
        struct {
            const float *res;
            int res_ps, post_relu;
        };
        struct {
            unsigned *fault;
            unsigned xcd_map, magic_split;
        };
    };
};

// Numbering of the blocks of a launch whose K slices meet inside one XCD.  The dispatcher deals workgroups to the XCDs
// round-robin, so the blocks with index % 8 == c share an XCD.  Class c owns the tiles [c * q + min(c, r), ...) (q + 1 of
// them for c < r, q for the others, where tiles = 8 q + r, the same ranges xcd_tile() uses) and its blocks, in index order,
// are (first tile, slice 0), (first tile, slice 1), ... : a launch has 8 * split * (q + (r > 0)) blocks, of which the last
// ones of the classes c >= r (when r > 0) have no tile and end at once.  `tile` is the value xcd_tile() takes
// (slot-in-class * 8 + c), which also numbers the tile's partial sums and its ticket: those arrays have
// 8 * (q + (r > 0)) entries.
struct XcdSlot {
    int tile, slice;
    bool idle;
};
__host__ __device__ inline int xcd_padded_tiles(int tiles) { return 8 * ((tiles + 7) / 8); }
__host__ __device__ inline int xcd_grid_blocks(int tiles, int split) { return xcd_padded_tiles(tiles) * split; }
__host__ __device__ inline XcdSlot xcd_slot(int local, int tile_in_class, int xcd_q, int xcd_r, int split) {
    // local: index of the block inside the launch (or inside its item of a fused launch); tile_in_class = (local / 8) / split
    const int c = local & 7;
    XcdSlot s;
    s.slice = (local >> 3) - tile_in_class * split;
    s.tile = tile_in_class * 8 + c;
    s.idle = tile_in_class >= xcd_q + (c < xcd_r ? 1 : 0);
    return s;
}

// XCC id of the executing wavefront (bits 3:0 of the hardware register XCC_ID)
__device__ __forceinline__ unsigned xcc_id() { return __builtin_amdgcn_s_getreg(20 | (3 << 11)); }

// One block of an XCD-local split-K launch: its slot, and the check that the dispatcher put it where the numbering assumes.
// `block` is the block's index in the whole launch (the XCD follows from it), `local` its index inside the convolution.
__device__ __forceinline__ XcdSlot xcd_enter(const ConvKernelArgs &a, int block, int local) {
    const XcdSlot s = xcd_slot(local, (int)__umulhi((unsigned)local >> 3, a.magic_split), a.xcd_q, a.xcd_r, a.split_k);
    const unsigned expected = (a.xcd_map >> (4 * (block & 7))) & 15u;
    if (xcc_id() != expected && threadIdx.x == 0) __hip_atomic_store(a.fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return s;
}

// Partial sums and tickets of the one-kernel split-K.  Device-wide form: the slices of a tile run on different XCDs, whose
// L2s are not coherent with each other, so partial sums travel with agent-scope stores and loads (written through to and
// read from memory) and the ticket is an agent-scope atomic.  XCD-local form: all slices share one L2; plain stores are
// written through the L1 to that L2, the ticket is a workgroup-scope atomic (executed in the L2), and the sums are read
// with workgroup-scope loads, which do not use a line the L1 might hold.  In both forms a block waits for its stores to
// be acknowledged before it takes its ticket.
template <bool LOCAL>
__device__ __forceinline__ void partial_store(float *p, float v) {
    if constexpr (LOCAL) *p = v;
    else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool LOCAL>
__device__ __forceinline__ float partial_load(const float *p) {
    if constexpr (LOCAL) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// thread 0 of the block: draws the tile's ticket; the block that draws the last one puts the counter back to zero
template <bool LOCAL>
__device__ __forceinline__ int draw_ticket(unsigned *counter, int split_k) {
    unsigned ticket;
    if constexpr (LOCAL) ticket = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else ticket = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int last = ticket == (unsigned)split_k - 1u ? 1 : 0;
    if (last) {
        if constexpr (LOCAL) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return last;
}

// Workgroups are dealt round-robin to the 8 XCDs, each with its own L2.  Tiles are renumbered so that an XCD
// receives a contiguous range of them, and the range runs along the operand that is cheaper to duplicate: the
// more expensive operand (filters at batch 1, activations at large batch) is then fetched into one L2 only.
__device__ __forceinline__ void xcd_tile(const ConvKernelArgs &a, int block, int &tm, int &tn) {
    // XCD x owns tiles [x * q + min(x, r), ...): q + 1 tiles for the first r XCDs, q for the others
    const int xcd = block & 7, slot = block >> 3;
    const int t = slot + xcd * a.xcd_q + min(xcd, a.xcd_r);
    const int q2 = (int)fast_div((unsigned)t, a.div_tile);
    const int rest = t - q2 * a.tile_div;
    tm = a.weights_major ? q2 : rest;
    tn = a.weights_major ? rest : q2;
}

typedef unsigned int uintx4 __attribute__((ext_vector_type(4)));
typedef float floatx4_u __attribute__((ext_vector_type(4), aligned(4)));   // 16 bytes at any 4-byte boundary

// Epilogue of four consecutive output channels m ... m + 3 of group g at pixel nn (all four accumulators of a lane that belong
// together, see Mfma::row): bias, activation, residual operand, one 16-byte store (element by element where the group ends
// inside).  RES, the residual form, is a compile-time property of a body: the plain form, which every fused stage launch uses,
// carries no test for it.
template <bool RES>
__device__ __forceinline__ void finish_quad(const ConvKernelArgs &a, floatx4 v, floatx4 bias, int g, int m, int nn) {
    const int channel = g * a.OCg + m;
    float out[4] = {v[0] + bias[0], v[1] + bias[1], v[2] + bias[2], v[3] + bias[3]};
    apply_activation(out, a.act);
    v = floatx4{out[0], out[1], out[2], out[3]};
    float *y = a.y + (long long)nn * a.y_ps + channel;
    const float *res = nullptr;
    if constexpr (RES) res = a.res + (long long)nn * a.res_ps + channel;
    if (m + 3 < a.OCg) {
        if constexpr (RES) {
            v += (floatx4)*reinterpret_cast<const floatx4_u *>(res);
            if (a.post_relu)
#pragma unroll
                for (int c = 0; c < 4; c++) v[c] = fmaxf(v[c], 0.0f);
        }
        *reinterpret_cast<floatx4_u *>(y) = v;
    } else {
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (m + c < a.OCg) {
                if constexpr (RES) {
                    v[c] += res[c];
                    if (a.post_relu) v[c] = fmaxf(v[c], 0.0f);
                }
                y[c] = v[c];
            }
    }
}

// The same for N pixels STEP apart from `first` on, below n_end; factor: of the four channels.
template <bool RES, int N, int STEP>
__device__ __forceinline__ void finish_quads(const ConvKernelArgs &a, floatx4 (&v)[N], floatx4 bias, floatx4 factor, int g, int m, int first, int n_end) {
    if (m >= a.OCg) return;
    float out[4 * N];
#pragma unroll
    for (int r = 0; r < N; r++)
#pragma unroll
        for (int c = 0; c < 4; c++) out[4 * r + c] = __builtin_fmaf(v[r][c], factor[c], bias[c]);
    apply_activation(out, a.act);
    const int channel = g * a.OCg + m;
#pragma unroll
    for (int r = 0; r < N; r++) {
        const int nn = first + r * STEP;
        if (nn >= n_end) break;
        floatx4 w = {out[4 * r], out[4 * r + 1], out[4 * r + 2], out[4 * r + 3]};
        float *y = a.y + (long long)nn * a.y_ps + channel;
        const float *res = nullptr;
        if constexpr (RES) res = a.res + (long long)nn * a.res_ps + channel;
        if (m + 3 < a.OCg) {
            if constexpr (RES) {
                w += (floatx4)*reinterpret_cast<const floatx4_u *>(res);
                if (a.post_relu)
#pragma unroll
                    for (int c = 0; c < 4; c++) w[c] = fmaxf(w[c], 0.0f);
            }
            *reinterpret_cast<floatx4_u *>(y) = w;
        } else {
#pragma unroll
            for (int c = 0; c < 4; c++)
                if (m + c < a.OCg) {
                    if constexpr (RES) {
                        w[c] += res[c];
                        if (a.post_relu) w[c] = fmaxf(w[c], 0.0f);
                    }
                    y[c] = w[c];
                }
        }
    }
}

// bias of output channels m ... m + 3 of group g (what lies behind the last bias value is not used; the arena goes on there)
__device__ __forceinline__ floatx4 bias_quad(const ConvKernelArgs &a, int g, int m) {
    return *reinterpret_cast<const floatx4_u *>(a.bias + g * a.OCg + min(m, a.OCg - 1));
}

// Raw buffer loads: a 32-bit byte offset against a base + extent descriptor; offsets at or beyond the extent
// read as zero, so an invalid element (padding, channel padding, tile overhang) is a load from kOutOfRange
// and no branch or select on the loaded value is needed.
constexpr unsigned kOutOfRange = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const float *base, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), 0, bytes, 0x00020000);
}
// `scalar_offset` must be wavefront-uniform; it is added to the address after the range check of `byte_offset`.
__device__ __forceinline__ float buffer_load_f32(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, unsigned scalar_offset = 0) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, byte_offset, scalar_offset, 0));
}
__device__ __forceinline__ floatx4 buffer_load_f32x4(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, unsigned scalar_offset = 0) {
    const uintx4 v = __builtin_amdgcn_raw_buffer_load_b128(r, byte_offset, scalar_offset, 0);
    floatx4 f = {__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w)};
    return f;
}

typedef unsigned int uintx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uintx2 buffer_load_u32x2(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, unsigned scalar_offset = 0) {
    return __builtin_amdgcn_raw_buffer_load_b64(r, byte_offset, scalar_offset, 0);
}

template <int MT>
struct Mfma;

template <>
struct Mfma<32> {
    static constexpr int KSTEP = 2;
    static constexpr int ACC = 16;
    typedef floatx16 acc_t;
    __device__ static __forceinline__ acc_t run(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
    }
    // row of accumulator element v held by `lane` inside the 32 x 32 tile; the column is lane % 32
    __device__ static __forceinline__ int row(int v, int lane) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); }
};

template <>
struct Mfma<16> {
    static constexpr int KSTEP = 4;
    static constexpr int ACC = 4;
    typedef floatx4 acc_t;
    __device__ static __forceinline__ acc_t run(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ int row(int v, int lane) { return 4 * (lane >> 4) + v; }
};

__device__ __forceinline__ floatx4 channel_scale_quad(const ConvKernelArgs &a, int g, int m);   // (with the two-term operands below)
__device__ __forceinline__ floatx4 channel_least_quad(const ConvKernelArgs &a, int g, int m);
template <int MT, int TM, int TN, typename Acc>
__device__ __forceinline__ void scale_channels(const ConvKernelArgs &a, Acc (&acc)[TM][TN], int g, int m_base);

// Bias (and what belongs to two terms, SCALED) of the four output channels per 32 rows that this lane finishes in the epilogue, m_base: row 0 of the
// wavefront's tiles; requested before the last barriers of a body, which their latency then overlaps.
template <int TM>
struct TailConstants { floatx4 bias[TM], factor[TM], least[TM]; };
template <int MT, bool SCALED, int TM>
__device__ __forceinline__ void tail_constants(const ConvKernelArgs &a, TailConstants<TM> &c, int g, int m_base) {
    if constexpr (MT == 32) {
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int m = m_base + i * 32 + 4 * (threadIdx.x & 7);
            c.bias[i] = bias_quad(a, g, m);
            if constexpr (SCALED) {
                c.factor[i] = channel_scale_quad(a, g, m);
                c.least[i] = channel_least_quad(a, g, m);
            }
        }
    }
}

// LDS of a wavefront in the epilogue: its tiles, pixel by pixel with the quads of channels exchanged so that eight pixels' quads and
// eight quads of a pixel meet all banks, and the constants
constexpr int tail_floats(int tm, int tn) { return tm * tn * 1024 + tm * 64; }
// what the lanes of a wavefront have written to LDS is there for its other lanes (accesses of a wavefront are executed in order)
__device__ __forceinline__ void wavefront_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Tail of the LDS-tiled kernels once a block holds its accumulators (wavefronts with wk == 0; the others only take part in the
// barriers): the split-K exchange in its three forms, then bias, activation and the store through the output view.
// `smem` is free when this is called.
// SCALED: the sums are those of scaled filters (see split_half2) where `scaled` says so, of the filters as they were given otherwise.
// THROUGH_LDS: `smem` holds tail_floats per wavefront too, and results are stored by whole lines of channels.
template <int MT, int BM, int BN, int TM, int TN, int WM, int WN, bool RES, bool SCALED = false, bool THROUGH_LDS = MT == 32>
__device__ __forceinline__ void tiled_tail(const ConvKernelArgs &a, float *smem, typename Mfma<MT>::acc_t (&acc)[TM][TN], int tile, int g, int z,
                                           int m0, int n0, int wm, int wn, int wk, const TailConstants<TM> &c, int n_limit = INT_MAX, bool scaled = false) {
    using M = Mfma<MT>;
    const int n_end = min(a.Npix, n_limit);   // (a tile that ends before the tensor does)
    constexpr int WTM = BM / WM, WTN = BN / WN;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int lc = lane % MT;
    // ---- split-K ----------------------------------------------------------------------------------------------
    if (a.split_k > 1) {
        if (SCALED && scaled) {   // (slices meet as sums of the filters as they were given)
            scale_channels<MT>(a, acc, g, m0 + wm * WTM);
            scaled = false;
        }
        if (a.counters == nullptr) {
            // two-kernel form: store this slice's partial tile; splitk_reduce_kernel adds the slices, bias and activation
            const size_t channels = (size_t)a.groups * a.OCg;
            float *wsz = a.ws + (size_t)z * channels * (size_t)a.Npix + (size_t)g * a.OCg;
            if (wk == 0) {
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int nn = n0 + wn * WTN + j * MT + lc;
                    if (nn >= n_end) continue;
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int v = 0; v < M::ACC; v++) {
                            const int m = m0 + wm * WTM + i * MT + M::row(v, lane);
                            if (m < a.OCg) wsz[(size_t)nn * channels + m] = acc[i][j][v];
                        }
                }
            }
            return;
        }
        // one-kernel form: every slice stores its partial tile in accumulator layout ([element][thread], so a
        // wavefront writes 256 contiguous bytes), then takes a ticket on the tile's counter; the block that
        // draws the last ticket adds all slices in slice order (its own included, so the sum does not depend
        // on which block came last) and runs the epilogue.  Partials and tickets move with device-scope
        // atomics, which are coherent across the per-XCD L2s without cache-wide write-backs or invalidations;
        // the wait on the outstanding stores before the barrier orders a block's partials before its ticket.
        constexpr int T0 = 64 * WM * WN;
        constexpr int E = TM * TN * M::ACC;
        static_assert(T0 * E == BM * BN, "accumulator layout covers the tile");
        const size_t tiles = (size_t)xcd_padded_tiles(a.tiles_m * a.tiles_n);   // (both forms size their arrays for the padded count)
        float *slices = a.ws + (((size_t)g * tiles + tile) * a.split_k) * (size_t)(BM * BN);
        unsigned *counter = a.counters + (size_t)g * tiles + tile;
        int *last_flag = reinterpret_cast<int *>(smem);
        auto exchange = [&](auto local) -> bool {   // true: this block drew the last ticket and holds the sum of all slices
            constexpr bool LOCAL = decltype(local)::value;
            if (wk == 0) {
                float *mine = slices + (size_t)z * (BM * BN) + tid;
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int v = 0; v < M::ACC; v++) partial_store<LOCAL>(mine + ((i * TN + j) * M::ACC + v) * T0, acc[i][j][v]);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (tid == 0) *last_flag = draw_ticket<LOCAL>(counter, a.split_k);
            __syncthreads();
            const int last = *last_flag;
            __syncthreads();   // (the flag's place is a wavefront's in the epilogue)
            if (last == 0) return false;
            if (wk == 0) {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int v = 0; v < M::ACC; v++) acc[i][j][v] = 0.f;
                for (int s = 0; s < a.split_k; s++) {
                    const float *theirs = slices + (size_t)s * (BM * BN) + tid;
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int j = 0; j < TN; j++)
#pragma unroll
                            for (int v = 0; v < M::ACC; v++) acc[i][j][v] += partial_load<LOCAL>(theirs + ((i * TN + j) * M::ACC + v) * T0);
                }
            }
            return true;
        };
        const bool last = a.xcd_local ? exchange(std::true_type{}) : exchange(std::false_type{});
        if (!last) return;
    }

    // ---- epilogue -------------------------------------------------------------------------------------------
    if constexpr (THROUGH_LDS) {
        // A lane holds four channels of a pixel, its neighbour the next pixel's: stored like that, every 16 bytes of a wavefront's store
        // go to another line, and the L2 takes a request for each.  So the tiles pass through LDS; eight lanes then take the 128 bytes
        // of a pixel, a lane the same four channels of every pixel of a tile.  What runs once is short (one copy of the code for all
        // tiles: instructions that a launch has not run yet come from memory, a line at a time).  64 x 128 tiles of 17 x 17 maps at
        // batch 64, 14 MB of results: 6.2 -> 3.9 us behind the K loop.
        if (wk != 0) return;
        float *place = smem + (wm * WN + wn) * tail_floats(TM, TN), *constants = place + TM * TN * 1024;
        const int quad = lane & 7, px = lane >> 3;
#pragma unroll
        for (int i = 0; i < TM; i++) {
            if (lane < 8) {
                *reinterpret_cast<floatx4 *>(constants + i * 64 + 4 * lane) = c.bias[i];
                if constexpr (SCALED) *reinterpret_cast<floatx4 *>(constants + i * 64 + 32 + 4 * lane) = c.factor[i];
            }
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < M::ACC / 4; q++)
                    *reinterpret_cast<floatx4 *>(place + (i * TN + j) * 1024 + lc * 32 + ((2 * q + (lane >> 5)) ^ (lc & 7)) * 4) =
                        floatx4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        }
        wavefront_lds_fence();
#pragma unroll 1
        for (int t = 0; t < TM * TN; t++) {
            const int i = t / TN, j = t - i * TN;
            const floatx4 bias = *reinterpret_cast<const floatx4 *>(constants + i * 64 + 4 * quad);
            floatx4 factor = {1.f, 1.f, 1.f, 1.f};
            if (SCALED && scaled) factor = *reinterpret_cast<const floatx4 *>(constants + i * 64 + 32 + 4 * quad);
            floatx4 v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = *reinterpret_cast<const floatx4 *>(place + t * 1024 + (8 * r + px) * 32 + (quad ^ px) * 4);
            finish_quads<RES, 4, 8>(a, v, bias, factor, g, m0 + wm * WTM + i * MT + 4 * quad, n0 + wn * WTN + j * MT + px, n_end);
        }
    } else {
    if (wk == 0) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int q = 0; q < M::ACC / 4; q++) {
                const int m = m0 + wm * WTM + i * MT + M::row(4 * q, lane);
                if (m >= a.OCg) continue;
                const floatx4 bias = bias_quad(a, g, m);
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int nn = n0 + wn * WTN + j * MT + lc;
                    if (nn >= n_end) continue;
                    const floatx4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                    finish_quad<RES>(a, v, bias, g, m, nn);
                }
            }
    }
    }
}

template <int BM, int BN, int BK, int WM, int WN, int WK, int MT, int PD>
struct ConvTiled {
    using M = Mfma<MT>;
    static constexpr int T = 64 * WM * WN * WK;
    static constexpr int THREADS = T;
    static constexpr int CPAD = BK;   // channel padding of the packed filters: a K tile never straddles two taps
    static constexpr int PAD = MT == 16 ? 16 : 4;   // MT 16 reads four rows per instruction: rows must not share banks
    static constexpr int LDA = BM + PAD, LDB = BN + PAD;
    static constexpr int TILE_FLOATS = 2 * BK * (LDA + LDB);
    static constexpr int RED_FLOATS = (WK - 1) * BM * BN;
    // The LDS-tiled bodies need 85 registers and more per lane; inside a fused stage launch they would lower the
    // occupancy of every other operator (the wave-split bodies that serve small problems need 32-72), so they
    // only run as stand-alone kernels.
    static constexpr bool FUSABLE = false;
    // Results go through LDS where two blocks still fit a compute unit (128 x 128 tiles, 33 -> 66 KB: 48 -> 192 channels 1 x 1 on 35 x 35 at
    // batch 64 41 -> 35 us, 192 -> 256 94 -> 90, 96 -> 192 3 x 3 313 -> 310; 192 x 128 tiles, 41 -> 99 KB: 41 -> 37, but 120 -> 136 and 268 -> 293).
    static constexpr int TAIL_FLOATS = WM * WN * tail_floats(BM / WM / MT, BN / WN / MT);
    static constexpr bool THROUGH_LDS = MT == 32 && TAIL_FLOATS <= 20480;
    static constexpr int SMEM_FLOATS = std::max({TILE_FLOATS, RED_FLOATS, THROUGH_LDS ? TAIL_FLOATS : 0});

    // one block: output tile `tile` of group `g`, K slice `z`; smem holds SMEM_FLOATS floats, 16-byte aligned
    template <bool RES = false>
    __device__ static __forceinline__ void run(const ConvKernelArgs &a, float *smem, int tile, int g, int z) {
    constexpr int WTM = BM / WM, WTN = BN / WN;
    constexpr int TM = WTM / MT, TN = WTN / MT;
    constexpr int KSLICE = BK / WK;
    constexpr int A_VEC_PER_ROW = BM / 4;
    constexpr int A_SLOTS = BK * A_VEC_PER_ROW;
    constexpr int A_ITERS = (A_SLOTS + T - 1) / T;
    constexpr int B_QUADS = BK / 4;                      // quads of channels of a pixel in a K tile
    constexpr int B_ITERS = B_QUADS * BN / T;            // pixels a thread stages, T / B_QUADS apart
    static_assert(WTM % MT == 0 && WTN % MT == 0, "wave tile must be a multiple of the MFMA tile");
    static_assert(KSLICE % M::KSTEP == 0, "K slice per wavefront must be a multiple of the MFMA depth");
    static_assert(T % B_QUADS == 0 && B_QUADS * BN % T == 0 && BN % (T / B_QUADS) == 0, "input loader shape");
    float *As = smem;                  // [2][BK][LDA]
    float *Bs = smem + 2 * BK * LDA;   // [2][BK][LDB]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: keeps per-wavefront K ranges and loop control on the SALU
    const int wn = wave % WN;
    const int wm = (wave / WN) % WM;
    const int wk = wave / (WN * WM);

    int tm, tn;
    xcd_tile(a, tile, tm, tn);
    const int m0 = tm * BM;
    const int n0 = tn * BN;
    const int k_begin = z * a.k_chunk;
    const int k_end = min(a.Kq, k_begin + a.k_chunk);
    const int nkt = (k_end - k_begin) / BK;   // Kq and k_chunk are multiples of BK

    // ---- per-thread loader state ---------------------------------------------------------------------
    const int bq = tid % B_QUADS;   // this thread's quad of channels inside a K tile
    const int bn_l = tid / B_QUADS; // its first pixel inside the output tile
    int ih0[B_ITERS], iw0[B_ITERS];
    unsigned n_kill[B_ITERS], b_off[B_ITERS];   // byte offset of (image, ih0, iw0, group, quad); may wrap below zero, the tap offset brings it back
#pragma unroll
    for (int i = 0; i < B_ITERS; i++) {
        const int n = n0 + bn_l + i * (T / B_QUADS);
        n_kill[i] = n < a.Npix ? 0u : kOutOfRange;
        const int nn = n < a.Npix ? n : 0;
        const int b = (int)fast_div((unsigned)nn, a.div_ohw);
        const int r = nn - b * a.OHW;
        const int oh = (int)fast_div((unsigned)r, a.div_ow);
        const int ow = r - oh * a.OW;
        ih0[i] = oh * a.sh - a.ph;
        iw0[i] = ow * a.sw - a.pw;
        b_off[i] = (((unsigned)(b * a.H + ih0[i]) * (unsigned)a.W + (unsigned)iw0[i]) * (unsigned)a.x_ps + (unsigned)(g * a.ICg + 4 * bq)) * 4u;
    }
    const __amdgpu_buffer_rsrc_t xr = buffer_of(a.x, a.x_bytes);
    const __amdgpu_buffer_rsrc_t wr = buffer_of(a.wp, a.w_bytes);
    // constant per-thread byte offsets inside a tile: filter element (row, 4 columns) and input row (channel)
    unsigned a_off[A_ITERS];
#pragma unroll
    for (int i = 0; i < A_ITERS; i++) {
        const int slot = tid + i * T;
        const int row = slot / A_VEC_PER_ROW;
        const int c4 = slot % A_VEC_PER_ROW;
        const bool ok = (A_SLOTS % T == 0 || slot < A_SLOTS) && m0 + c4 * 4 < a.OCgP;
        a_off[i] = ok ? (unsigned)(((size_t)g * a.Kq * a.OCgP + (size_t)row * a.OCgP + m0 + c4 * 4) * 4) : kOutOfRange;
    }
    floatx4 a_reg[PD][A_ITERS];
    floatx4 b_reg[PD][B_ITERS];

    // K is ordered tap-major: row k of the packed filters is (tap = k / ICgP, c = k % ICgP) with ICgP a
    // multiple of BK, so a K tile lies inside one filter tap: (kh, kw) and the tile's base offsets are scalar and
    // the padding test is one compare pair per pixel.
    auto load_tile = [&](int kt, floatx4(&ar)[A_ITERS], floatx4(&br)[B_ITERS]) {
        const int k0 = k_begin + kt * BK;
        const int tap = (int)__umulhi((unsigned)k0, a.magic_icgp);
        const int c0 = k0 - tap * a.ICgP;
        const int kh = a.KW == 1 ? tap : (int)__umulhi((unsigned)tap, a.magic_kw);
        const int kw = tap - kh * a.KW;
        const unsigned w_tile = (unsigned)(k0 * a.OCgP) * 4u;
        const unsigned tile_kill = kt < nkt ? 0u : kOutOfRange;   // tiles past the end of the K range load zeros
#pragma unroll
        for (int i = 0; i < A_ITERS; i++) ar[i] = buffer_load_f32x4(wr, (a_off[i] + w_tile) | tile_kill);
        // invalid elements get the top offset bit set, which is beyond every extent; plain bit arithmetic keeps
        // the loads of a tile in one basic block so that they are issued back to back
        const unsigned x_tile = (unsigned)((kh * a.W + kw) * a.x_ps + c0) * 4u;
        const int c_left = a.ICg - c0 - 4 * bq;   // real channels from this quad on
        const unsigned pad = (unsigned)(c_left - 1) & kOutOfRange;   // sign bit: the quad is channel padding
#pragma unroll
        for (int i = 0; i < B_ITERS; i++) {
            const unsigned in_h = (unsigned)(ih0[i] + kh) < (unsigned)a.H ? 1u : 0u;
            const unsigned in_w = (unsigned)(iw0[i] + kw) < (unsigned)a.W ? 1u : 0u;
            const unsigned kill = (((in_h & in_w) ^ 1u) << 31) | n_kill[i] | tile_kill | pad;
            br[i] = buffer_load_f32x4(xr, (b_off[i] + x_tile) | kill);
#pragma unroll
            for (int u = 1; u < 4; u++) br[i][u] = u < c_left ? br[i][u] : 0.f;   // channels of the quad beyond the group's
        }
    };

    const float floor = relu_floor(a.pre_relu != 0);
    auto store_tile = [&](int buf, const floatx4(&ar)[A_ITERS], const floatx4(&br)[B_ITERS]) {
        float *Ab = As + buf * BK * LDA;
        float *Bb = Bs + buf * BK * LDB;
#pragma unroll
        for (int i = 0; i < A_ITERS; i++) {
            const int slot = tid + i * T;
            if (A_SLOTS % T == 0 || slot < A_SLOTS) {
                const int row = slot / A_VEC_PER_ROW;
                const int c4 = slot % A_VEC_PER_ROW;
                *reinterpret_cast<floatx4 *>(Ab + row * LDA + c4 * 4) = ar[i];
            }
        }
#pragma unroll
        for (int i = 0; i < B_ITERS; i++) {
            // folded ReLU of the producer
#pragma unroll
            for (int u = 0; u < 4; u++)
                Bb[(4 * bq + u) * LDB + bn_l + i * (T / B_QUADS)] = relu_above(floor, br[i][u]);
        }
    };

    typename M::acc_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < M::ACC; v++) acc[i][j][v] = 0.f;

    // ---- main loop: global -> registers (PD tiles ahead) -> LDS (double buffered) -> MFMA -----------------
    // Register stage s holds tile kt with kt % PD == s.  In iteration kt the stage of tile kt is free (the
    // tile already sits in LDS buffer kt & 1), so it is refilled with tile kt + PD; the stage of tile kt + 1,
    // requested PD - 1 iterations ago, is written to the other LDS buffer after the math.
    // The loop runs in rounds of PD tiles with a straight-line body; tiles past the end of the K range are
    // loaded as zeros (see tile_kill) and cost at most PD - 1 idle MFMA tiles per block.
#pragma unroll
    for (int s = 0; s < PD; s++) load_tile(s, a_reg[s], b_reg[s]);
    store_tile(0, a_reg[0], b_reg[0]);
    __syncthreads();
    const int lk = lane / MT;   // k offset of this lane inside an MFMA step
    const int lc = lane % MT;   // row (A) / column (B) of this lane inside an MFMA tile
    for (int kt0 = 0; kt0 < nkt; kt0 += PD) {
#pragma unroll
        for (int s = 0; s < PD; s++) {
            const int kt = kt0 + s;
            const int buf = kt & 1;
            load_tile(kt + PD, a_reg[s], b_reg[s]);
            const float *Ab = As + buf * BK * LDA + (wk * KSLICE + lk) * LDA + wm * WTM + lc;
            const float *Bb = Bs + buf * BK * LDB + (wk * KSLICE + lk) * LDB + wn * WTN + lc;
#pragma unroll
            for (int kk = 0; kk < KSLICE; kk += M::KSTEP) {
                float av[TM], bv[TN];
#pragma unroll
                for (int i = 0; i < TM; i++) av[i] = Ab[kk * LDA + i * MT];
#pragma unroll
                for (int j = 0; j < TN; j++) bv[j] = Bb[kk * LDB + j * MT];
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) acc[i][j] = M::run(av[i], bv[j], acc[i][j]);
            }
            store_tile(buf ^ 1, a_reg[(s + 1) % PD], b_reg[(s + 1) % PD]);
            __syncthreads();
        }
    }

    // ---- fold the WK wavefronts that worked on the same output tile -------------------------------------------
    if (WK > 1) {
        constexpr int PER_WAVE = TM * TN * M::ACC;        // accumulator floats per lane
        constexpr int MN_WAVES = WM * WN;
        float *red = smem;                                // [(WK-1)][PER_WAVE][MN_WAVES * 64]
        const int slot = (wm * WN + wn) * 64 + lane;
        if (wk > 0) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int v = 0; v < M::ACC; v++)
                        red[((size_t)(wk - 1) * PER_WAVE + (i * TN + j) * M::ACC + v) * (MN_WAVES * 64) + slot] =
                            acc[i][j][v];
        }
        __syncthreads();
        if (wk == 0) {
            for (int s = 0; s < WK - 1; s++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int v = 0; v < M::ACC; v++)
                            acc[i][j][v] += red[((size_t)s * PER_WAVE + (i * TN + j) * M::ACC + v) * (MN_WAVES * 64) + slot];
        }
        __syncthreads();
    }

    TailConstants<TM> constants;
    tail_constants<MT, false>(a, constants, g, m0 + wm * WTM);
    tiled_tail<MT, BM, BN, TM, TN, WM, WN, RES, false, THROUGH_LDS>(a, smem, acc, tile, g, z, m0, n0, wm, wn, wk, constants);
    }   // run
};

// ---- LDS-tiled kernel on the bfloat16 matrix pipe with fp32-exact operands ---------------------------------------------------
// The fp32 matrix instructions run at 1/16 of the rate of the bfloat16 ones (measured: 149-156 against 2340 TFLOP/s).  An fp32
// number is exactly the sum of three bfloat16 numbers (its 24 significant bits in three groups of eight: x = hi + mid + lo,
// each term obtained by truncating the remainder to its leading eight bits, all subtractions exact), so a product of two
// fp32 numbers is the sum of nine products of bfloat16 numbers, each exact in fp32.  This kernel adds the six largest of them
// (hi*hi, hi*mid, mid*hi, hi*lo, mid*mid, lo*hi) on v_mfma_f32_32x32x16_bf16 with fp32 accumulation; the three that are left
// out are below 2^-23 of the product, the size of the rounding error of an fp32 multiplication.  Six instructions of 8 passes
// cover 16 k where the fp32 form needs eight instructions of 16 passes: 2.7 times the matrix throughput at fp32 accuracy.
//
// Filters are split when they are packed: three planes of bfloat16 in octets of eight consecutive k, [k / 8][plane][m][8],
// which is the operand layout of the instruction (lane l: row l % 32, k = 8 * (l / 32) ... + 7): a wavefront reads the filter
// operand of a 32 x 32 tile straight from global memory, one 16-byte load per lane and plane, PD K tiles ahead (the filters
// are small and stay in the caches; the LDS, whose bandwidth bounds this kernel, carries the inputs only).  Inputs are split
// by the thread that stages them: eight channels of one pixel, two 16-byte loads PD K tiles ahead into registers, three 16-byte
// LDS stores into [plane][pixel][octet][8 k], again the operand layout: an input operand is one conflict-free 16-byte LDS load
// per lane and plane.  K tiles are 16 deep and lie inside one filter tap (channels padded to 16); LDS is double buffered, one
// barrier per K tile.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// the three bfloat16 terms of an fp32 value, each in the upper half of a word (hi + mid + lo == x exactly for normal x)
__device__ __host__ inline void split3(float x, unsigned &hi, unsigned &mid, unsigned &lo) {
    union { float f; unsigned u; } v, r;
    v.f = x;
    hi = v.u & 0xffff0000u;
    r.u = hi;
    v.f = x - r.f;
    mid = v.u & 0xffff0000u;
    r.u = mid;
    v.f = v.f - r.f;
    lo = v.u & 0xffff0000u;
}

// three bfloat16 terms of eight fp32 values, each term as four words of two bfloat16 (lower k in the lower half)
__device__ __forceinline__ void split_bf16x3(const float (&x)[8], uintx4 &hi, uintx4 &mid, uintx4 &lo) {
    unsigned h[8], m[8], l[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        h[i] = __float_as_uint(x[i]) & 0xffff0000u;
        const float r1 = x[i] - __uint_as_float(h[i]);
        m[i] = __float_as_uint(r1) & 0xffff0000u;
        const float r2 = r1 - __uint_as_float(m[i]);
        l[i] = __float_as_uint(r2);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {   // high halves of two words side by side
        hi[i] = __builtin_amdgcn_perm(h[2 * i + 1], h[2 * i], 0x07060302u);
        mid[i] = __builtin_amdgcn_perm(m[2 * i + 1], m[2 * i], 0x07060302u);
        lo[i] = __builtin_amdgcn_perm(l[2 * i + 1], l[2 * i], 0x07060302u);
    }
}

// ---- fp32 operands as two terms of IEEE half -------------------------------------------------------------------------------
// x = hi + lo with hi the nearest half of x and lo the nearest half of the remainder holds 23 of an fp32 value's 24 significant
// bits (the remainder has twelve bits and a sign, a half takes eleven of them: the last one is lost for a quarter of the values,
// the other values are exact).  A product is then the sum of three products of halves, each exact in fp32 (hi * hi, hi * lo,
// lo * hi; the fourth is below 2^-22 of it), against the six of three bfloat16 terms: half the matrix instructions, two operand
// planes instead of three.  What bounds an fp32 result is the rounding of its sum, and a sum of half as many terms is rounded half as
// often.  Below K = 64 the lost bits of the operands weigh more (see conv_variant_precise): the tuner does not let the two-term
// kernels compete there.
//
// A half has five bits of exponent, so operands are scaled by powers of two (exact).  Filters: every output channel by its own factor,
// which puts its largest filter value into [2^14, 2^15).  Inputs: a tile's by one that its first values choose, with room for two to four
// more binades below 2^15; where a later value is beyond that, the tile is computed once more with another.  (In the wave-split kernels
// the lanes that stage a pixel also hold its sums: every pixel has its own factor, and the sums follow when it shrinks.)  The lower terms
// are taken times 2^8 (inputs) and 2^4 (filters) and their partners in a product, the upper terms, times 2^-8 and 2^-4: as far up from the
// subnormal halves as the others come down to them.  So an input keeps its 23 bits down to 2^-11 scaled, 2^-22 of the largest or less, a filter
// down to 2^-7, 2^-21 of the largest of its channel.
//
// What lies below is off by an amount that does not shrink with it.  No result may show that, whatever the others are: filters like that are
// known when they are packed (channel_least), octets of inputs that are all below are counted where they are staged (InputWatch), and
// a result of theirs that is not 2^22 times what they may have added to it is computed again in fp32 from the filters as they were given
// (sums_hold), as is one that an infinite value takes part in.  (Of values of a normal distribution one filter in 10^6 is that small, one
// octet in 10^7, and few of their results.  Every single input held against the window costs the pipelined kernels 8 % more; where the
// largest of eight neighbouring channels is in it, the others are off by 2^-21 of that one at most.)
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
constexpr float kInputLift = 256.f, kFilterLift = 16.f, kFilterFloor = 0x1p-7f;
constexpr unsigned kWindow = 26u << 23;   // binades from the limit of the inputs down to 2^-11 scaled, in bits of a float
// An input below the window is off by 2^-33, its upper term times 2^-4 by 2^-21 against a lower one of 2^-11 of its filter, and the product of
// lower terms that is left out is 2^-34 of its filter: 2^-31 together, against filters below 2^15.  Eight of them, times 2^22:
constexpr float kLeastOfOctet = 512.f;

// A factor as the bits of the power of two that the values stay below: 2^n means a factor of 2^(15 - n).  Values too far from 1
// (from 2^89 on, and infinities) share the last limit, and their results are computed again; 1 (the smallest subnormal): none chosen.
constexpr unsigned kNoLimit = 1, kLeastLimit = 39u << 23, kMostLimit = 220u << 23;
__device__ __forceinline__ float limit_scale(unsigned limit) { return __uint_as_float((269u << 23) - limit); }
__device__ __forceinline__ float limit_unscale(unsigned limit) { return __uint_as_float(max(limit, kLeastLimit) - (15u << 23)); }
// limit of values of which `peak` > 0 is the largest
__device__ __forceinline__ unsigned limit_for(float peak) { return min(max(__float_as_uint(peak) & 0x7f800000u, kLeastLimit - (3u << 23)) + (3u << 23), kMostLimit); }

// Largest magnitude of eight values; NaN does not count.  (The empty assembly keeps the maximum where the values are: put off to the end
// of the loop that stages them, it keeps all of them in registers.)
__device__ __forceinline__ float octet_peak(const float (&x)[8]) {
    float peak = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i += 2) peak = fmaxf(fmaxf(fabsf(x[i]), fabsf(x[i + 1])), peak);
    asm("" : "+v"(peak));
    return peak;
}
// of two magnitudes that are numbers (they compare as integers; a maximum of floats is preceded by one of each for signalling NaN)
__device__ __forceinline__ float larger(float a, float b) { return __uint_as_float(max(__float_as_uint(a), __float_as_uint(b))); }
// over the lanes of a wavefront that hold the octets of a pixel in the operand layout (lanes equal modulo MT)
template <int MT>
__device__ __forceinline__ float pixel_peak(float peak) {
    uintx2 s = __builtin_bit_cast(uintx2, __builtin_amdgcn_permlane32_swap(__float_as_uint(peak), __float_as_uint(peak), false, false));
    peak = larger(__uint_as_float(s.x), __uint_as_float(s.y));
    if constexpr (MT == 16) {
        s = __builtin_bit_cast(uintx2, __builtin_amdgcn_permlane16_swap(__float_as_uint(peak), __float_as_uint(peak), false, false));
        peak = larger(__uint_as_float(s.x), __uint_as_float(s.y));
    }
    return peak;
}
// what a pixel's sums so far are multiplied by when its limit grows
__device__ __forceinline__ float limit_ratio(unsigned from, unsigned to) {
    const unsigned d = (to >> 23) - (from >> 23);
    return d < 127u ? __uint_as_float((127u - d) << 23) : 0.f;
}
// so far that what they held may be lost, or to the last one
__device__ __forceinline__ bool limit_loses(unsigned from, unsigned to) { return to >= kMostLimit || (from != kNoLimit && to - from > (60u << 23)); }
// What a thread has seen of the inputs: their largest, and how many octets its wavefront staged that have any but zeros and all of those below
// the window
struct InputWatch {
    float peak = 0.f;
    unsigned below = 0;
    __device__ __forceinline__ void octet(float most, unsigned limit) {
        peak = larger(peak, most);
        below += (unsigned)__popcll(__ballot(__float_as_uint(most) - 1u < limit - (kWindow + 1u)));
    }
};

// over a wavefront
__device__ __forceinline__ float wave_peak(float peak) {
    auto with = [&](auto control) {
        return fmaxf(peak, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(peak), decltype(control)::value, 0xf, 0xf, true)));
    };
    peak = with(std::integral_constant<int, 0xb1>{});    // lanes 1 0 3 2 of every four
    peak = with(std::integral_constant<int, 0x4e>{});    // 2 3 0 1
    peak = with(std::integral_constant<int, 0x141>{});   // 7 ... 0 of every eight
    peak = with(std::integral_constant<int, 0x140>{});   // 15 ... 0 of every sixteen
    peak = pixel_peak<16>(peak);
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(peak)));
}

// What the wavefronts of a block have seen, or-ed; words: one per wavefront that nothing else uses until the next barrier
template <int WAVES>
__device__ __forceinline__ unsigned block_or(unsigned mine, unsigned *words) {
    if ((threadIdx.x & 63) == 0) words[threadIdx.x >> 6] = mine;
    __syncthreads();
    unsigned all = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) all |= words[w];
    return __builtin_amdgcn_readfirstlane(all);
}
template <int WAVES>
__device__ __forceinline__ unsigned block_sum(unsigned mine, unsigned *words) {   // of the wavefronts
    __syncthreads();
    if ((threadIdx.x & 63) == 0) words[threadIdx.x >> 6] = mine;
    __syncthreads();
    unsigned all = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) all += words[w];
    return __builtin_amdgcn_readfirstlane(all);
}
template <int WAVES>
__device__ __forceinline__ float block_peak(float peak, unsigned *words) {
    peak = wave_peak(peak);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) words[threadIdx.x >> 6] = __float_as_uint(peak);
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; w++) peak = fmaxf(peak, __uint_as_float(words[w]));
    __syncthreads();
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(peak)));
}
// A tile's limit by the largest of its first values in every thread, with room for two to four binades.  Magnitudes that are common find
// theirs by a step of comparisons and a barrier.
template <int WAVES>
__device__ __forceinline__ unsigned first_limit(float most, unsigned *words) {
    unsigned state = 0;
#pragma unroll
    for (int i = 0; i < 5; i++) state |= __ballot(most >= (i == 0 ? 32.f : i == 1 ? 8.f : i == 2 ? 2.f : i == 3 ? 0.5f : 0.125f)) != 0 ? 16u >> i : 0u;
    state = block_or<WAVES>(state, words);
    if (__builtin_expect(state != 0 && state < 16u, 1)) return (state >= 8u ? 134u : state >= 4u ? 132u : state >= 2u ? 130u : 128u) << 23;   // 2^7, 2^5, 2^3, 2
    const float peak = block_peak<WAVES>(most, words);
    return peak > 0.f ? limit_for(peak) : 132u << 23;
}

// the two terms of eight values times `scale` (the lower one times 2^8), each as four words of two halves (lower k in the lower
// half): four multiplications, two conversions of pairs and two mixed-precision multiply-adds for two values, four cycles each.  (As
// v_fma_mixlo_f16 / v_fma_mixhi_f16, seven instructions, it takes 48 instead of 32: these two are issued at half the rate.  Four 1 x 1 convolutions
// of 768 channels on 17 x 17 at batch 64, 704 outputs: 100 -> 94 us; 2048 on 8 x 8, batch 7: 33.7 -> 31.8.)  No assembly: the compiler does not know
// what wait the matrix instructions need behind that.
__device__ __forceinline__ void split_pair(float x0, float x1, float scale, unsigned &hi, unsigned &lo) {
    const float lifted = scale * kInputLift;
    const floatx2 scaled = {x0 * scale, x1 * scale};
    const halfx2 h = __builtin_convertvector(scaled, halfx2);
    const floatx2 rest = {__builtin_fmaf((float)h[0], -kInputLift, x0 * lifted), __builtin_fmaf((float)h[1], -kInputLift, x1 * lifted)};   // (exact)
    hi = __builtin_bit_cast(unsigned, h);
    lo = __builtin_bit_cast(unsigned, __builtin_convertvector(rest, halfx2));
}
__device__ __forceinline__ void split_half2(const float (&x)[8], float scale, uintx4 &hi, uintx4 &lo) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        unsigned h, l;
        split_pair(x[2 * i], x[2 * i + 1], scale, h, l);
        hi[i] = h;
        lo[i] = l;
    }
}

// upper terms, for their partners
__device__ __forceinline__ uintx4 half_down(uintx4 v, float lift) { return __builtin_bit_cast(uintx4, __builtin_bit_cast(halfx8, v) * (_Float16)(1.f / lift)); }

// What follows the packed planes: per output channel the factor that undoes its scaling, and 2^22 times what its filters below the window are
// off by, 0 where it has none: what a sum must be, over the largest input, for that not to show (see above).  Both arrays are read in quads and end in three words of padding.
__device__ __forceinline__ const float *channel_scales(const ConvKernelArgs &a) {
    return reinterpret_cast<const float *>(reinterpret_cast<const char *>(a.wp) + a.w_bytes);
}
__device__ __forceinline__ floatx4 channel_scale_quad(const ConvKernelArgs &a, int g, int m) {
    return *reinterpret_cast<const floatx4_u *>(channel_scales(a) + g * a.OCg + min(m, a.OCg - 1));
}
__device__ __forceinline__ floatx4 channel_least_quad(const ConvKernelArgs &a, int g, int m) {
    return *reinterpret_cast<const floatx4_u *>(channel_scales(a) + a.groups * a.OCg + 3 + g * a.OCg + min(m, a.OCg - 1));
}

// sums of scaled filters -> sums of the filters as they were given (exact); m_base: row 0 of the tiles
template <int MT, int TM, int TN, typename Acc>
__device__ __forceinline__ void scale_channels(const ConvKernelArgs &a, Acc (&acc)[TM][TN], int g, int m_base) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int q = 0; q < Mfma<MT>::ACC / 4; q++) {
            const floatx4 factor = channel_scale_quad(a, g, m_base + i * MT + Mfma<MT>::row(4 * q, lane));
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[i][j][4 * q + v] *= factor[v];
        }
}

// the scale of the inputs is undone
template <int TM, int TN, typename Acc>
__device__ __forceinline__ void unscale_inputs(Acc (&acc)[TM][TN], const unsigned (&limit)[TN]) {
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const float unscale = limit_unscale(limit[j]);
#pragma unroll
        for (int i = 0; i < TM; i++) acc[i][j] *= unscale;
    }
}

// What a wavefront knows of its inputs: the limit of those of this lane's pixels, whether it did not serve them, and how many octets may
// have been below the window.
template <int TN>
struct InputRange {
    unsigned limit[TN];
    bool wild[TN];
    unsigned octets;
};
// The sums of a wavefront again that small operands may show in, in fp32 from the filters as they were given.  `tiles`: its unscaled sums in
// LDS, quad q of lane l of tile e = i * TN + j at [(e * Q + q) * 64 + l]; m_base: row 0 of the tiles; n_of(j): this lane's pixel in tile column j, or negative; K as [k_begin, k_end) of the packed rows, restricted to channels [c_begin, c_end).  Returns false where there were any: all sums
// of the wavefront have then become those of the filters as they were given.  Few of a tile are computed one by one, a lane every 64th
// of the products, more of them by matrix instructions.  Rare, so the code is short.
template <int MT, int TM, int TN, typename Pixel>
__device__ __forceinline__ bool sums_hold(const ConvKernelArgs &a, floatx4 *tiles, const InputRange<TN> &in, int g, int m_base, Pixel n_of,
                                          int k_begin, int k_end, int c_begin, int c_end) {
    using M = Mfma<MT>;
    constexpr int Q = M::ACC / 4, U = 8, kFew = 24;
    const int lane = threadIdx.x & 63, lk = lane / MT, lc = lane % MT;
    auto off_in = [&](int e) {   // a bit per sum of this lane in tile e
        const int i = e / TN, j = e - i * TN;
        unsigned limit = in.limit[0], bits = 0;
        bool wild = in.wild[0];
#pragma unroll
        for (int c = 1; c < TN; c++) {
            limit = j == c ? in.limit[c] : limit;
            wild = j == c ? in.wild[c] : wild;
        }
        const bool counts = limit != kNoLimit && n_of(j) >= 0;
        const float of_inputs = kLeastOfOctet * (float)in.octets * limit_unscale(limit);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int m = m_base + i * MT + M::row(4 * q, lane);
            const floatx4 least = channel_least_quad(a, g, m), sum = tiles[(e * Q + q) * 64 + lane];
#pragma unroll
            for (int v = 0; v < 4; v++)   // (NaN comes from NaN inputs, unless the factors did not serve)
                bits |= counts && m + v < a.OCg && (fabsf(sum[v]) < least[v] * __uint_as_float(limit) + of_inputs || wild || least[v] == __builtin_inff()) ? 1u << (4 * q + v) : 0u;
        }
        return bits;
    };
    unsigned any = 0;
#pragma unroll 1
    for (int e = 0; e < TM * TN; e++) any |= off_in(e);
    if (__ballot(any != 0) == 0) return true;
    const __amdgpu_buffer_rsrc_t xr = buffer_of(a.x, a.x_bytes);
    const float floor = relu_floor(a.pre_relu != 0);
    const int taps = a.Kq / a.ICgP;
    const unsigned fan = (unsigned)(a.ICg * taps);
    const __amdgpu_buffer_rsrc_t wr = buffer_of(a.w, (unsigned)(a.groups * a.OCg) * fan * 4u);
    // channels [first, last) of a tap are within the K range
    auto first_of = [&](int tap) { return max(c_begin, k_begin - tap * a.ICgP); };
    auto last_of = [&](int tap) { return min(min(c_end, a.ICg), k_end - tap * a.ICgP); };
    const int c_span = min(c_end, a.ICg) - c_begin;
#pragma unroll 1
    for (int e = 0; e < TM * TN; e++) {
        const int i = e / TN, j = e - i * TN;
        unsigned bits = off_in(e);   // (the next lines change the sums)
#pragma unroll
        for (int q = 0; q < Q; q++) {
            tiles[(e * Q + q) * 64 + lane] *= channel_scale_quad(a, g, m_base + i * MT + M::row(4 * q, lane));
        }
        const int n_mine = n_of(j);
        // place of output pixel n's tap in the input, in bytes, or beyond the extent
        auto input_at = [&](int n, int tap) {
            const int nn = n >= 0 ? n : 0;
            const int b = (int)fast_div((unsigned)nn, a.div_ohw);
            const int r = nn - b * a.OHW;
            const int oh = (int)fast_div((unsigned)r, a.div_ow), ow = r - oh * a.OW;
            const int kh = tap / a.KW, kw = tap - kh * a.KW;
            const int ih = oh * a.sh - a.ph + kh, iw = ow * a.sw - a.pw + kw;
            const bool ok = n >= 0 && (unsigned)ih < (unsigned)a.H && (unsigned)iw < (unsigned)a.W;
            return ok ? (((unsigned)(b * a.H + ih) * (unsigned)a.W + (unsigned)iw) * (unsigned)a.x_ps + (unsigned)(g * a.ICg)) * 4u : kOutOfRange;
        };
        // (a sum of zeros is as it should be)
        unsigned zeros = 0;
#pragma unroll
        for (int q = 0; q < Q; q++)
#pragma unroll
            for (int v = 0; v < 4; v++) zeros |= tiles[(e * Q + q) * 64 + lane][v] == 0.f ? bits & 1u << (4 * q + v) : 0u;
        if (__ballot(zeros != 0) != 0) {
            bool any_input = false;
#pragma unroll 1
            for (int tap = 0; tap < taps; tap++) {
                const unsigned at = zeros != 0 ? input_at(n_mine, tap) : kOutOfRange;
                const int last = last_of(tap);
#pragma unroll 4
                for (int c = first_of(tap); c < last; c += 4) {
                    const floatx4 x = buffer_load_f32x4(xr, (at + (unsigned)c * 4u) | (at & kOutOfRange));
#pragma unroll
                    for (int u = 0; u < 4; u++) any_input = any_input || (c + u < last && relu_above(floor, x[u]) != 0.f);
                }
            }
            if (!any_input) bits &= ~zeros;
        }
        int total = __popc(bits);
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) total += __shfl_xor(total, d);
        if (__builtin_amdgcn_readfirstlane(total) <= kFew) {
            while (true) {
                const unsigned long long lanes = __ballot(bits != 0);
                if (lanes == 0) break;
                const int owner = __builtin_ctzll(lanes);
                const int v = __builtin_ctz((unsigned)__builtin_amdgcn_readlane((int)bits, owner)), n = __builtin_amdgcn_readlane(n_mine, owner);
                const int m = m_base + i * MT + M::row(v, owner);
                float sum = 0.f;
                // (all of K, a value of another tap in every lane where the channels are few: the loads of eight rounds are under way together)
                int tap = c_span > 0 ? lane / c_span : taps, c = lane - tap * c_span;
#pragma unroll 1
                while (__ballot(tap < taps) != 0) {
                    float x[8], w[8];
#pragma unroll
                    for (int u = 0; u < 8; u++) {
                        const int channel = c_begin + c, k = tap * a.ICgP + channel;
                        const bool ok = tap < taps && k >= k_begin && k < k_end;
                        const unsigned at = input_at(ok ? n : -1, tap);
                        x[u] = buffer_load_f32(xr, (at + (unsigned)channel * 4u) | (at & kOutOfRange));
                        w[u] = buffer_load_f32(wr, ok ? ((unsigned)(g * a.OCg + m) * fan + (unsigned)(channel * taps + tap)) * 4u : kOutOfRange);
                        c += 64;
                        while (c >= c_span && tap < taps) {
                            c -= c_span;
                            tap++;
                        }
                    }
#pragma unroll
                    for (int u = 0; u < 8; u++) sum = __builtin_fmaf(w[u], relu_above(floor, x[u]), sum);
                }
#pragma unroll
                for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d);
                if (lane == owner) {
                    tiles[(e * Q + (v >> 2)) * 64 + lane][v & 3] = sum;
                    bits &= bits - 1u;
                }
            }
            continue;
        }
        const int m = m_base + i * MT + lc;
        const unsigned w_row = m < a.OCg ? (unsigned)(g * a.OCg + m) * fan * 4u : kOutOfRange;
        typename M::acc_t sum;
#pragma unroll
        for (int v = 0; v < M::ACC; v++) sum[v] = 0.f;
#pragma unroll 1
        for (int tap = 0; tap < taps; tap++) {
            const unsigned at = input_at(n_mine, tap);
            const int last = last_of(tap);
#pragma unroll 1
            for (int c0 = first_of(tap); c0 < last; c0 += U * M::KSTEP) {
                float w[U], x[U];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int c = c0 + u * M::KSTEP + lk;
                    const unsigned kill = c < last ? 0u : kOutOfRange;
                    w[u] = buffer_load_f32(wr, (w_row + (unsigned)(c * taps + tap) * 4u) | (w_row & kOutOfRange) | kill);
                    x[u] = buffer_load_f32(xr, (at + (unsigned)c * 4u) | (at & kOutOfRange) | kill);
                }
#pragma unroll
                for (int u = 0; u < U; u++) sum = M::run(w[u], relu_above(floor, x[u]), sum);
            }
        }
#pragma unroll
        for (int v = 0; v < M::ACC; v++)
            if (bits >> v & 1u) tiles[(e * Q + (v >> 2)) * 64 + lane][v & 3] = sum[v];
    }
    return false;
}

// Whether sums_hold need look at a wavefront's unscaled sums, in registers; in and n_of as there.  least: channel_least of the rows of the tiles, a
// quad 4 * (lane % (MT / 4)) rows into each.  Few rows have one, if any: only theirs are looked at.
template <int MT, int TM, int TN, typename Pixel>
__device__ __forceinline__ bool sums_look_off(const ConvKernelArgs &a, const typename Mfma<MT>::acc_t (&acc)[TM][TN], const InputRange<TN> &in, const floatx4 (&least)[TM], int m_base,
                                              Pixel n_of) {
    using M = Mfma<MT>;
    float most = 0.f;   // (what lies behind the last channel may be anything)
    unsigned quads[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = m_base + i * MT + 4 * ((threadIdx.x & 63) % (MT / 4));
        float mine = 0.f;
#pragma unroll
        for (int k = 0; k < 4; k++) mine = fmaxf(mine, m + k < a.OCg ? least[i][k] : 0.f);
        most = fmaxf(most, mine);
        quads[i] = (unsigned)__ballot(mine > 0.f) & ((1u << (MT / 4)) - 1u);   // a bit per quad of rows
    }
    bool off = in.octets != 0;
#pragma unroll
    for (int j = 0; j < TN; j++) off = off || in.wild[j];
    if (__builtin_expect(__ballot(off || most > 0.f) == 0, 1)) return false;
    most = wave_peak(most);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int q = 0; q < M::ACC / 4; q++) {
            unsigned mine = 0;   // the quads of rows that the lanes hold in these four registers
#pragma unroll
            for (int l = 0; l < 64; l += MT) mine |= 1u << (M::row(4 * q, l) / 4);
            if ((quads[i] & mine) == 0) continue;
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int v = 4 * q; v < 4 * q + 4; v++)
                    off = off || (n_of(j) >= 0 && in.limit[j] != kNoLimit && m_base + i * MT + M::row(v, threadIdx.x & 63) < a.OCg &&
                                  !(fabsf(acc[i][j][v]) >= most * __uint_as_float(in.limit[j])));
        }
    return __ballot(off) != 0;
}

// Both, for sums in registers; `tiles` is free.
template <int MT, int TM, int TN, typename Pixel>
__device__ __forceinline__ bool check_sums(const ConvKernelArgs &a, typename Mfma<MT>::acc_t (&acc)[TM][TN], floatx4 *tiles, const InputRange<TN> &in, const floatx4 (&least)[TM], int g,
                                           int m_base, Pixel n_of, int k_begin, int k_end, int c_begin, int c_end) {
    constexpr int Q = Mfma<MT>::ACC / 4;
    const int lane = threadIdx.x & 63;
    if (__builtin_expect(!sums_look_off<MT>(a, acc, in, least, m_base, n_of), 1)) return true;
#pragma unroll
    for (int e = 0; e < TM * TN; e++)
#pragma unroll
        for (int q = 0; q < Q; q++)
            tiles[(e * Q + q) * 64 + lane] = floatx4{acc[e / TN][e % TN][4 * q], acc[e / TN][e % TN][4 * q + 1], acc[e / TN][e % TN][4 * q + 2], acc[e / TN][e % TN][4 * q + 3]};
    if (sums_hold<MT, TM, TN>(a, tiles, in, g, m_base, n_of, k_begin, k_end, c_begin, c_end)) return true;
#pragma unroll
    for (int e = 0; e < TM * TN; e++)
#pragma unroll
        for (int q = 0; q < Q; q++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[e / TN][e % TN][4 * q + v] = tiles[(e * Q + q) * 64 + lane][v];
    return false;
}

// eight fp32 values rounded to bfloat16 (nearest even), as four words of two (lower k in the lower half)
typedef float floatx8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ uintx4 round_bf16x8(const float (&x)[8]) {
    const floatx8 v = {x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]};
    return __builtin_bit_cast(uintx4, __builtin_convertvector(v, bf16x8));
}

// TM x TN tiles of 32 x 32 and one unit of 16 k, or of 16 x 16 and 32 k: filter operands av, input operands bv, a plane per term.  Two terms take three
// instructions; the tiles of a product are independent instructions.
__device__ __forceinline__ floatx16 multiply_half(uintx4 a, uintx4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
}
__device__ __forceinline__ floatx4 multiply_half(uintx4 a, uintx4 b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
}
template <bool HALF, int TM, int TN, typename Acc>
__device__ __forceinline__ void multiply_planes(Acc (&acc)[TM][TN], const uintx4 (&av)[TM], const uintx4 (&bv)[TN]) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if constexpr (HALF)
                acc[i][j] = multiply_half(av[i], bv[j], acc[i][j]);
            else
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av[i]), __builtin_bit_cast(bf16x8, bv[j]), acc[i][j], 0, 0, 0);
        }
}
template <int TERMS, bool HALF, int TM, int TN, typename Acc>
__device__ __forceinline__ void multiply_terms(Acc (&acc)[TM][TN], const uintx4 (&av)[TERMS][TM], const uintx4 (&bv)[TERMS][TN]) {
    if constexpr (TERMS == 2) {   // smallest products first
        uintx4 ad[TM], bd[TN];
#pragma unroll
        for (int j = 0; j < TN; j++) bd[j] = half_down(bv[0][j], kFilterLift);
        multiply_planes<HALF>(acc, av[1], bd);
#pragma unroll
        for (int i = 0; i < TM; i++) ad[i] = half_down(av[0][i], kInputLift);
        multiply_planes<HALF>(acc, ad, bv[1]);
    }
    multiply_planes<HALF>(acc, av[0], bv[0]);
}

// The same for two terms in a fixed order, between(n) behind the n-th of 3 TM TN matrix instructions: what it does is issued while they run (an
// instruction waits for the one before it in the matrix pipe, and all that follows in the wavefront with it).
template <int TM, int TN, typename Acc, typename Between>
__device__ __forceinline__ void multiply_terms_between(Acc (&acc)[TM][TN], const uintx4 (&av)[2][TM], const uintx4 (&bv)[2][TN], Between between) {
    uintx4 ad[TM], bd[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) bd[j] = half_down(bv[0][j], kFilterLift);
    __builtin_amdgcn_sched_barrier(0);
    int n = 0;
#pragma unroll
    for (int t = 0; t < 3; t++)
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                acc[i][j] = multiply_half(t == 0 ? av[1][i] : t == 1 ? ad[i] : av[0][i], t == 0 ? bd[j] : t == 1 ? bv[1][j] : bv[0][j], acc[i][j]);
                if (t == 0 && j == 0) {
                    ad[i] = half_down(av[0][i], kInputLift);
                    asm volatile("" : "+v"(ad[i]));
                }
                between(n++);
                __builtin_amdgcn_sched_barrier(0);
            }
}

// TMW x TNW MFMA tiles of 32 x 32 per wavefront, WM x WN wavefronts per block
// TERMS = 3: fp32 accuracy as described above.  TERMS = 1: the reduced-precision mode with bfloat16 operands (inputs and
// filters rounded to nearest even, fp32 accumulation): one plane, one matrix instruction per tile and K tile, a sixth of the
// matrix work and a third of the LDS traffic.
template <int TMW, int TNW, int WM, int WN, int PD, int TERMS = 3>
struct ConvSplit3 {
    static_assert(TERMS == 3 || TERMS == 1, "three exact terms or one rounded term");
    static constexpr int MT = 32, BK = 16;
    using M = Mfma<32>;
    static constexpr int BM = 32 * TMW * WM, BN = 32 * TNW * WN;
    static constexpr int WAVES = WM * WN;
    static constexpr int T = 64 * WAVES;
    static constexpr int THREADS = T;
    static constexpr int CPAD = BK;
    static constexpr bool FUSABLE = false;
    // LDS in slots of 16 bytes (eight bfloat16): per stage the input planes [TERMS][2][BN]
    static constexpr int STAGE = 2 * TERMS * BN;
    static constexpr int SMEM_FLOATS = std::max(2 * STAGE * 4, WAVES * tail_floats(TMW, TNW));
    static constexpr int B_OCT = 2 * BN;
    static constexpr int B_IT = (B_OCT + T - 1) / T;                   // octets a thread stages per K tile
    static_assert(B_OCT % T == 0 || B_IT == 1, "whole passes, or one with surplus threads");

    template <bool RES = false>
    __device__ static __forceinline__ void run(const ConvKernelArgs &a, float *smem, int tile, int g, int z) {
    constexpr int WTM = 32 * TMW, WTN = 32 * TNW;
    constexpr int TM = TMW, TN = TNW;
    uintx4 *lds = reinterpret_cast<uintx4 *>(smem);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN;
    const int wm = wave / WN;
    const int lk = lane >> 5;   // which eight k of a K tile this lane supplies to the matrix instruction
    const int lc = lane & 31;   // row (A) / column (B) of this lane inside an MFMA tile
    int tm, tn;
    xcd_tile(a, tile, tm, tn);
    const int m0 = tm * BM;
    const int n0 = tn * BN;
    const int k_begin = z * a.k_chunk;
    const int k_end = min(a.Kq, k_begin + a.k_chunk);
    const int nkt = (k_end - k_begin) / BK;

    // ---- filters: every wavefront reads the operands of its own tiles from global memory, in operand layout -------------
    const __amdgpu_buffer_rsrc_t xr = buffer_of(a.x, a.x_bytes);
    const __amdgpu_buffer_rsrc_t wr = buffer_of(a.wp, a.w_bytes);
    unsigned a_off[TM];      // byte offset of this lane's slot (plane 0) inside a K tile of the packed filters, or out of range
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = m0 + wm * WTM + i * MT + lc;
        // packed filters: [g][k / 8][plane][OCgP] slots of 16 bytes
        a_off[i] = m < a.OCgP ? (unsigned)(((((size_t)g * (a.Kq >> 3) + lk) * TERMS) * a.OCgP + m) * 16) : kOutOfRange;
    }
    const unsigned a_plane = (unsigned)a.OCgP * 16u;
    // ---- inputs: this thread's pixels and its octet of channels ----------------------------------------------------------
    // Two neighbouring threads take the two octets of a pixel: 64 contiguous bytes of the input.
    const int oct = tid & 1;
    int ih0[B_IT], iw0[B_IT];
    unsigned x_off[B_IT], n_kill[B_IT];
#pragma unroll
    for (int i = 0; i < B_IT; i++) {
        const int n = n0 + ((tid + i * T) >> 1);
        // (more threads than octets: the surplus stages nothing)
        const bool ok = n < a.Npix && (B_OCT % T == 0 || tid < B_OCT);
        n_kill[i] = ok ? 0u : kOutOfRange;
        const int nn = ok ? n : 0;
        const int b = (int)fast_div((unsigned)nn, a.div_ohw);
        const int r = nn - b * a.OHW;
        const int oh = (int)fast_div((unsigned)r, a.div_ow);
        const int ow = r - oh * a.OW;
        ih0[i] = oh * a.sh - a.ph;
        iw0[i] = ow * a.sw - a.pw;
        x_off[i] = (((unsigned)(b * a.H + ih0[i]) * (unsigned)a.W + (unsigned)iw0[i]) * (unsigned)a.x_ps + (unsigned)(g * a.ICg + 8 * oct)) * 4u;
    }
    // LDS slot of (pixel, octet) inside a plane: the two octets of a pixel side by side, exchanged in every other group of four
    // pixels, so that eight consecutive pixels of one octet (an operand read) and four pixels of both (a store) use all banks
    auto slot_of = [](int pixel, int octet) { return 2 * pixel + (octet ^ ((pixel >> 2) & 1)); };

    uintx4 a_reg[PD][TERMS][TM];
    floatx4 b_reg[PD][B_IT][2];
    int b_left[PD];   // real channels of this thread's octet in the stage's K tile
    auto load_tile = [&](int kt, uintx4 (&ar)[TERMS][TM], floatx4 (&br)[B_IT][2], int &left) {
        const int k0 = k_begin + kt * BK;
        const int tap = (int)__umulhi((unsigned)k0, a.magic_icgp);
        const int c0 = k0 - tap * a.ICgP;
        const int kh = a.KW == 1 ? tap : (int)__umulhi((unsigned)tap, a.magic_kw);
        const int kw = tap - kh * a.KW;
        const unsigned tile_kill = kt < nkt ? 0u : kOutOfRange;   // tiles past the end of the K range load zeros
        const unsigned w_tile = (unsigned)((k0 >> 3) * TERMS * a.OCgP) * 16u;
#pragma unroll
        for (int p = 0; p < TERMS; p++)
#pragma unroll
            for (int i = 0; i < TM; i++) ar[p][i] = __builtin_amdgcn_raw_buffer_load_b128(wr, (a_off[i] + w_tile) | tile_kill, (unsigned)p * a_plane, 0);
        const unsigned x_tile = (unsigned)((kh * a.W + kw) * a.x_ps + c0) * 4u;
        const int c_left = a.ICg - c0 - 8 * oct;   // real channels from this octet on
        const unsigned pad0 = (unsigned)(c_left - 1) & kOutOfRange, pad1 = (unsigned)(c_left - 5) & kOutOfRange;   // sign bits
#pragma unroll
        for (int i = 0; i < B_IT; i++) {
            const unsigned in_h = (unsigned)(ih0[i] + kh) < (unsigned)a.H ? 1u : 0u;
            const unsigned in_w = (unsigned)(iw0[i] + kw) < (unsigned)a.W ? 1u : 0u;
            const unsigned at = (x_off[i] + x_tile) | (((in_h & in_w) ^ 1u) << 31) | n_kill[i] | tile_kill;
            // (no branch around loads inside the loop: where paths that issued loads join, the compiler waits for all of them)
            br[i][0] = buffer_load_f32x4(xr, at | pad0);
            br[i][1] = buffer_load_f32x4(xr, at | pad1, 16u);
        }
        left = c_left;
    };
    const float floor = relu_floor(a.pre_relu != 0);
    const bool ragged = (a.ICg & 3) != 0;   // a quad of channels may straddle the end of the group's
    auto store_inputs = [&](int buf, const floatx4 (&br)[B_IT][2], int left) {
        uintx4 *stage = lds + buf * STAGE;
#pragma unroll
        for (int i = 0; i < B_IT; i++) {
            if (B_OCT % T != 0 && tid + i * T >= B_OCT) continue;
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = relu_above(floor, br[i][j >> 2][j & 3]);   // folded ReLU of the producer
            if (ragged)
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = j < left ? v[j] : 0.f;
            const int slot = slot_of((tid + i * T) >> 1, oct);
            if constexpr (TERMS == 3) {
                uintx4 hi, mid, lo;
                split_bf16x3(v, hi, mid, lo);
                stage[slot] = hi;
                stage[2 * BN + slot] = mid;
                stage[4 * BN + slot] = lo;
            } else {
                stage[slot] = round_bf16x8(v);
            }
        }
    };

    typename M::acc_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < M::ACC; v++) acc[i][j][v] = 0.f;

    // ---- main loop ---------------------------------------------------------------------------------------------------------
    // Register stage s holds K tile kt with kt % PD == s (filter operands of this wavefront, inputs of this thread).  Iteration
    // kt: the matrix work of tile kt from registers (filters) and LDS stage kt & 1 (inputs), the stage's registers requested
    // again for tile kt + PD, the inputs of tile kt + 1 split and stored into the other LDS stage, one barrier.
#pragma unroll
    for (int s = 0; s < PD; s++) load_tile(s, a_reg[s], b_reg[s], b_left[s]);
    store_inputs(0, b_reg[0], b_left[0]);
    __syncthreads();
    for (int kt0 = 0; kt0 < nkt; kt0 += PD) {
#pragma unroll
        for (int s = 0; s < PD; s++) {
            const int kt = kt0 + s;
            const int buf = kt & 1;
            const uintx4 *Bb = lds + buf * STAGE + slot_of(wn * WTN + lc, lk);   // (tiles are 32 pixels apart: the same exchange in all)
            bf16x8 av[TERMS][TM], bv[TERMS][TN];
#pragma unroll
            for (int p = 0; p < TERMS; p++) {
#pragma unroll
                for (int i = 0; i < TM; i++) av[p][i] = __builtin_bit_cast(bf16x8, a_reg[s][p][i]);
#pragma unroll
                for (int j = 0; j < TN; j++) bv[p][j] = __builtin_bit_cast(bf16x8, Bb[p * 2 * BN + j * 2 * MT]);
            }
            // all LDS reads of the tile are requested before its first matrix instruction (left to itself the scheduler
            // requests each operand right in front of its first use and the wavefront pays the LDS latency once per plane)
            __builtin_amdgcn_sched_barrier(0);
            // the six terms, smallest first; the tiles of a term are independent instructions
            constexpr int NT = TERMS == 3 ? 6 : 1;
            constexpr int TA[6] = {TERMS == 3 ? 2 : 0, 0, 1, 1, 0, 0}, TB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[TA[t]][i], bv[TB[t]][j], acc[i][j], 0, 0, 0);
            store_inputs(buf ^ 1, b_reg[(s + 1) % PD], b_left[(s + 1) % PD]);
            load_tile(kt + PD, a_reg[s], b_reg[s], b_left[s]);
            __syncthreads();
        }
    }
    TailConstants<TM> constants;
    tail_constants<MT, false>(a, constants, g, m0 + wm * WTM);
    tiled_tail<MT, BM, BN, TM, TN, WM, WN, RES>(a, smem, acc, tile, g, z, m0, n0, wm, wn, 0, constants);
    }   // run
};

// y[n][oc] = act(bias[oc] + sum_s ws[s][n][oc]) (+ residual); slices are added in index order
struct ReduceArgs {
    const float *ws;
    const float *bias;
    float *y;
    int slices, OC, Npix, y_ps, act;
    long long slice_floats;
    const float *res;      // residual operand as in ConvKernelArgs, or null
    int res_ps, post_relu;
};

__device__ __forceinline__ void splitk_reduce_body(const ReduceArgs &a, int block, int num_blocks, unsigned threads) {
    const long long total = (long long)a.OC * a.Npix;
    for (long long i = block * (long long)threads + threadIdx.x; i < total; i += (long long)num_blocks * threads) {
        const int n = (int)(i / a.OC);
        const int oc = (int)(i - (long long)n * a.OC);
        float sum = 0.f;
        for (int s = 0; s < a.slices; s++) sum += a.ws[s * a.slice_floats + i];
        float out[1] = {sum + a.bias[oc]};
        apply_activation(out, a.act);
        float v = out[0];
        if (a.res != nullptr) {
            v += a.res[(long long)n * a.res_ps + oc];
            if (a.post_relu) v = fmaxf(v, 0.0f);
        }
        a.y[(long long)n * a.y_ps + oc] = v;
    }
}


// ---- wave-split variant: no LDS staging, K divided among the wavefronts of a block ---------------------------------------
// For batch-1 layers (tens to hundreds of pixels, K in the thousands) the LDS-tiled kernel is bound by the chain
// load -> LDS -> barrier per K tile, and slicing K over blocks costs a second kernel.  Here every wavefront of a
// block owns a contiguous K range of the same BM x BN output tile and feeds the MFMA straight from global memory in
// the instruction's operand layout (lane l: A[k = l / MT][m = l % MT], B[k = l / MT][n = l % MT]); there is no barrier
// inside the K loop, two register batches of U k-steps keep dozens of loads in flight per lane, and the NW partial
// tiles meet once in LDS, where the wavefronts share the bias + activation + store work.  The sum order is fixed
// (k ascending inside a wavefront, wavefronts ascending), so results are reproducible.
//
// QUAD: within a batch of U k-steps (U * KSTEP consecutive k) the lane group lk supplies k = U * lk + u in step u
// instead of KSTEP * u + lk.  The MFMA only needs A and B to agree on k, and this assignment gives a lane U
// consecutive filter rows, which the quad-packed filter layout [k / 4][m][4] delivers as 16-byte loads: a quarter
// of the filter load instructions.  Channels are padded to the batch (U * KSTEP), so a batch lies inside one tap.
//
// BF16 (reduced-precision mode): filters are packed as bfloat16 in the quad layout (a lane's four k are one 8-byte
// load), inputs are rounded to bfloat16 (nearest even) after loading, and one v_mfma_f32_16x16x16_bf16 consumes
// the four k of a lane group at once - the same k assignment as QUAD; accumulation stays fp32.
//
// CP: channel padding of the packed filters when it should differ from the default (8, or the batch with QUAD); 4 serves
// layers with a handful of input channels (the first layer of an image network), whose K would otherwise be mostly padding.
template <int MT, int TM, int TN, int NW, int U, bool QUAD = false, int D = 2, int RP = 0, int CP = 0>
struct ConvWsplit {
    using M = Mfma<MT>;
    static constexpr int BM = TM * MT, BN = TN * MT;
    static constexpr int E = TM * TN * M::ACC;
    static constexpr int THREADS = 64 * NW;
    static constexpr int SMEM_FLOATS = NW * E * 64 + (RP == 3 ? NW : 0);   // (two terms: a flag per wavefront behind the tiles)
    static constexpr int CPAD = CP ? CP : (QUAD ? U * M::KSTEP : 8);   // channel padding of the packed filters this kernel expects
    static_assert(CP == 0 || (!QUAD && CP % M::KSTEP == 0), "a k-step must lie inside one filter tap");
    static constexpr bool KQUAD = QUAD;                    // packed filters are [k / 4][m][4] instead of [k][m]
    // accumulators + staged operands per lane decide whether the body fits the register budget of a fused launch
    // (the channel-padding-4 forms serve first layers, which are stages of their own: kept out of the fused launches)
    static constexpr bool FUSABLE = RP < 3 && CP == 0 && E + D * U * (TM + TN) <= (QUAD ? (MT == 32 ? 48 : 56) : 48);   // per-step addressing of the plain layout needs more registers, and so do the 16-register accumulator tuples of the 32 x 32 tiles
    // the two-term bodies of up to two 32 x 32 tiles per wavefront run inside fused launches of the
    // wide-register kernel family (fused_kernel_wide)
    static constexpr bool FUSABLE_WIDE = RP == 3 && MT == 32 && NW <= 8 && TM * TN <= 2;
    static constexpr int KREDUCED = RP;                    // 0: fp32 filters; 1: packed filters hold bfloat16; 2: IEEE half; 3: two planes of half; 4: one of bfloat16; 5: one of half
    static constexpr int PLANES = RP == 3 ? 2 : 1;
    static constexpr int WAVES_PER_SIMD = RP != 3 || MT == 16 ? 1 : TM * TN == 1 ? 4 : TM * TN == 2 ? 3 : 2;
    // RP == 4, 5: the reduced-precision modes on the same instruction and layout: one plane of filters rounded to bfloat16 or half, inputs
    // rounded after the load, one matrix instruction per tile and batch.
    // RP == 3: fp32 results from the half matrix pipe (operands as two terms, three products on v_mfma_f32_32x32x16_f16, see
    // split_half2): filters are split when packed, [k / 8][plane][m][8], and read as operands straight from global memory; a lane
    // splits the eight input values it loads for a batch itself.  The scale of a pixel is kept by the lanes that hold its sums.
    static_assert(!QUAD || U % 4 == 0, "quad loads need whole groups of four k per lane");
    static_assert(RP >= 0 && RP <= 5 && (RP == 0 || (RP >= 3 ? QUAD && U == 8 && (MT == 32 || RP == 3) : QUAD && MT == 16 && U == 4)),
                  "the 16-bit paths are the 16 x 16 x 16 form of the quad layout, or the 32 x 32 x 16 and 16 x 16 x 32 forms of the octet layout");

    template <bool RES = false>
    __device__ static __forceinline__ void run(const ConvKernelArgs &a, float *red, int tile, int g, int z) {

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: keeps per-wavefront K ranges and loop control on the SALU
    const int lk = lane / MT;
    const int lc = lane % MT;
    int tm, tn;
    xcd_tile(a, tile, tm, tn);
    const int m0 = tm * BM;
    const int n0 = tn * BN;

    // K slice z of the grid (k_chunk is a multiple of the batch U * KSTEP), divided among the wavefronts; the host did the
    // divisions (every wavefront of a block repeats this prologue on the SIMD's one scalar issue slot, so it is kept short)
    const int s_lo = z * a.steps_chunk;
    const int s_hi = min(a.steps_total, s_lo + a.steps_chunk);
    const int s_begin = s_lo + wave * a.steps_per_wave;
    const int s_end = min(s_hi, s_begin + a.steps_per_wave);

    // the bias of the outputs this lane finishes in the epilogue (and the factors of their channels, with two terms), requested
    // ahead of the K loop so that its latency hides behind it (a wavefront finishes whole quads of consecutive output channels)
    constexpr int G = E / 4;
    constexpr int GPW = (G + NW - 1) / NW;
    auto quad_row = [&](int e4) { return m0 + (4 * e4 / (M::ACC * TN)) * MT + M::row((4 * e4) % M::ACC, lane); };
    floatx4 bias_pre[GPW], factor_pre[RP == 3 ? GPW : 1];
    auto request_bias = [&] {
#pragma unroll
        for (int t = 0; t < GPW; t++) {
            const int row = quad_row(min(wave + t * NW, G - 1));
            bias_pre[t] = bias_quad(a, g, row);
            if constexpr (RP == 3) factor_pre[t] = channel_scale_quad(a, g, row);
        }
    };
    typename M::acc_t acc[TM][TN];
    // two terms: the limits of this lane's pixels, which follow their values
    InputRange<TN> in;
    unsigned below = 0;
#pragma unroll
    for (int j = 0; j < TN; j++) {
        in.limit[j] = kNoLimit;
        in.wild[j] = false;
    }
    int ih0[TN], iw0[TN];
    unsigned x_lane[TN];   // byte offset of (image, ih0, iw0, first channel of the lane); may wrap below zero, the tap offset brings it back
    bool n_ok[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = n0 + j * MT + lc;
        n_ok[j] = n < a.Npix;
        const int nn = n_ok[j] ? n : 0;
        // image sizes are below 2^15 per side and OH * OW below 2^23 (checked on the host): signed 24-bit multiplies, which
        // run at full rate, are exact here; byte offsets are wanted modulo 2^32, so 32-bit arithmetic gives them
        const int b = (int)fast_div((unsigned)nn, a.div_ohw);
        const int r = nn - __mul24(b, a.OHW);
        const int oh = (int)fast_div((unsigned)r, a.div_ow);
        const int ow = r - __mul24(oh, a.OW);
        ih0[j] = __mul24(oh, a.sh) - a.ph;
        iw0[j] = __mul24(ow, a.sw) - a.pw;
        const int lane_channel = QUAD ? U * lk : lk;   // first channel of this lane inside a step / batch
        x_lane[j] = ((unsigned)(__mul24(b, a.H) + ih0[j]) * (unsigned)a.W + (unsigned)iw0[j]) * (unsigned)(a.x_ps * 4) +
                    (unsigned)(g * a.ICg + lane_channel) * 4u;
    }
    const __amdgpu_buffer_rsrc_t xr = buffer_of(a.x, a.x_bytes);
    const __amdgpu_buffer_rsrc_t wr = buffer_of(a.wp, a.w_bytes);
    unsigned w_lane[TM], w_kill[TM], n_kill[TN];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        w_kill[i] = m0 + i * MT + lc < a.OCgP ? 0u : kOutOfRange;
        // byte offsets below 2^31 (checked on the host)
        if (RP >= 3)   // [g][k / 8][plane][m] slots of 16 bytes: this lane's octet of a batch is lk
            w_lane[i] = ((((unsigned)g * ((unsigned)a.Kq >> 3) + (unsigned)lk) * (unsigned)PLANES) * (unsigned)a.OCgP + (unsigned)(m0 + i * MT + lc)) * 16u;
        else if (QUAD)   // [g][k / 4][m][4]: this lane's first quad of a batch is row (U / 4) * lk
            w_lane[i] = (((unsigned)g * ((unsigned)a.Kq >> 2) + (unsigned)((U / 4) * lk)) * (unsigned)a.OCgP + (unsigned)(m0 + i * MT + lc)) * (RP != 0 ? 8u : 16u);
        else
            w_lane[i] = (((unsigned)g * (unsigned)a.Kq + (unsigned)lk) * (unsigned)a.OCgP + (unsigned)(m0 + i * MT + lc)) * 4u;
    }
#pragma unroll
    for (int j = 0; j < TN; j++) n_kill[j] = n_ok[j] ? 0u : kOutOfRange;

    if constexpr (RP != 3 || GPW == 1) request_bias();
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < M::ACC; v++) acc[i][j][v] = 0.f;

    // D register batches in flight: filter operands (fp32: U steps x TM tiles; bf16: four packed k per tile) and inputs
    struct FilterStageF32 {
        float v[U][TM];
    };
    struct FilterStageBf16 {
        uintx2 v[TM];
    };
    struct FilterStageX3 {
        uintx4 v[PLANES][TM];
    };
    using FilterStage = std::conditional_t<(RP >= 3), FilterStageX3, std::conditional_t<(RP != 0), FilterStageBf16, FilterStageF32>>;
    FilterStage av[D];
    float bv[D][U][TN];
    int left[D];

    // k-step s covers rows k = s * KSTEP + lk of the tap-major packed filters; ICgP is a multiple of KSTEP, so a
    // step lies inside one filter tap and (tap, kh, kw, first channel) are wavefront-uniform
    // QUAD: scalar state of the next batch to request (batches are requested in K order starting at s_begin)
    int q_cb = 0, q_kh = 0, q_kw = 0;
    unsigned q_w = 0;
    const int c_lane_last = a.ICg - 1 - U * lk;   // QUAD: the lane's first channel of a batch starting at channel cb is real while cb <= c_lane_last
    if constexpr (QUAD) {
        const int kb = s_begin * M::KSTEP;
        const int tap = (int)__umulhi((unsigned)kb, a.magic_icgp);
        q_cb = kb - tap * a.ICgP;
        q_kh = a.KW == 1 ? tap : (int)__umulhi((unsigned)tap, a.magic_kw);
        q_kw = tap - q_kh * a.KW;
        q_w = RP >= 3 ? (unsigned)((kb / 8) * PLANES * a.OCgP) * 16u : (unsigned)((kb / 4) * a.OCgP) * (RP != 0 ? 8u : 16u);
    }
    // `live` (wavefront-uniform) is false for a batch beyond the wavefront's K range: its loads are still issued, against
    // descriptors of extent zero, and return zeros without touching memory.  Loads are never skipped by a branch inside
    // the K loop: where a path with and a path without newly issued loads join, the compiler can only wait for *all*
    // outstanding loads before the next use of an older one, which serialises load latency and matrix work.
    // `left` (QUAD): the last real channel among those the lane has loaded, counted from its first one; where the group's channel
    // count is no multiple of four, the quad that straddles its end holds a neighbour's channels and is masked before use.
    auto load_batch = [&](int s0, FilterStage &A, float(&B)[U][TN], int &left, bool live) {
        if constexpr (QUAD) {
            // The whole batch lies inside one tap (channels are padded to the batch).  Batches are requested in K
            // order, so (first channel, kh, kw) and the filter offset advance incrementally on the SALU.  Lane-constant
            // offsets go into the vector operand of the buffer loads, the per-batch / per-step parts into the scalar
            // operand: a filter load costs no VALU instruction, an input load one add + one or per batch and tile.
            (void)s0;
            const __amdgpu_buffer_rsrc_t xr = buffer_of(a.x, live ? a.x_bytes : 0u);
            const __amdgpu_buffer_rsrc_t wr = buffer_of(a.wp, live ? a.w_bytes : 0u);
            if constexpr (RP >= 3) {
#pragma unroll
                for (int p = 0; p < PLANES; p++)
#pragma unroll
                    for (int i = 0; i < TM; i++)   // eight bfloat16 = the lane's eight k of this batch, one plane
                        A.v[p][i] = __builtin_amdgcn_raw_buffer_load_b128(wr, w_lane[i] | w_kill[i], q_w + (unsigned)(p * a.OCgP) * 16u, 0);
            } else if constexpr (RP != 0) {
#pragma unroll
                for (int i = 0; i < TM; i++) {   // four 16-bit values = the lane's four k of this batch
                    A.v[i] = buffer_load_u32x2(wr, w_lane[i] | w_kill[i], q_w);
                }
            } else {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int q = 0; q < U / 4; q++) {
                        const floatx4 w4 = buffer_load_f32x4(wr, w_lane[i] | w_kill[i], q_w + (unsigned)(q * a.OCgP) * 16u);
                        A.v[q * 4 + 0][i] = w4.x;
                        A.v[q * 4 + 1][i] = w4.y;
                        A.v[q * 4 + 2][i] = w4.z;
                        A.v[q * 4 + 3][i] = w4.w;
                    }
            }
            const unsigned x_tap = (unsigned)((q_kh * a.W + q_kw) * a.x_ps) * 4u;
            const unsigned x_chan = (unsigned)q_cb * 4u;
            const int c_left = c_lane_last - q_cb;   // the lane's channels beyond c_left are padding (the tap's last batch)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const unsigned in_h = (unsigned)(ih0[j] + q_kh) < (unsigned)a.H ? 1u : 0u;
                const unsigned in_w = (unsigned)(iw0[j] + q_kw) < (unsigned)a.W ? 1u : 0u;
                const unsigned voff = (x_lane[j] + x_tap) | (((in_h & in_w) ^ 1u) << 31);
#pragma unroll
                for (int q = 0; q < U / 4; q++) {
                    const unsigned c_kill = (unsigned)(c_left - 4 * q) & kOutOfRange;   // sign bit: the whole quad is padding
                    const floatx4 x4 = buffer_load_f32x4(xr, voff | c_kill, x_chan + (unsigned)(16 * q));
#pragma unroll
                    for (int u = 0; u < 4; u++) B[4 * q + u][j] = x4[u];
                }
            }
            left = c_left;
            // next batch (selects, not branches: the loop body stays one basic block)
            q_w += RP >= 3 ? (unsigned)((U * M::KSTEP / 8) * PLANES * a.OCgP) * 16u : (unsigned)((U * M::KSTEP / 4) * a.OCgP) * (RP != 0 ? 8u : 16u);
            q_cb += U * M::KSTEP;
            const bool next_tap = q_cb >= a.ICgP;
            q_cb = next_tap ? 0 : q_cb;
            q_kw += next_tap ? 1 : 0;
            const bool next_row = q_kw == a.KW;
            q_kw = next_row ? 0 : q_kw;
            q_kh += next_row ? 1 : 0;
            return;
        }
        (void)live;   // steps at or beyond s_end are dead by their index
        (void)left;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const bool s_ok = (s0 + u) < s_end;
            const int kb = (s0 + u) * M::KSTEP;
            const int tap = (int)__umulhi((unsigned)kb, a.magic_icgp);
            const int cb = kb - tap * a.ICgP;
            const int kh = a.KW == 1 ? tap : (int)__umulhi((unsigned)tap, a.magic_kw);
            const int kw = tap - kh * a.KW;
            const unsigned w_step = (unsigned)(kb * a.OCgP) * 4u;
            const unsigned step_kill = s_ok ? 0u : kOutOfRange;   // wavefront-uniform
#pragma unroll
            for (int i = 0; i < TM; i++) A.v[u][i] = buffer_load_f32(wr, (w_lane[i] + w_step) | w_kill[i] | step_kill);
            const unsigned x_step = (unsigned)((kh * a.W + kw) * a.x_ps + cb) * 4u;
            const unsigned c_kill = (unsigned)(a.ICg - 1 - cb - lk) & kOutOfRange;   // sign bit: channel padding
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const unsigned in_h = (unsigned)(ih0[j] + kh) < (unsigned)a.H ? 1u : 0u;
                const unsigned in_w = (unsigned)(iw0[j] + kw) < (unsigned)a.W ? 1u : 0u;
                const unsigned kill = ((in_h & in_w) ^ 1u) << 31;
                B[u][j] = buffer_load_f32(xr, (x_lane[j] + x_step) | kill | c_kill | n_kill[j] | step_kill);
            }
        }
    };
    // folded ReLU of the producer: as integers, negative floats are below 0 and everything is above INT_MIN
    const float floor = relu_floor(a.pre_relu != 0);
    const bool ragged = QUAD && (a.ICg & 3) != 0;   // (a branch around register work only, see load_batch)
    auto compute = [&](const FilterStage &A, float(&B)[U][TN], int left) {
        if (ragged) {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int j = 0; j < TN; j++) B[u][j] = u <= left ? B[u][j] : 0.f;
        }
        if constexpr (RP == 3) {
            uintx4 bq[2][TN];
#pragma unroll
            for (int j = 0; j < TN; j++) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = relu_above(floor, B[u][j]);
                const float mine = octet_peak(v), peak = pixel_peak<MT>(mine);
                unsigned &limit = in.limit[j];
                if (__builtin_expect(__ballot(peak >= __uint_as_float(limit)) != 0, 0)) {   // the sums follow
                    const unsigned next = peak >= __uint_as_float(limit) ? limit_for(peak) : limit;
                    in.wild[j] = in.wild[j] || (next != limit && limit_loses(limit, next));
                    const float ratio = limit_ratio(limit, next);
                    limit = next;
#pragma unroll
                    for (int i = 0; i < TM; i++) acc[i][j] *= ratio;
                }
                const unsigned long long small = __ballot(__float_as_uint(mine) - 1u < limit - (kWindow + 1u));
                if (__builtin_expect(small != 0, 0)) below += (unsigned)__popcll(small);
                split_half2(v, limit_scale(limit), bq[0][j], bq[1][j]);
            }
            multiply_terms<2, true>(acc, A.v, bq);
            return;
        } else if constexpr (RP == 5) {
#pragma unroll
            for (int j = 0; j < TN; j++) {
                floatx8 v;
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = relu_above(floor, B[u][j]);
                const uintx4 bq = __builtin_bit_cast(uintx4, __builtin_convertvector(v, halfx8));   // round to nearest even, overflow to infinity
#pragma unroll
                for (int i = 0; i < TM; i++) acc[i][j] = multiply_half(A.v[0][i], bq, acc[i][j]);
            }
            return;
        } else if constexpr (RP == 4) {
            // one rounded term: the reduced-precision mode on the 32 x 32 x 16 instruction
#pragma unroll
            for (int j = 0; j < TN; j++) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = relu_above(floor, B[u][j]);
                const bf16x8 bq = __builtin_bit_cast(bf16x8, round_bf16x8(v));
#pragma unroll
                for (int i = 0; i < TM; i++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, A.v[0][i]), bq, acc[i][j], 0, 0, 0);
            }
            return;
        } else if constexpr (RP != 0) {
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const floatx4 b32 = {relu_above(floor, B[0][j]), relu_above(floor, B[1][j]),
                                     relu_above(floor, B[2][j]), relu_above(floor, B[3][j])};
                if constexpr (RP == 1) {
                    const bf16x4 b4 = __builtin_convertvector(b32, bf16x4);   // round to nearest even
#pragma unroll
                    for (int i = 0; i < TM; i++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(bf16x4, A.v[i]), b4, acc[i][j], 0, 0, 0);
                } else {
                    const halfx4 b4 = __builtin_convertvector(b32, halfx4);   // round to nearest even, overflow to infinity
#pragma unroll
                    for (int i = 0; i < TM; i++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(halfx4, A.v[i]), b4, acc[i][j], 0, 0, 0);
                }
            }
            return;
        } else {
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        const float bval = relu_above(floor, B[u][j]);
                        acc[i][j] = M::run(A.v[u][i], bval, acc[i][j]);
                    }
        }
    };

    const int batches = (s_end - s_begin + U - 1) / U;   // <= 0 for wavefronts beyond the end of K
    auto k_loop = [&]() {
        if (batches <= 0) return;
        if constexpr (D == 2) {
            // Two stages, peeled so that every load sits in straight-line code: the steady state requests batch b + 1,
            // consumes batch b, requests b + 2, consumes b + 1 with both requests known to be in range; the last one or two
            // batches are consumed behind the loop.  The waits in front of the matrix instructions then count exactly the
            // loads issued since, and the next batch's latency overlaps this batch's matrix work.  (The scheduling fences
            // keep a stage's requests behind the matrix work that still reads the stage: moved ahead of it they need a
            // second set of registers.)
            load_batch(s_begin, av[0], bv[0], left[0], true);
            int b = 0;
            for (; b + 2 < batches; b += 2) {
                load_batch(s_begin + (b + 1) * U, av[1], bv[1], left[1], true);
                __builtin_amdgcn_sched_barrier(0);
                compute(av[0], bv[0], left[0]);
                __builtin_amdgcn_sched_barrier(0);
                load_batch(s_begin + (b + 2) * U, av[0], bv[0], left[0], true);
                __builtin_amdgcn_sched_barrier(0);
                compute(av[1], bv[1], left[1]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (b + 1 < batches) {
                load_batch(s_begin + (b + 1) * U, av[1], bv[1], left[1], true);
                __builtin_amdgcn_sched_barrier(0);
                compute(av[0], bv[0], left[0]);
                compute(av[1], bv[1], left[1]);
            } else {
                compute(av[0], bv[0], left[0]);
            }
        } else {
            // deeper pipeline: D batches requested before the first one is consumed.  The loop body is straight-line
            // (requests beyond the range are issued dead, see load_batch: at most D - 1 of them in the last round that
            // requests anything); the last D batches are consumed behind the loop, where nothing is requested any more.
#pragma unroll
            for (int st = 0; st < D; st++) load_batch(s_begin + st * U, av[st], bv[st], left[st], st < batches);
            int b = 0;
            for (; b + D < batches; b += D) {
#pragma unroll
                for (int st = 0; st < D; st++) {
                    compute(av[st], bv[st], left[st]);
                    __builtin_amdgcn_sched_barrier(0);
                    load_batch(s_begin + (b + st + D) * U, av[st], bv[st], left[st], b + st + D < batches);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int st = 0; st < D; st++)
                if (b + st < batches) compute(av[st], bv[st], left[st]);
        }
    };
    k_loop();
    // partial tiles meet in LDS: quad e4 (accumulator elements 4 * e4 ... + 3) of lane l of wavefront w lives in
    // red4[(w * G + e4) * 64 + l]
    floatx4 *red4 = reinterpret_cast<floatx4 *>(red);
    auto hand_over = [&](const typename M::acc_t (&acc)[TM][TN]) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < M::ACC / 4; q++) {
                    const floatx4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                    red4[(wave * G + (i * TN + j) * (M::ACC / 4) + q) * 64 + lane] = v;
                }
    };
    // two terms: whether a wavefront's sums are those of the filters as they were given, not of the scaled ones
    int *exact_flags = reinterpret_cast<int *>(red) + NW * E * 64;
    if constexpr (RP != 3) {
        hand_over(acc);
    } else {
        auto pixel_of = [&](int j) {
            const int n = n0 + j * MT + lc;
            return n < a.Npix ? n : -1;
        };
        unscale_inputs(acc, in.limit);
        in.octets = below;
        floatx4 least[TM];
#pragma unroll
        for (int i = 0; i < TM; i++) least[i] = channel_least_quad(a, g, m0 + i * MT + 4 * (lane % (MT / 4)));
        const bool off = batches > 0 && sums_look_off<MT>(a, acc, in, least, m0, pixel_of);
        hand_over(acc);
        if constexpr (GPW > 1) request_bias();   // (more of them wait until the K loop has given its registers back)
        bool scaled = true;
        if (__builtin_expect(off, 0)) scaled = sums_hold<MT, TM, TN>(a, red4 + wave * G * 64, in, g, m0, pixel_of, s_begin * M::KSTEP, s_end * M::KSTEP, 0, a.ICgP);
        if (lane == 0) exact_flags[wave] = scaled ? 0 : 1;
    }
    __syncthreads();
    auto meet = [&](int t) {   // quad wave + t * NW of the tile: wavefronts in ascending order
        const int e4 = wave + t * NW;
        floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; w++) sum += red4[(w * G + e4) * 64 + lane];
        if constexpr (RP == 3) {
            int any = 0;
#pragma unroll
            for (int w = 0; w < NW; w++) any |= exact_flags[w];
            sum *= factor_pre[t];
            if (__builtin_expect(__builtin_amdgcn_readfirstlane(any) != 0, 0)) {
                sum = floatx4{0.f, 0.f, 0.f, 0.f};
                for (int w = 0; w < NW; w++) {
                    const floatx4 part = red4[(w * G + e4) * 64 + lane];
                    sum += exact_flags[w] != 0 ? part : part * factor_pre[t];
                }
            }
        }
        return sum;
    };
    auto quad_pixel = [&](int e4) { return n0 + ((4 * e4 / M::ACC) % TN) * MT + lc; };
    if (a.split_k > 1 && a.counters == nullptr) {
        // two-kernel split-K: this slice's partial outputs as [slice][pixel][channel] for splitk_reduce_kernel
        const size_t channels = (size_t)a.groups * a.OCg;
        float *wsz = a.ws + (size_t)z * channels * (size_t)a.Npix + (size_t)g * a.OCg;
#pragma unroll
        for (int t = 0; t < GPW; t++) {
            const int e4 = wave + t * NW;
            if (e4 >= G) break;
            const floatx4 sum = meet(t);
            const int m = quad_row(e4), nn = quad_pixel(e4);
#pragma unroll
            for (int c = 0; c < 4; c++)
                if (m + c < a.OCg && nn < a.Npix) wsz[(size_t)nn * channels + m + c] = sum[c];
        }
        return;
    }
    float *slices = nullptr;
    if (a.split_k > 1) {
        // one-kernel split-K, as in the LDS-tiled kernel: partial tiles in [element][lane] order, a ticket per
        // tile, the block drawing the last ticket adds the slices in slice order
        const size_t tiles = (size_t)xcd_padded_tiles(a.tiles_m * a.tiles_n);
        slices = a.ws + (((size_t)g * tiles + tile) * a.split_k) * (size_t)(BM * BN);
        unsigned *counter = a.counters + (size_t)g * tiles + tile;
        int *last_flag = reinterpret_cast<int *>(red);
        auto hand_in = [&](auto local) {
            constexpr bool LOCAL = decltype(local)::value;
            float *mine = slices + (size_t)z * (BM * BN) + lane;
#pragma unroll
            for (int t = 0; t < GPW; t++) {
                const int e4 = wave + t * NW;
                if (e4 >= G) break;
                const floatx4 sum = meet(t);
#pragma unroll
                for (int c = 0; c < 4; c++) partial_store<LOCAL>(mine + (4 * e4 + c) * 64, sum[c]);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (tid == 0) *last_flag = draw_ticket<LOCAL>(counter, a.split_k);
        };
        if (a.xcd_local) hand_in(std::true_type{});
        else hand_in(std::false_type{});
        __syncthreads();
        if (*last_flag == 0) return;
    }
    const bool xcd_local = a.xcd_local != 0;
#pragma unroll
    for (int t = 0; t < GPW; t++) {
        const int e4 = wave + t * NW;
        if (e4 >= G) break;
        floatx4 sum = {0.f, 0.f, 0.f, 0.f};
        if (a.split_k > 1) {
            const float *theirs = slices + 4 * e4 * 64 + lane;
            for (int s2 = 0; s2 < a.split_k; s2++)
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const float *p = theirs + (size_t)s2 * (BM * BN) + c * 64;
                    sum[c] += xcd_local ? partial_load<true>(p) : partial_load<false>(p);
                }
        } else {
            sum = meet(t);
        }
        const int m = quad_row(e4), nn = quad_pixel(e4);
        if (m < a.OCg && nn < a.Npix) finish_quad<RES>(a, sum, bias_pre[t], g, m, nn);
    }
}   // run
};

// ---- kernel configurations ------------------------------------------------------------------------------------------
// X(index, name, BM, BN, BK, WM, WN, WK, MT, PD) for the LDS-tiled kernel
#define IOS_TILED_VARIANTS(X)                                    \
    X(0, "m64n64k32_w2x2x1_t32", 64, 64, 32, 2, 2, 1, 32, 3)     \
    X(1, "m128n128k16_w2x2x1_t32", 128, 128, 16, 2, 2, 1, 32, 3) \
    X(2, "m32n32k64_w1x1x4_t32", 32, 32, 64, 1, 1, 4, 32, 4)     \
    X(3, "m64n32k32_w2x1x2_t32", 64, 32, 32, 2, 1, 2, 32, 4)     \
    X(4, "m32n64k32_w1x2x2_t32", 32, 64, 32, 1, 2, 2, 32, 4)     \
    X(5, "m128n64k16_w2x2x1_t32", 128, 64, 16, 2, 2, 1, 32, 3)   \
    X(6, "m64n16k64_w4x1x1_t16", 64, 16, 64, 4, 1, 1, 16, 3)     \
    X(7, "m32n16k64_w2x1x2_t16", 32, 16, 64, 2, 1, 2, 16, 4)     \
    X(8, "m16n16k128_w1x1x4_t16", 16, 16, 128, 1, 1, 4, 16, 3)   \
    X(9, "m64n128k16_w2x2x1_t32", 64, 128, 16, 2, 2, 1, 32, 3)   \
    X(10, "m64n64k16_w2x2x1_t32", 64, 64, 16, 2, 2, 1, 32, 4)    \
    X(11, "m32n128k16_w1x4x1_t32", 32, 128, 16, 1, 4, 1, 32, 4)  \
    X(12, "m192n64k16_w2x2x1_t32", 192, 64, 16, 2, 2, 1, 32, 3)  \
    X(13, "m96n128k16_w1x4x1_t32", 96, 128, 16, 1, 4, 1, 32, 3)  \
    X(14, "m192n128k16_w2x2x1_t32", 192, 128, 16, 2, 2, 1, 32, 3) \
    X(15, "m160n128k16_w1x4x1_t32", 160, 128, 16, 1, 4, 1, 32, 3)
// X(index, name, MT, TM, TN, NW, U, QUAD, D, BF16) for the wave-split kernel
#define IOS_WSPLIT_VARIANTS(X)                     \
    X(16, "ws_m32n16_w16_t16", 16, 2, 1, 16, 4, false, 2, false)    \
    X(17, "ws_m16n16_w16_t16", 16, 1, 1, 16, 8, false, 2, false)    \
    X(18, "ws_m32n32_w16_t16", 16, 2, 2, 16, 4, false, 2, false)    \
    X(19, "ws_m64n16_w16_t16", 16, 4, 1, 16, 4, false, 2, false)    \
    X(20, "ws_m32n16_w8_t16", 16, 2, 1, 8, 4, false, 2, false)      \
    X(21, "ws_m32n16_w4_t16", 16, 2, 1, 4, 8, false, 2, false)      \
    X(22, "ws_m32n32_w16_t32", 32, 1, 1, 16, 8, false, 2, false)    \
    X(23, "ws_m16n32_w16_t16", 16, 1, 2, 16, 4, false, 2, false)    \
    X(24, "wq_m32n16_w16_t16", 16, 2, 1, 16, 4, true, 2, false)     \
    X(25, "wq_m32n16_w8_t16", 16, 2, 1, 8, 4, true, 2, false)       \
    X(26, "wq_m32n32_w16_t16", 16, 2, 2, 16, 4, true, 2, false)     \
    X(27, "wq_m16n16_w16_t16", 16, 1, 1, 16, 4, true, 2, false)     \
    X(28, "wq_m64n16_w8_t16", 16, 4, 1, 8, 4, true, 2, false)       \
    X(29, "wq_m64n32_w8_t16", 16, 4, 2, 8, 4, true, 2, false)       \
    X(30, "wq_m64n64_w4_t16", 16, 4, 4, 4, 4, true, 2, false)       \
    X(31, "wq_m64n32_w4_t16", 16, 4, 2, 4, 4, true, 2, false)       \
    X(32, "wq_m32n32_w8_t16", 16, 2, 2, 8, 4, true, 2, false)       \
    X(33, "wq_m64n64_w4_t32", 32, 2, 2, 4, 8, true, 2, false)       \
    X(34, "wq_m16n16_w16_t16_d4", 16, 1, 1, 16, 4, true, 4, false) \
    X(35, "wq_m32n16_w8_t16_d4", 16, 2, 1, 8, 4, true, 4, false)   \
    X(36, "wq_m32n16_w16_t16_d4", 16, 2, 1, 16, 4, true, 4, false) \
    X(37, "wq_m16n16_w8_t16_d4", 16, 1, 1, 8, 4, true, 4, false)   \
    X(38, "wq_m32n32_w4_t16", 16, 2, 2, 4, 4, true, 2, false)      \
    X(39, "wq_m32n32_w2_t16_d4", 16, 2, 2, 2, 4, true, 4, false)   \
    X(40, "wq_m64n32_w2_t16", 16, 4, 2, 2, 4, true, 2, false)      \
    X(41, "wq_m32n64_w4_t16", 16, 2, 4, 4, 4, true, 2, false)      \
    X(42, "wq_m64n32_w4_t16_d4", 16, 4, 2, 4, 4, true, 4, false) \
    X(43, "wb_m16n16_w16", 16, 1, 1, 16, 4, true, 2, true)    \
    X(44, "wb_m16n16_w8_d4", 16, 1, 1, 8, 4, true, 4, true)   \
    X(45, "wb_m32n16_w8", 16, 2, 1, 8, 4, true, 2, true)      \
    X(46, "wb_m32n16_w16", 16, 2, 1, 16, 4, true, 2, true)    \
    X(47, "wb_m32n32_w8", 16, 2, 2, 8, 4, true, 2, true)      \
    X(48, "wb_m32n32_w4_d4", 16, 2, 2, 4, 4, true, 4, true)   \
    X(49, "wb_m64n16_w8", 16, 4, 1, 8, 4, true, 2, true)      \
    X(50, "wb_m64n32_w8", 16, 4, 2, 8, 4, true, 2, true)      \
    X(51, "wb_m64n32_w4_d4", 16, 4, 2, 4, 4, true, 4, true)   \
    X(52, "wb_m64n64_w4", 16, 4, 4, 4, 4, true, 2, true)
// X(index, name, MT, TM, TN, NW, U, QUAD, D, BF16): wave-split configurations with channels padded to 4
#define IOS_WSPLIT_C4_VARIANTS(X)                                \
    X(53, "ws_m32n32_w1_t16_c4", 16, 2, 2, 1, 4, false, 2, false) \
    X(54, "ws_m32n64_w1_t16_c4", 16, 2, 4, 1, 4, false, 2, false) \
    X(55, "ws_m32n32_w2_t16_c4", 16, 2, 2, 2, 4, false, 2, false) \
    X(56, "ws_m32n16_w4_t16_c4", 16, 2, 1, 4, 4, false, 2, false)
// X(index, name, MT, TM, TN, NW, U, QUAD, D, BF16): quad-load wave-split configurations on the 32 x 32 x 2 MFMA.  A
// wavefront's input load covers two channels x 32 consecutive pixels (two full 128-byte lines) instead of four
// channels x 16 pixels, and the instruction's ceiling is higher than that of the 16 x 16 x 4 form.
#define IOS_WSPLIT_T32_VARIANTS(X)                                   \
    X(57, "wq_m32n32_w8_t32", 32, 1, 1, 8, 8, true, 2, false)        \
    X(58, "wq_m32n32_w16_t32", 32, 1, 1, 16, 8, true, 2, false)      \
    X(59, "wq_m32n32_w4_t32", 32, 1, 1, 4, 8, true, 2, false)        \
    X(60, "wq_m64n32_w8_t32", 32, 2, 1, 8, 8, true, 2, false)        \
    X(61, "wq_m64n32_w4_t32", 32, 2, 1, 4, 8, true, 2, false)        \
    X(62, "wq_m32n64_w8_t32", 32, 1, 2, 8, 8, true, 2, false)        \
    X(63, "wq_m32n64_w4_t32", 32, 1, 2, 4, 8, true, 2, false)        \
    X(64, "wq_m64n64_w8_t32", 32, 2, 2, 8, 8, true, 2, false)        \
    X(65, "wq_m32n32_w8_t32_u4", 32, 1, 1, 8, 4, true, 2, false)     \
    X(66, "wq_m64n32_w8_t32_u4", 32, 2, 1, 8, 4, true, 2, false)     \
    X(67, "wq_m64n64_w4_t32_u4", 32, 2, 2, 4, 4, true, 2, false)     \
    X(68, "wq_m64n32_w4_t32_u4_d4", 32, 2, 1, 4, 4, true, 4, false)
// X(index, name, MT, TM, TN, NW, U, QUAD, D, RP): the reduced-precision configurations once more with IEEE half operands
// (RP = 2, option precision=fp16), the literal counterpart of the reference's USE_FLOAT16 build
#define IOS_WSPLIT_F16_VARIANTS(X)                          \
    X(69, "wh_m16n16_w16", 16, 1, 1, 16, 4, true, 2, 2)     \
    X(70, "wh_m16n16_w8_d4", 16, 1, 1, 8, 4, true, 4, 2)    \
    X(71, "wh_m32n16_w8", 16, 2, 1, 8, 4, true, 2, 2)       \
    X(72, "wh_m32n16_w16", 16, 2, 1, 16, 4, true, 2, 2)     \
    X(73, "wh_m32n32_w8", 16, 2, 2, 8, 4, true, 2, 2)       \
    X(74, "wh_m32n32_w4_d4", 16, 2, 2, 4, 4, true, 4, 2)    \
    X(75, "wh_m64n16_w8", 16, 4, 1, 8, 4, true, 2, 2)       \
    X(76, "wh_m64n32_w8", 16, 4, 2, 8, 4, true, 2, 2)       \
    X(77, "wh_m64n32_w4_d4", 16, 4, 2, 4, 4, true, 4, 2)    \
    X(78, "wh_m64n64_w4", 16, 4, 4, 4, 4, true, 2, 2)
// X(index, name, MT, TM, TN, NW, U, QUAD, D, RP): quad-load configurations with one or two wavefronts per output tile, for
// layers with many pixels and a short K (the first layers of an image network at batch 1, everything at large batches):
// a wavefront walks (half of) K by itself, its next batch's loads in flight under this batch's matrix instructions
#define IOS_WSPLIT_LONGK_VARIANTS(X)                                  \
    X(79, "wq_m32n32_w1_t32", 32, 1, 1, 1, 8, true, 2, 0)             \
    X(80, "wq_m32n32_w2_t32", 32, 1, 1, 2, 8, true, 2, 0)             \
    X(81, "wq_m64n32_w2_t32", 32, 2, 1, 2, 8, true, 2, 0)             \
    X(82, "wq_m64n32_w1_t32", 32, 2, 1, 1, 8, true, 2, 0)             \
    X(83, "wq_m32n64_w2_t32", 32, 1, 2, 2, 8, true, 2, 0)             \
    X(84, "wq_m32n32_w2_t32_d4", 32, 1, 1, 2, 8, true, 4, 0)          \
    X(85, "wq_m64n32_w2_t32_u4_d4", 32, 2, 1, 2, 4, true, 4, 0)       \
    X(86, "wq_m32n32_w1_t16_d4", 16, 2, 2, 1, 4, true, 4, 0)          \
    X(87, "wq_m64n32_w1_t16", 16, 4, 2, 1, 4, true, 2, 0)             \
    X(88, "wq_m64n64_w2_t32", 32, 2, 2, 2, 8, true, 2, 0)
// X(index, name, TMW, TNW, WM, WN, PD): the LDS-tiled kernel with operands split into three bfloat16 terms (ConvSplit3);
// TMW x TNW tiles of 32 x 32 per wavefront, WM x WN wavefronts
#define IOS_SPLIT3_VARIANTS(X)                     \
    X(89, "x3_m64n128_w2x2", 1, 2, 2, 2, 2)        \
    X(90, "x3_m64n128_w2x2_p3", 1, 2, 2, 2, 3)     \
    X(91, "x3_m64n256_w2x4", 1, 2, 2, 4, 2)        \
    X(92, "x3_m64n64_w2x2", 1, 1, 2, 2, 2)         \
    X(93, "x3_m64n64_w1x1", 2, 2, 1, 1, 2)         \
    X(94, "x3_m64n128_w1x2", 2, 2, 1, 2, 2)        \
    X(95, "x3_m128n64_w4x1", 1, 2, 4, 1, 2)        \
    X(96, "x3_m128n128_w4x2", 1, 2, 4, 2, 2)       \
    X(97, "x3_m192n128_w6x2", 1, 2, 6, 2, 2)
// X(index, name, TM, TN, NW, D): wave-split configurations with operands as two terms of half (ConvWsplit, RP = 3),
// 32 x 32 x 16 tiles, 16 k per batch
#define IOS_WSPLIT_X3_VARIANTS(X)            \
    X(98, "x3w_m32n32_w8", 1, 1, 8, 2)       \
    X(99, "x3w_m32n32_w4", 1, 1, 4, 2)       \
    X(100, "x3w_m32n32_w16", 1, 1, 16, 2)    \
    X(101, "x3w_m64n32_w8", 2, 1, 8, 2)      \
    X(102, "x3w_m64n32_w4", 2, 1, 4, 2)      \
    X(103, "x3w_m32n64_w4", 1, 2, 4, 2)      \
    X(104, "x3w_m32n64_w8", 1, 2, 8, 2)      \
    X(105, "x3w_m64n64_w4", 2, 2, 4, 2)      \
    X(106, "x3w_m64n32_w2", 2, 1, 2, 2)
// X(index, name, TMW, TNW, WM, WN, PD): ConvSplit3 with one rounded term (option precision=bf16), up to 64 x 64 per wavefront
#define IOS_SPLIT1_VARIANTS(X)                      \
    X(107, "wb_x1_m64n128_w2x2", 1, 2, 2, 2, 2)     \
    X(108, "wb_x1_m128n128_w2x2", 2, 2, 2, 2, 2)    \
    X(109, "wb_x1_m128n256_w2x4", 2, 2, 2, 4, 2)    \
    X(110, "wb_x1_m64n128_w1x2", 2, 2, 1, 2, 2)     \
    X(111, "wb_x1_m128n64_w4x1", 1, 2, 4, 1, 2)     \
    X(112, "wb_x1_m64n256_w2x4", 1, 2, 2, 4, 2)
// X(index, name, TM, TN, NW, D): the wave-split kernel with one rounded term (ConvWsplit, RP = 4)
#define IOS_WSPLIT_X1_VARIANTS(X)              \
    X(113, "wb_x1w_m32n32_w4", 1, 1, 4, 2)     \
    X(114, "wb_x1w_m64n32_w4", 2, 1, 4, 2)     \
    X(115, "wb_x1w_m32n64_w4", 1, 2, 4, 2)     \
    X(116, "wb_x1w_m64n64_w4", 2, 2, 4, 2)     \
    X(117, "wb_x1w_m32n32_w8", 1, 1, 8, 2)     \
    X(118, "wb_x1w_m64n64_w2", 2, 2, 2, 2)
// X(index, name, TM, TN, NW, D): two terms of half on 16 x 16 tiles and 32 k per batch (v_mfma_f32_16x16x32_f16), three instructions of
// 16 cycles where the fp32 form takes eight of 32: for problems of few tiles, bound by what the wavefronts of a SIMD issue one after the
// other.  At most 100 registers up to 32 x 16: these run inside every fused launch.  Against the fp32 form, microseconds: 288 -> 384
// 3 x 3 / 2 on 35 x 35 at batch 1 10.9 -> 10.1, 160 -> 192 7 x 1 on 17 x 17 5.9 -> 5.6, 448 -> 384 3 x 3 on 8 x 8 at batch 5 15.0 -> 13.5.
#define IOS_WSPLIT_X3S_VARIANTS(X)                \
    X(156, "x3w_m16n16_w16_t16", 1, 1, 16, 2)     \
    X(157, "x3w_m16n16_w8_t16", 1, 1, 8, 2)       \
    X(158, "x3w_m32n16_w16_t16", 2, 1, 16, 2)     \
    X(159, "x3w_m32n16_w8_t16", 2, 1, 8, 2)       \
    X(160, "x3w_m32n16_w4_t16", 2, 1, 4, 2)       \
    X(161, "x3w_m32n32_w8_t16", 2, 2, 8, 2)       \
    X(162, "x3w_m64n16_w8_t16", 4, 1, 8, 2)       \
    X(163, "x3w_m64n32_w4_t16", 4, 2, 4, 2)
// X(index, name, TM, TN, NW, D): the wave-split kernel with one term rounded to half (ConvWsplit, RP = 5; option precision=fp16).  Against the
// 16 x 16 x 16 forms at batch 7: 192 -> 192 1 x 7 on 17 x 17 9.9 -> 8.6 us, 768 -> 192 7.2 -> 6.7.  (Inside the wide-register fused launches
// they cost a pass of Inception-v3 at batch 7 more than they gain: 789 against 739 us.)
#define IOS_WSPLIT_XH_VARIANTS(X)              \
    X(164, "wh_x1w_m32n32_w4", 1, 1, 4, 2)     \
    X(165, "wh_x1w_m64n32_w4", 2, 1, 4, 2)     \
    X(166, "wh_x1w_m32n64_w4", 1, 2, 4, 2)     \
    X(167, "wh_x1w_m64n64_w4", 2, 2, 4, 2)     \
    X(168, "wh_x1w_m32n32_w8", 1, 1, 8, 2)     \
    X(169, "wh_x1w_m64n32_w8", 2, 1, 8, 2)

// A stand-alone kernel and its residual form
struct KernelPair {
    void (*kernel)(ConvKernelArgs) = nullptr, (*kernel_residual)(ConvKernelArgs) = nullptr;
};
// conv_tiled.hip, in the order of the lists above
extern const KernelPair kTiledKernels[], kSplit3Kernels[], kSplit1Kernels[];
// conv_wsplit_half.hip, likewise
extern const KernelPair kWsplitX3sKernels[], kWsplitXhKernels[];
constexpr int kFirstSplit3Variant = 89, kFirstSplit1Variant = 107, kFirstWsplitX3sVariant = 156, kFirstWsplitXhVariant = 164;
}  // namespace ios
