// Device-side bodies of the memory-bound kernels (pooling, depth-wise and direct convolution, n-ary add /
// multiply / activation / strided copy).  Every body processes the elements of logical block `block` out of
// `num_blocks` with a block-stride loop, so the same code serves a stand-alone launch and a slice of the
// fused stage kernel.  Tensors are NHWC views; a thread takes V consecutive channels of a pixel (V = 4: 16-byte loads and
// stores, for tensors that fill the device with them; V = 1: four times the threads, for the small ones, whose time is the
// latency of a thread's chain), consecutive lanes take consecutive channels, then the next pixel.
#pragma once

#include "kernels.h"

namespace ios {

typedef float pw_floatx4 __attribute__((ext_vector_type(4)));
typedef float pw_floatx4_u __attribute__((ext_vector_type(4), aligned(4)));
typedef float pw_floatx2_u __attribute__((ext_vector_type(2), aligned(4)));

// V consecutive channels; a load may run past the last channel of a pixel (what it brings from there is not stored)
template <int V>
struct Channels {
    float v[V];
};
template <int V>
__device__ __forceinline__ Channels<V> load_channels(const float *p) {
    Channels<V> c;
    if constexpr (V == 4) {
        const pw_floatx4_u q = *reinterpret_cast<const pw_floatx4_u *>(p);
        c.v[0] = q.x; c.v[1] = q.y; c.v[2] = q.z; c.v[3] = q.w;
    } else if constexpr (V == 2) {
        const pw_floatx2_u q = *reinterpret_cast<const pw_floatx2_u *>(p);
        c.v[0] = q.x; c.v[1] = q.y;
    } else {
        c.v[0] = p[0];
    }
    return c;
}
// `left`: channels of the tensor from the first one on
template <int V>
__device__ __forceinline__ void store_channels(float *p, const Channels<V> &c, int left) {
    if (V == 1) {
        p[0] = c.v[0];
    } else if (left >= V) {
        if constexpr (V == 4) {
            const pw_floatx4_u q = {c.v[0], c.v[1], c.v[2], c.v[3]};
            *reinterpret_cast<pw_floatx4_u *>(p) = q;
        } else {
            const pw_floatx2_u q = {c.v[0], c.v[1 % V]};
            *reinterpret_cast<pw_floatx2_u *>(p) = q;
        }
    } else {
#pragma unroll
        for (int k = 0; k < V; k++)
            if (k < left) p[k] = c.v[k];
    }
}

struct PoolArgs {
    const float *x;
    float *y;
    // the pool behind a bias-free convolution (an average pool and a 1 x 1 convolution exchanged): y = act(pool(x) + bias[c]);
    // nullptr for a plain pool
    const float *bias;
    PoolProblem p;
    int x_ps, y_ps;   // elements between pixels
    int strip_rows;   // 3 x 3 windows: output rows per thread (see pool3x3_body); 0 selects the generic body
    int channels;     // channels per thread, 1 or 4
    int act;
    FastDiv div_cv, div_ow, div_strips;   // by channel groups of a pixel, by OW, by strips of a column (rows of outputs without strips)
};

// `bias`: pool_bias() of the channels, requested ahead of the window
template <int V>
__device__ __forceinline__ Channels<V> pool_bias(const PoolArgs &a, int c) {
    Channels<V> b;
#pragma unroll
    for (int k = 0; k < V; k++) b.v[k] = 0.f;
    if (a.bias != nullptr) b = load_channels<V>(a.bias + c);   // (what lies behind the last bias value is not used)
    return b;
}
template <int V>
__device__ __forceinline__ void pool_store(const PoolArgs &a, unsigned pixel, int c, Channels<V> v, const Channels<V> &bias) {
    if (a.bias != nullptr) {
#pragma unroll
        for (int k = 0; k < V; k++) v.v[k] += bias.v[k];
        apply_activation(v.v, a.act);
    }
    store_channels<V>(a.y + (long long)pixel * a.y_ps + c, v, a.p.C - c);
}

template <int V>
__device__ __forceinline__ void pool_generic_body(const PoolArgs &a, int block, int num_blocks, unsigned threads) {
    const PoolProblem &p = a.p;
    // 32-bit index arithmetic: the host side rejects tensors with 2^31 or more elements
    const unsigned cv = (unsigned)((p.C + V - 1) / V);
    const unsigned total = (unsigned)(p.B * p.OH * p.OW) * cv;
    const float inv = 1.0f / (float)(p.KH * p.KW);
    const bool is_max = p.is_max != 0;
    for (unsigned i = block * threads + threadIdx.x; i < total; i += num_blocks * threads) {
        const unsigned pixel = fast_div(i, a.div_cv);
        const int c = (int)(i - pixel * cv) * V;
        const unsigned line = fast_div(pixel, a.div_ow);
        const int ow = (int)(pixel - line * (unsigned)p.OW);
        const unsigned b = fast_div(line, a.div_strips);
        const int oh = (int)(line - b * (unsigned)p.OH);
        const float *xb = a.x + (long long)b * p.H * p.W * a.x_ps + c;
        const int h0 = oh * p.sh - p.ph, w0 = ow * p.sw - p.pw;
        const int hb = max(h0, 0), he = min(h0 + p.KH, p.H);
        const int wb = max(w0, 0), we = min(w0 + p.KW, p.W);
        const Channels<V> bias = pool_bias<V>(a, c);
        Channels<V> out;
#pragma unroll
        for (int k = 0; k < V; k++) out.v[k] = is_max ? -INFINITY : 0.f;
        for (int h = hb; h < he; h++)
            for (int w = wb; w < we; w++) {
                const Channels<V> v = load_channels<V>(xb + (long long)(h * p.W + w) * a.x_ps);
#pragma unroll
                for (int k = 0; k < V; k++) out.v[k] = is_max ? fmaxf(out.v[k], v.v[k]) : out.v[k] + v.v[k];
            }
        if (!is_max)
#pragma unroll
            for (int k = 0; k < V; k++) out.v[k] *= inv;
        pool_store<V>(a, pixel, c, out, bias);
    }
}

// 3 x 3 windows, stride 1 or 2 in h (any stride in w).  A thread walks down a.strip_rows outputs of a column and keeps the
// horizontal partial results of the input rows that consecutive windows share: per output it reads 3 * (1 + 2 / R) (stride 1)
// or 3 * (2 + 1 / R) (stride 2) elements instead of 9.  Clamped addresses and selects instead of conditional loads: the loads
// of a window are independent and in flight together.
constexpr int kPoolStripRows = 8;

template <int V>
__device__ __forceinline__ void pool3x3_body(const PoolArgs &a, int block, int num_blocks, unsigned threads) {
    const PoolProblem &p = a.p;
    const int R = a.strip_rows;
    const unsigned cv = (unsigned)((p.C + V - 1) / V);
    const unsigned strips = (unsigned)((p.OH + R - 1) / R);
    const unsigned total = (unsigned)p.B * strips * (unsigned)p.OW * cv;
    const bool is_max = p.is_max != 0;
    const float neutral = is_max ? -INFINITY : 0.f;
    for (unsigned i = block * threads + threadIdx.x; i < total; i += num_blocks * threads) {
        const unsigned column = fast_div(i, a.div_cv);
        const int c = (int)(i - column * cv) * V;
        const unsigned line = fast_div(column, a.div_ow);
        const int ow = (int)(column - line * (unsigned)p.OW);
        const unsigned b = fast_div(line, a.div_strips);
        const int strip = (int)(line - b * strips);
        const float *xb = a.x + (long long)b * p.H * p.W * a.x_ps + c;
        const unsigned y0 = b * (unsigned)(p.OH * p.OW) + (unsigned)ow;
        const Channels<V> bias = pool_bias<V>(a, c);
        const int w0 = ow * p.sw - p.pw;
        const bool c0 = (unsigned)w0 < (unsigned)p.W, c1 = (unsigned)(w0 + 1) < (unsigned)p.W, c2 = (unsigned)(w0 + 2) < (unsigned)p.W;
        const int wa = min(max(w0, 0), p.W - 1) * a.x_ps, wb = min(max(w0 + 1, 0), p.W - 1) * a.x_ps, wc = min(max(w0 + 2, 0), p.W - 1) * a.x_ps;
        auto row = [&](int h) -> Channels<V> {
            const bool in_h = (unsigned)h < (unsigned)p.H;
            const float *xr = xb + (long long)(min(max(h, 0), p.H - 1) * p.W) * a.x_ps;
            const Channels<V> l0 = load_channels<V>(xr + wa), l1 = load_channels<V>(xr + wb), l2 = load_channels<V>(xr + wc);
            Channels<V> r;
#pragma unroll
            for (int k = 0; k < V; k++) {
                const float v0 = (c0 && in_h) ? l0.v[k] : neutral;
                const float v1 = (c1 && in_h) ? l1.v[k] : neutral;
                const float v2 = (c2 && in_h) ? l2.v[k] : neutral;
                r.v[k] = is_max ? fmaxf(fmaxf(v0, v1), v2) : (v0 + v1) + v2;
            }
            return r;
        };
        auto store = [&](int oh, const Channels<V> &r0, const Channels<V> &r1, const Channels<V> &r2) {
            Channels<V> o;
#pragma unroll
            for (int k = 0; k < V; k++)
                o.v[k] = is_max ? fmaxf(fmaxf(r0.v[k], r1.v[k]), r2.v[k]) : ((r0.v[k] + r1.v[k]) + r2.v[k]) * (1.0f / 9.0f);
            pool_store<V>(a, y0 + (unsigned)(oh * p.OW), c, o, bias);
        };
        const int oh_begin = strip * R;
        const int oh_end = min(p.OH, oh_begin + R);
        if (p.sh == 1) {
            Channels<V> r0 = row(oh_begin - p.ph), r1 = row(oh_begin - p.ph + 1);
            for (int oh = oh_begin; oh < oh_end; oh++) {
                const Channels<V> r2 = row(oh - p.ph + 2);
                store(oh, r0, r1, r2);
                r0 = r1;
                r1 = r2;
            }
        } else {
            Channels<V> r0 = row(oh_begin * 2 - p.ph);
            for (int oh = oh_begin; oh < oh_end; oh++) {
                const Channels<V> r1 = row(oh * 2 - p.ph + 1);
                const Channels<V> r2 = row(oh * 2 - p.ph + 2);
                store(oh, r0, r1, r2);
                r0 = r2;
            }
        }
    }
}

__device__ __forceinline__ void pool_body(const PoolArgs &a, int block, int num_blocks, unsigned threads) {
    if (a.strip_rows > 0) {
        if (a.channels == 4) pool3x3_body<4>(a, block, num_blocks, threads);
        else pool3x3_body<1>(a, block, num_blocks, threads);
    } else {
        if (a.channels == 4) pool_generic_body<4>(a, block, num_blocks, threads);
        else pool_generic_body<1>(a, block, num_blocks, threads);
    }
}

// window == whole map: a wavefront takes kGlobalPoolChannels neighbouring channels of an image (64 contiguous bytes per pixel),
// a quarter of the pixels each lane, and the four quarters meet across the lanes
constexpr int kGlobalPoolChannels = 16;

__device__ __forceinline__ void global_pool_body(const PoolArgs &a, int block, int num_blocks, unsigned threads) {
    const PoolProblem &p = a.p;
    const int HW = p.H * p.W;
    const unsigned groups = (unsigned)((p.C + kGlobalPoolChannels - 1) / kGlobalPoolChannels);
    const unsigned units = groups * (unsigned)p.B;
    const unsigned waves_per_block = threads >> 6;
    const int lane = threadIdx.x & 63;
    for (unsigned unit = block * waves_per_block + (threadIdx.x >> 6); unit < units; unit += num_blocks * waves_per_block) {
        const unsigned b = unit / groups;
        const int c = (int)(unit - b * groups) * kGlobalPoolChannels + (lane & 15);
        const float *xc = a.x + (long long)b * HW * a.x_ps + min(c, p.C - 1);
        float best = -INFINITY, sum = 0.f;
        int i = lane >> 4;
        for (; i + 28 < HW; i += 32) {   // eight pixels in flight
            float v[8];
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = xc[(long long)(i + 4 * k) * a.x_ps];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                best = fmaxf(best, v[k]);
                sum += v[k];
            }
        }
        for (; i < HW; i += 4) {
            const float v = xc[(long long)i * a.x_ps];
            best = fmaxf(best, v);
            sum += v;
        }
        for (int off = 16; off < 64; off <<= 1) {
            best = fmaxf(best, __shfl_xor(best, off, 64));
            sum += __shfl_xor(sum, off, 64);
        }
        if (lane < 16 && c < p.C) {
            Channels<1> out;
            out.v[0] = p.is_max ? best : sum / (float)HW;
            pool_store<1>(a, b, c, out, pool_bias<1>(a, c));
        }
    }
}

struct DirectConvArgs {
    const float *x;
    const float *w;   // depth-wise: [tap][C rounded up to 4], else [OC][C / groups][KH][KW]
    const float *bias;
    float *y;
    ConvProblem p;
    int x_ps, y_ps;     // elements between pixels
    unsigned x_bytes;   // extent of the input view in bytes when it is below 2^31 (branch-free depth-wise loads), else 0
    int channels;       // depth-wise: channels per thread
    FastDiv div_cv, div_ow, div_oh;
    // depth-wise convolution of a sum: the input is x + more[0] + ... + more[nmore - 1] (added left to right, then the
    // folded ReLU), every view of the shape of x; the reference adds them with a kernel of its own (src/ios/ops.cu:26-48)
    int nmore;
    const float *more[kMaxNaryInputs - 1];
    int more_ps[kMaxNaryInputs - 1];
    unsigned more_bytes[kMaxNaryInputs - 1];
};

// raw buffer loads as in the matrix-path convolution: an offset with the top bit set is out of range and reads zero
template <int V>
__device__ __forceinline__ Channels<V> pw_buffer_load(__amdgpu_buffer_rsrc_t r, unsigned byte_offset) {
    Channels<V> c;
    if constexpr (V == 4) {
        const auto q = __builtin_amdgcn_raw_buffer_load_b128(r, byte_offset, 0, 0);
#pragma unroll
        for (int k = 0; k < 4; k++) c.v[k] = __uint_as_float(q[k]);
    } else if constexpr (V == 2) {
        const auto q = __builtin_amdgcn_raw_buffer_load_b64(r, byte_offset, 0, 0);
        c.v[0] = __uint_as_float(q[0]);
        c.v[1] = __uint_as_float(q[1]);
    } else {
        c.v[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, byte_offset, 0, 0));
    }
    return c;
}

// Depth-wise convolution.  Fixed windows: every tap is one independent load, taps outside the image get the out-of-range bit.
// V = 1: all KH * KW loads of an output are in flight together (and, for a sum, those of two further inputs for 3 x 3 windows).
// V = 4: a window row at a time with the next one in flight, which is what fits the registers.
// SUM: the instantiation that adds further inputs in its loader (kept apart so that the common single-input form stays small)
template <int KH, int KW, int V, bool SUM = false>
__device__ __forceinline__ void dwconv_body(const DirectConvArgs &a, int block, int num_blocks, unsigned threads) {
    const ConvProblem &p = a.p;
    const int kh_n = KH > 0 ? KH : p.KH, kw_n = KW > 0 ? KW : p.KW;
    const unsigned cv = (unsigned)((p.OC + V - 1) / V);
    const unsigned total = (unsigned)(p.B * p.OH * p.OW) * cv;
    const int w_ps = (p.OC + 3) & ~3;
    const float floor = relu_floor(p.pre_relu != 0);
    for (unsigned i = block * threads + threadIdx.x; i < total; i += num_blocks * threads) {
        const unsigned pixel = fast_div(i, a.div_cv);
        const int c = (int)(i - pixel * cv) * V;
        const unsigned line = fast_div(pixel, a.div_ow);
        const int ow = (int)(pixel - line * (unsigned)p.OW);
        const unsigned b = fast_div(line, a.div_oh);
        const int oh = (int)(line - b * (unsigned)p.OH);
        const float *wc = a.w + c;
        const int h0 = oh * p.sh - p.ph, w0 = ow * p.sw - p.pw;
        Channels<V> acc;
#pragma unroll
        for (int k = 0; k < V; k++) acc.v[k] = a.bias[c + k];   // (what lies behind the last bias value is not used)
        auto add_tap = [&](const Channels<V> &x, int tap) {
            const Channels<V> f = load_channels<V>(wc + tap * w_ps);
#pragma unroll
            for (int k = 0; k < V; k++) acc.v[k] = fmaf(relu_above(floor, x.v[k]), f.v[k], acc.v[k]);
        };
        bool done = false;
        if constexpr (KH > 0) if (a.x_bytes != 0) {
            done = true;
            const unsigned corner = (unsigned)((int)(b * (unsigned)p.H) + h0) * (unsigned)p.W + (unsigned)w0;   // may wrap below zero
            constexpr int ROWS = V == 1 || SUM ? KH : 1;   // window rows in flight as one set
            // one set of rows of one input
            auto load_rows = [&](__amdgpu_buffer_rsrc_t r, int ps, int first, Channels<V>(&v)[ROWS > 0 ? ROWS * KW : 1]) {
                const unsigned base = (corner * (unsigned)ps + (unsigned)c) * 4u;
#pragma unroll
                for (int i2 = 0; i2 < ROWS; i2++) {
                    const unsigned row_kill = (unsigned)(h0 + first + i2) < (unsigned)p.H ? 0u : 0x80000000u;
#pragma unroll
                    for (int j = 0; j < KW; j++) {
                        const unsigned kill = (unsigned)(w0 + j) < (unsigned)p.W ? row_kill : 0x80000000u;
                        v[i2 * KW + j] = pw_buffer_load<V>(r, (base + (unsigned)(((first + i2) * p.W + j) * ps) * 4u) | kill);
                    }
                }
            };
            const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.x), 0, a.x_bytes, 0x00020000);
            if constexpr (ROWS == KH) {
                Channels<V> v[KH > 0 ? KH * KW : 1];
                load_rows(xr, a.x_ps, 0, v);
                if constexpr (SUM) {
                    // two further inputs at a time for 3 x 3 windows of one channel per thread, where a missing second one has
                    // extent zero and reads zeros, else one at a time
                    constexpr int PAIR = KH * KW * V <= 18 ? 2 : 1;
                    // unrolled with wavefront-uniform guards: indexing the argument arrays with a loop variable would move them to scratch memory
#pragma unroll
                    for (int s = 0; s < kMaxNaryInputs - 1; s += PAIR) {
                        if (s >= a.nmore) break;
                        Channels<V> u[PAIR][KH > 0 ? KH * KW : 1];
#pragma unroll
                        for (int e = 0; e < PAIR; e++) {
                            constexpr int kLast = kMaxNaryInputs - 2;
                            const int se = s + e < kLast ? s + e : kLast;
                            const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.more[se]), 0,
                                                                                                 s + e < a.nmore ? a.more_bytes[se] : 0u, 0x00020000);
                            load_rows(sr, a.more_ps[se], 0, u[e]);
                        }
#pragma unroll
                        for (int t = 0; t < KH * KW; t++)
#pragma unroll
                            for (int k = 0; k < V; k++) {
                                v[t].v[k] += u[0][t].v[k];
                                if (PAIR > 1 && s + 1 < a.nmore) v[t].v[k] += u[PAIR - 1][t].v[k];   // wavefront-uniform; skipping keeps -0.0 + 0.0 out of the sum
                            }
                    }
                }
#pragma unroll
                for (int t = 0; t < KH * KW; t++) add_tap(v[t], t);
            } else {
                Channels<V> v[2][KW > 0 ? KW : 1];
                load_rows(xr, a.x_ps, 0, v[0]);
#pragma unroll
                for (int i2 = 0; i2 < KH; i2++) {
                    if (i2 + 1 < KH) load_rows(xr, a.x_ps, i2 + 1, v[(i2 + 1) & 1]);
#pragma unroll
                    for (int j = 0; j < KW; j++) add_tap(v[i2 & 1][j], i2 * KW + j);
                }
            }
        }
        if (!done) {
            const float *xb = a.x + (long long)b * p.H * p.W * a.x_ps + c;
            for (int i2 = 0; i2 < kh_n; i2++) {
                const int h = h0 + i2;
                if ((unsigned)h >= (unsigned)p.H) continue;
                for (int j = 0; j < kw_n; j++) {
                    const int ww = w0 + j;
                    if ((unsigned)ww >= (unsigned)p.W) continue;
                    add_tap(load_channels<V>(xb + (long long)(h * p.W + ww) * a.x_ps), i2 * kw_n + j);
                }
            }
        }
        apply_activation(acc.v, p.act);
        store_channels<V>(a.y + (long long)pixel * a.y_ps + c, acc, p.OC - c);
    }
}

__device__ __forceinline__ void dwconv_dispatch(const DirectConvArgs &a, int block, int num_blocks, unsigned threads) {
    const ConvProblem &p = a.p;
    if (a.nmore > 0) {   // the host only builds such launches for 3 x 3 and 5 x 5 windows
        if (p.KH == 3) {
            if (a.channels == 2) dwconv_body<3, 3, 2, true>(a, block, num_blocks, threads);
            else dwconv_body<3, 3, 1, true>(a, block, num_blocks, threads);
        } else {
            dwconv_body<5, 5, 1, true>(a, block, num_blocks, threads);
        }
        return;
    }
    if (a.channels == 4) {
        if (p.KH == 3 && p.KW == 3) dwconv_body<3, 3, 4>(a, block, num_blocks, threads);
        else if (p.KH == 5 && p.KW == 5) dwconv_body<5, 5, 4>(a, block, num_blocks, threads);
        else if (p.KH == 7 && p.KW == 7) dwconv_body<7, 7, 4>(a, block, num_blocks, threads);
        else dwconv_body<0, 0, 4>(a, block, num_blocks, threads);
        return;
    }
    if (p.KH == 3 && p.KW == 3) dwconv_body<3, 3, 1>(a, block, num_blocks, threads);
    else if (p.KH == 5 && p.KW == 5) dwconv_body<5, 5, 1>(a, block, num_blocks, threads);
    else if (p.KH == 7 && p.KW == 7) dwconv_body<7, 7, 1>(a, block, num_blocks, threads);
    else dwconv_body<0, 0, 1>(a, block, num_blocks, threads);
}

// 3 x 3 convolution of a 3-channel image: the first layer of a network at large batches, bound by the bytes of its output.  A
// block takes 4 * 32 consecutive output pixels and kThinConvChannels output channels; a wavefront multiplies its 32 pixels (rows)
// with 32 channels (columns) by 32 x 32 x 2 fp32 MFMAs, the two k of an instruction being one input channel of two taps, so that a
// lane's operands are whole pixels: five 16-byte loads, the next pixels' in flight.  An accumulator register then holds 32
// channels of two pixels, and a store writes two whole 128-byte lines.  (As vector arithmetic, a thread per pixel with filters
// read from LDS, the same layer takes 94 us at 64 images of 299 x 299, 32 channels: 62 us of LDS reads alone; in this form 60 us, 250 MB.)
constexpr int kThinConvChannels = 32, kThinConvPixels = 128;
typedef float thin_floatx16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ void conv_thin_body(const DirectConvArgs &a, int block, int num_blocks) {
    const ConvProblem &p = a.p;
    const unsigned npix = (unsigned)(p.OH * p.OW) * (unsigned)p.B;
    const unsigned pix_blocks = (npix + kThinConvPixels - 1) / kThinConvPixels;
    const int lane = (int)(threadIdx.x & 63), lk = lane >> 5, lc = lane & 31;
    const unsigned first = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * 32u;   // of the wavefront's pixels
    // taps 2 s + lk of the lane's pixel; the tenth tap does not exist
    auto request = [&](unsigned pb, Channels<4>(&v)[5]) {
        const unsigned n = min(pb * kThinConvPixels + first + (unsigned)lc, npix - 1);
        const unsigned line = fast_div(n, a.div_ow);
        const int ow = (int)(n - line * (unsigned)p.OW);
        const unsigned b = fast_div(line, a.div_oh);
        const int oh = (int)(line - b * (unsigned)p.OH);
        const int h0 = oh * p.sh - p.ph, w0 = ow * p.sw - p.pw;
        const float *xb = a.x + (long long)b * p.H * p.W * a.x_ps;
#pragma unroll
        for (int s = 0; s < 5; s++) {
            const int t = 2 * s + lk, i = t / 3, h = h0 + i, w = w0 + t - 3 * i;
            const bool inside = t < 9 && (unsigned)h < (unsigned)p.H && (unsigned)w < (unsigned)p.W;
            v[s] = load_channels<4>(xb + (inside ? (h * p.W + w) * a.x_ps : 0));   // (no branch: where paths with loads join, all of them are waited for)
#pragma unroll
            for (int c = 0; c < 3; c++) v[s].v[c] = inside ? v[s].v[c] : 0.f;
        }
    };
    for (int oc0 = 0; oc0 < p.OC; oc0 += kThinConvChannels) {
        const int oc = oc0 + lc;
        float filter[5][3];
#pragma unroll
        for (int s = 0; s < 5; s++)
#pragma unroll
            for (int c = 0; c < 3; c++) filter[s][c] = 2 * s + lk < 9 && oc < p.OC ? a.w[(size_t)oc * 27 + c * 9 + 2 * s + lk] : 0.f;
        const float bias = oc < p.OC ? a.bias[oc] : 0.f;
        Channels<4> now[5];
        request(min((unsigned)block, pix_blocks - 1), now);
        for (unsigned pb = (unsigned)block; pb < pix_blocks; pb += (unsigned)num_blocks) {
            Channels<4> next[5];
            request(min(pb + (unsigned)num_blocks, pix_blocks - 1), next);
            thin_floatx16 acc;
#pragma unroll
            for (int k = 0; k < 16; k++) acc[k] = bias;
#pragma unroll
            for (int s = 0; s < 5; s++)
#pragma unroll
                for (int c = 0; c < 3; c++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(p.pre_relu ? fmaxf(now[s].v[c], 0.f) : now[s].v[c], filter[s][c], acc, 0, 0, 0);
            float out[16];
#pragma unroll
            for (int k = 0; k < 16; k++) out[k] = acc[k];
            apply_activation(out, p.act);
            const unsigned n0 = pb * kThinConvPixels + first + 4u * (unsigned)lk;
            float *y = a.y + (long long)n0 * a.y_ps + oc;
            if (oc < p.OC) {
#pragma unroll
                for (int k = 0; k < 16; k++) {
                    const int row = 8 * (k >> 2) + (k & 3);
                    if (n0 + row < npix) y[row * a.y_ps] = out[k];
                }
            }
#pragma unroll
            for (int s = 0; s < 5; s++) now[s] = next[s];
        }
    }
}

__device__ __forceinline__ void conv_direct_body(const DirectConvArgs &a, int block, int num_blocks, unsigned threads) {
    const ConvProblem &p = a.p;
    const int icg = p.IC / p.groups, ocg = p.OC / p.groups;
    const long long total = (long long)p.B * p.OH * p.OW * p.OC;
    for (long long i = block * (long long)threads + threadIdx.x; i < total; i += (long long)num_blocks * threads) {
        const int pixel = (int)(i / p.OC);
        const int oc = (int)(i - (long long)pixel * p.OC);
        const int line = pixel / p.OW, ow = pixel - line * p.OW;
        const int b = line / p.OH, oh = line - b * p.OH;
        const int g = oc / ocg;
        const float *xg = a.x + (long long)b * p.H * p.W * a.x_ps + (long long)g * icg;
        const float *wo = a.w + (size_t)oc * icg * p.KH * p.KW;
        const int h0 = oh * p.sh - p.ph, w0 = ow * p.sw - p.pw;
        float acc = a.bias[oc];
        for (int c = 0; c < icg; c++)
            for (int i2 = 0; i2 < p.KH; i2++) {
                const int h = h0 + i2;
                if ((unsigned)h >= (unsigned)p.H) continue;
                for (int j = 0; j < p.KW; j++) {
                    const int ww = w0 + j;
                    if ((unsigned)ww >= (unsigned)p.W) continue;
                    float v = xg[(long long)(h * p.W + ww) * a.x_ps + c];
                    if (p.pre_relu) v = fmaxf(v, 0.f);
                    acc = fmaf(v, wo[(c * p.KH + i2) * p.KW + j], acc);
                }
            }
        float out[1] = {acc};
        apply_activation(out, p.act);
        a.y[(long long)pixel * a.y_ps + oc] = out[0];
    }
}

struct NaryKernelArgs {
    NaryArgs in;
    float *y;
    // units of V channels: `row` of them in a pixel (or, where all views are dense, one row of everything)
    unsigned total, row;
    FastDiv div_row;
    int C, y_ps;
    int multiply, accumulate, act, vec;
};

template <int V>
__device__ __forceinline__ void nary_body(const NaryKernelArgs &k, int block, int num_blocks, unsigned threads) {
    const NaryArgs &a = k.in;
    for (unsigned i = block * threads + threadIdx.x; i < k.total; i += num_blocks * threads) {
        const unsigned pixel = fast_div(i, k.div_row);
        const int c = (int)((i - pixel * k.row) * V);
        Channels<V> r;
        float *dst = k.y + (long long)pixel * k.y_ps + c;
        int first = 0;
        if (k.accumulate) {
            r = load_channels<V>(dst);
        } else {
            r = load_channels<V>(a.src[0] + (long long)pixel * a.src_pstride[0] + c);
            first = 1;
        }
        for (int j = first; j < a.count; j++) {
            const Channels<V> t = load_channels<V>(a.src[j] + (long long)pixel * a.src_pstride[j] + c);
#pragma unroll
            for (int e = 0; e < V; e++) r.v[e] = k.multiply ? r.v[e] * t.v[e] : r.v[e] + t.v[e];
        }
        apply_activation(r.v, k.act);
        store_channels<V>(dst, r, k.C - c);
    }
}

__device__ __forceinline__ void nary_dispatch(const NaryKernelArgs &k, int block, int num_blocks, unsigned threads) {
    if (k.vec == 4) nary_body<4>(k, block, num_blocks, threads);
    else nary_body<1>(k, block, num_blocks, threads);
}

}  // namespace ios
