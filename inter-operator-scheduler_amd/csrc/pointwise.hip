// Stand-alone memory-bound kernels and their launchers.  Device code: pointwise_body.h.
#include "pointwise_body.h"

#include <algorithm>
#include <stdexcept>

#include "launch_internal.h"

namespace ios {

__global__ void pool_kernel(PoolArgs a) { pool_body(a, blockIdx.x, gridDim.x, blockDim.x); }
__global__ void global_pool_kernel(PoolArgs a) { global_pool_body(a, blockIdx.x, gridDim.x, blockDim.x); }
__global__ void dwconv_kernel(DirectConvArgs a) { dwconv_dispatch(a, blockIdx.x, gridDim.x, blockDim.x); }
__global__ void conv_direct_kernel(DirectConvArgs a) { conv_direct_body(a, blockIdx.x, gridDim.x, blockDim.x); }
__global__ __launch_bounds__(256) void conv_thin_kernel(DirectConvArgs a) {
    conv_thin_body(a, blockIdx.x, gridDim.x);
}
__global__ void nary_kernel(NaryKernelArgs a) { nary_dispatch(a, blockIdx.x, gridDim.x, blockDim.x); }

static int blocks_for(long long n, int per_block, int cap) {
    return (int)std::max<long long>(1, std::min<long long>((n + per_block - 1) / per_block, cap));
}

// ---- argument builders (shared with the fused stage kernel) ---------------------------------------------------------
// Channels per thread: four where the device is full with a quarter of the threads (64 threads per compute unit), else one.
static int channels_per_thread(long long pixels, int C) { return pixels * ((C + 3) / 4) >= (1LL << 14) && C > 2 ? 4 : 1; }

PoolArgs make_pool_args(const PoolProblem &p, const TensorView &x, const TensorView &y, bool global, int *blocks, const float *bias, int act) {
    if (x.C != p.C || x.H != p.H || x.W != p.W || y.C != p.C || y.H != p.OH || y.W != p.OW)
        throw std::runtime_error("pool: tensor views do not match the problem");
    if (global && (p.KH != p.H || p.KW != p.W || p.OH != 1 || p.OW != 1))
        throw std::runtime_error("global pool: window must be the whole map");
    if ((long long)p.B * p.C * p.OH * p.OW >= (1LL << 31)) throw std::runtime_error("pool: tensor too large for 32-bit indexing");
    PoolArgs a;
    a.x = x.ptr;
    a.y = y.ptr;
    a.x_ps = x.pstride;
    a.y_ps = y.pstride;
    a.p = p;
    a.strip_rows = 0;
    a.bias = bias;
    a.act = act;
    const long long pixels = (long long)p.B * p.OH * p.OW;
    a.channels = channels_per_thread(pixels, p.C);
    int lines = p.OH;
    if (global) {
        *blocks = blocks_for((long long)p.B * ((p.C + kGlobalPoolChannels - 1) / kGlobalPoolChannels), 4, 8192);
    } else {
        const int cv = (p.C + a.channels - 1) / a.channels;
        long long threads = pixels * cv;
        if (p.KH == 3 && p.KW == 3 && (p.sh == 1 || p.sh == 2)) {
            // one thread per strip of output rows; the longest strip that still leaves half a million threads
            int rows = p.sh == 1 ? kPoolStripRows : 2;
            auto strips = [&](int r) { return (long long)p.B * ((p.OH + r - 1) / r) * p.OW * cv; };
            while (rows > 1 && strips(rows) < (1LL << 19)) rows >>= 1;
            a.strip_rows = rows;
            threads = strips(rows);
            lines = (p.OH + rows - 1) / rows;
        }
        *blocks = blocks_for(threads, 256, 1 << 16);
    }
    a.div_cv = make_fast_div((unsigned)((p.C + a.channels - 1) / a.channels));
    a.div_ow = make_fast_div((unsigned)p.OW);
    a.div_strips = make_fast_div((unsigned)lines);
    return a;
}

DirectConvArgs make_direct_conv_args(const ConvProblem &p, const TensorView &x, const float *w, const float *bias,
                                     const TensorView &y, int *blocks, bool thin) {
    if (x.C != p.IC || x.H != p.H || x.W != p.W || y.C != p.OC || y.H != p.OH || y.W != p.OW)
        throw std::runtime_error("conv: tensor views do not match the problem");
    if ((long long)p.B * p.OC * p.OH * p.OW >= (1LL << 31)) throw std::runtime_error("conv: tensor too large for 32-bit indexing");
    DirectConvArgs a;
    a.x = x.ptr;
    a.w = w;
    a.bias = bias;
    a.y = y.ptr;
    a.x_ps = x.pstride;
    a.y_ps = y.pstride;
    a.p = p;
    const unsigned long long x_bytes = conv_input_extent(p, x.pstride);
    a.x_bytes = x_bytes < (1ull << 31) ? (unsigned)x_bytes : 0u;
    a.nmore = 0;
    for (int s = 0; s < kMaxNaryInputs - 1; s++) {
        a.more[s] = x.ptr;
        a.more_ps[s] = x.pstride;
        a.more_bytes[s] = 0;
    }
    const long long pixels = (long long)p.B * p.OH * p.OW;
    a.channels = p.is_depthwise() ? channels_per_thread(pixels, p.OC) : 1;
    a.div_cv = make_fast_div((unsigned)((p.OC + a.channels - 1) / a.channels));
    a.div_ow = make_fast_div((unsigned)p.OW);
    a.div_oh = make_fast_div((unsigned)p.OH);
    *blocks = blocks_for(pixels * ((p.OC + a.channels - 1) / a.channels), 256, 8192);
    if (thin) {
        if (!conv_thin_applies(p)) throw std::runtime_error("conv: the thin-input kernel serves 3 x 3 convolutions of 3-channel inputs");
        // up to eight blocks of four wavefronts per compute unit, each on several tiles of pixels
        *blocks = (int)std::min<long long>((pixels + kThinConvPixels - 1) / kThinConvPixels, 2048);
    }
    return a;
}

bool dwconv_sums_inputs(const ConvProblem &p) { return p.is_depthwise() && p.KH == p.KW && (p.KH == 3 || p.KH == 5); }

void add_dwconv_sources(DirectConvArgs &a, const TensorView *more, int count, int *blocks) {
    if (count < 0 || count > kMaxNaryInputs - 1) throw std::runtime_error("dwconv: too many summed inputs");
    const ConvProblem &p = a.p;
    if (count == 0) return;
    if (!dwconv_sums_inputs(p)) throw std::runtime_error("dwconv: this window does not add inputs in its loader");
    for (int s = 0; s < count; s++) {
        if (more[s].C != p.IC || more[s].H != p.H || more[s].W != p.W) throw std::runtime_error("dwconv: summed inputs of different shapes");
        const unsigned long long bytes = conv_input_extent(p, more[s].pstride);
        if (bytes >= (1ull << 31) || a.x_bytes == 0) throw std::runtime_error("dwconv: summed inputs beyond 31-bit offsets");
        a.more[s] = more[s].ptr;
        a.more_ps[s] = more[s].pstride;
        a.more_bytes[s] = (unsigned)bytes;
    }
    a.nmore = count;
    // the summing form holds whole windows of several inputs in registers: two channels per thread at most, for 3 x 3 windows
    a.channels = a.channels == 4 && p.KH == 3 ? 2 : 1;
    const int cv = (p.OC + a.channels - 1) / a.channels;
    a.div_cv = make_fast_div((unsigned)cv);
    *blocks = blocks_for((long long)p.B * p.OH * p.OW * cv, 256, 8192);
}

NaryKernelArgs make_nary_args(const NaryArgs &in, int multiply, int accumulate, int act, int B, const TensorView &y, int *blocks) {
    if (in.count < 1 || in.count > kMaxNaryInputs) throw std::runtime_error("nary: bad input count");
    const long long pixels = (long long)B * y.H * y.W;
    if (pixels * y.C >= (1LL << 31)) throw std::runtime_error("nary: tensor too large for 32-bit indexing");
    NaryKernelArgs a;
    a.in = in;
    a.y = y.ptr;
    a.y_ps = y.pstride;
    bool dense = y.pstride == y.C;
    for (int j = 0; j < in.count; j++) dense = dense && in.src_pstride[j] == y.C;
    const long long rows = dense ? 1 : pixels, length = dense ? pixels * y.C : y.C;
    a.vec = length >= 4 && rows * ((length + 3) / 4) >= (1LL << 14) ? 4 : 1;
    a.C = (int)length;
    a.row = (unsigned)((length + a.vec - 1) / a.vec);
    a.total = (unsigned)(rows * a.row);
    a.div_row = make_fast_div(a.row);
    a.multiply = multiply;
    a.accumulate = accumulate;
    a.act = act;
    *blocks = blocks_for(a.total, 256, 8192);
    return a;
}

// ---- launchers ---------------------------------------------------------------------------------------------------------
void launch_pool(const PoolProblem &p, const TensorView &x, const TensorView &y, hipStream_t stream, const float *bias, int act) {
    int blocks;
    const PoolArgs a = make_pool_args(p, x, y, false, &blocks, bias, act);
    hipLaunchKernelGGL(pool_kernel, dim3(blocks), dim3(256), 0, stream, a);
}

void launch_global_pool(const PoolProblem &p, const TensorView &x, const TensorView &y, hipStream_t stream) {
    int blocks;
    const PoolArgs a = make_pool_args(p, x, y, true, &blocks);
    hipLaunchKernelGGL(global_pool_kernel, dim3(blocks), dim3(256), 0, stream, a);
}

void launch_dwconv(const ConvProblem &p, const TensorView &x, const float *w, const float *bias, const TensorView &y,
                   hipStream_t stream, const TensorView *more, int nmore) {
    if (!p.is_depthwise()) throw std::runtime_error("dwconv: not a depth-wise problem");
    int blocks;
    DirectConvArgs a = make_direct_conv_args(p, x, w, bias, y, &blocks);
    add_dwconv_sources(a, more, nmore, &blocks);
    hipLaunchKernelGGL(dwconv_kernel, dim3(blocks), dim3(256), 0, stream, a);
}

void launch_conv_direct(const ConvProblem &p, const TensorView &x, const float *w, const float *bias, const TensorView &y,
                        hipStream_t stream, bool thin) {
    int blocks;
    const DirectConvArgs a = make_direct_conv_args(p, x, w, bias, y, &blocks, thin);
    if (thin) hipLaunchKernelGGL(conv_thin_kernel, dim3(blocks), dim3(256), 0, stream, a);
    else hipLaunchKernelGGL(conv_direct_kernel, dim3(blocks), dim3(256), 0, stream, a);
}

void launch_nary(const NaryArgs &in, int multiply, int accumulate, int act, int B, const TensorView &y, hipStream_t stream) {
    int blocks;
    const NaryKernelArgs a = make_nary_args(in, multiply, accumulate, act, B, y, &blocks);
    hipLaunchKernelGGL(nary_kernel, dim3(blocks), dim3(256), 0, stream, a);
}

void launch_unary(const TensorView &x, const TensorView &y, int act, int B, hipStream_t stream) {
    if (x.C != y.C || x.H != y.H || x.W != y.W) throw std::runtime_error("unary: shape mismatch");
    NaryArgs a;
    a.count = 1;
    a.src[0] = x.ptr;
    a.src_pstride[0] = x.pstride;
    launch_nary(a, 0, 0, act, B, y, stream);
}

// ---- depth-wise filters -------------------------------------------------------------------------------------------------
__global__ void pack_depthwise_kernel(const float *w, float *packed, int C, int padded, int taps) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < taps * padded; i += gridDim.x * blockDim.x) {
        const int tap = i / padded, c = i - tap * padded;
        packed[i] = c < C ? w[c * taps + tap] : 0.f;
    }
}

void launch_pack_depthwise(const ConvProblem &p, const float *w, float *packed, hipStream_t stream) {
    const int padded = (p.OC + 3) & ~3, taps = p.KH * p.KW;
    hipLaunchKernelGGL(pack_depthwise_kernel, dim3(blocks_for((long long)padded * taps, 256, 1024)), dim3(256), 0, stream, w, packed, p.OC, padded, taps);
}

// ---- from the host's layout to views -------------------------------------------------------------------------------------
// Bound by bytes (or by the link, where `nchw` lies in host memory).  Few channels (images): a thread takes a pixel, reads its
// channels from their planes, consecutive threads consecutive pixels, and writes one pixel.  Otherwise a block turns a tile of
// 32 channels x 240 pixels through LDS: a row of the tile is read from line to line, 64 lanes of 16 bytes, wherever it begins.
// Rows of 64 pixels at odd places straddle five lines instead of four, and no cache keeps host memory for the block that reads
// the rest: three images of 131 channels x 37 x 53 took 115 us until they were there and take 96 like this (3.1 MB; 54 is the
// link).  Up to four channels the planes' rows are long: whole lines through LDS gave nothing there (seven images of 299 x 299
// 209 us against 203, five of 224 x 224 93 against 87).
constexpr int kLine = 16;   // floats
constexpr int kTileRow = 240, kTileChannels = 32;

// Floats [at, at + 4) behind `line`, at a multiple of four; those outside [lead, total) are zero and not read.
__device__ __forceinline__ pw_floatx4 line_quad(const float *line, long long at, int lead, long long total) {
    if (at >= lead && at + 4 <= total) return *reinterpret_cast<const pw_floatx4 *>(line + at);
    pw_floatx4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (at + j >= lead && at + j < total) v[j] = line[at + j];
    return v;
}

// lead: floats from the last multiple of a line in memory to the first element; total: floats from there to behind the last
__global__ __launch_bounds__(256) void to_view_kernel(const float *nchw, float *view, int B, int C, int HW, long long plane, int ps, int lead, long long total) {
    if (C <= 4) {
        const long long pixels = (long long)B * HW;
        for (long long i = blockIdx.x * 256LL + threadIdx.x; i < pixels; i += gridDim.x * 256LL) {
            const long long b = i / HW, r = i - b * HW;
            const float *first = nchw + b * C * plane + r;
            float *pixel = view + i * ps;
            float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 4; c++)
                if (c < C) v[c] = first[c * plane];
            if (ps == 4) {
                const pw_floatx4 q = {v[0], v[1], v[2], v[3]};
                *reinterpret_cast<pw_floatx4_u *>(pixel) = q;
            } else {
#pragma unroll
                for (int c = 0; c < 4; c++)
                    if (c < C) pixel[c] = v[c];
            }
        }
        return;
    }
    const float *line = nchw - lead;   // (what lies in front of the first element is not read)
    constexpr int STRIDE = kTileRow + kLine + 4;
    __shared__ float rows[kTileChannels * STRIDE];
    const int tid = threadIdx.x;
    const int tiles_c = (C + kTileChannels - 1) / kTileChannels, tiles_p = (HW + kTileRow - 1) / kTileRow;
    const int lane = tid & 63, wave = tid >> 6;              // of the host's layout: four floats of a row, a channel of four
    const int cx = tid & 31, p8 = tid >> 5;                  // of the view: channel, pixel of eight
    for (long long t = blockIdx.x; t < (long long)B * tiles_c * tiles_p; t += gridDim.x) {
        const long long bt = t / tiles_p;
        const int p0 = (int)(t - bt * tiles_p) * kTileRow, pixels = min(kTileRow, HW - p0);
        const long long b = bt / tiles_c;
        const int c0 = (int)(bt - b * tiles_c) * kTileChannels;
        const long long first = lead + (b * C + c0) * plane + p0;
        pw_floatx4 v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int c = wave + 4 * i;
            const long long at = first + c * plane, from = at & ~(long long)(kLine - 1);
            v[i] = pw_floatx4{0.f, 0.f, 0.f, 0.f};
            if (c0 + c < C && 4 * lane < (int)(at - from) + pixels) v[i] = line_quad(line, from + 4 * lane, lead, total);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; i++) *reinterpret_cast<pw_floatx4 *>(rows + (wave + 4 * i) * STRIDE + 4 * lane) = v[i];
        __syncthreads();
        if (c0 + cx < C) {
            const float *row = rows + cx * STRIDE + (int)((first + cx * plane) & (kLine - 1));
            float *out = view + (b * HW + p0) * ps + c0 + cx;
            for (int p = p8; p < pixels; p += 8) out[(long long)p * ps] = row[p];
        }
    }
}

static int layout_blocks(int B, int C, int HW) {
    return C <= 4 ? blocks_for((long long)B * HW, 256, 1024)
                  : blocks_for((long long)B * ((C + kTileChannels - 1) / kTileChannels) * ((HW + kTileRow - 1) / kTileRow), 1, 2048);
}

void launch_to_view(const float *nchw, const TensorView &y, int B, hipStream_t stream, long long plane) {
    const int HW = y.H * y.W;
    const long long step = plane > 0 ? plane : HW;
    const int lead = (int)(reinterpret_cast<uintptr_t>(nchw) / sizeof(float) % kLine);
    const long long total = lead + ((long long)B * y.C - 1) * step + HW;
    hipLaunchKernelGGL(to_view_kernel, dim3(layout_blocks(B, y.C, HW)), dim3(256), 0, stream, nchw, y.ptr, B, y.C, HW, step, y.pstride, lead, total);
}

// ---- fills ---------------------------------------------------------------------------------------------------------
__global__ void fill_pattern_kernel(float *dst, size_t n, unsigned seed, float most) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        unsigned h = (unsigned)i * 2654435761u ^ seed;
        h ^= h >> 16;
        h *= 0x85ebca6bu;
        h ^= h >> 13;
        h *= 0xc2b2ae35u;
        h ^= h >> 16;
        dst[i] = ((float)(h >> 8) * (1.0f / 8388608.0f) - 1.0f) * most;
    }
}

__global__ void fill_u32_kernel(unsigned *dst, size_t n, unsigned value) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) dst[i] = value;
}

void launch_fill_pattern(float *dst, size_t n, unsigned seed, hipStream_t stream, float most) {
    if (n == 0) return;
    hipLaunchKernelGGL(fill_pattern_kernel, dim3(blocks_for((long long)n, 256, 65535)), dim3(256), 0, stream, dst, n, seed, most);
}

void launch_fill_u32(unsigned *dst, size_t n, unsigned value, hipStream_t stream) {
    if (n == 0) return;
    hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks_for((long long)n, 256, 65535)), dim3(256), 0, stream, dst, n, value);
}

// One wavefront that sleeps for about 4 us per step (8128 clocks at 2.1 to 2.4 GHz).
__global__ void delay_kernel(int steps) {
    for (int i = 0; i < steps; i++) __builtin_amdgcn_s_sleep(127);
}

void launch_delay(int steps, hipStream_t stream) { hipLaunchKernelGGL(delay_kernel, dim3(1), dim3(64), 0, stream, steps); }

}  // namespace ios
