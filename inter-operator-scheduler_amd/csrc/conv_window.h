// Convolutions of stride 1 with several taps at large batches, on a window of the input that is staged once: ConvWindow.
//
// The LDS-tiled kernels of conv_body.h and conv_pipe.h walk K tap by tap: for a 3 x 3 filter they load, convert (into two terms of
// half, some 40 instructions per eight values) and store every input value nine times.  At stride 1 the pixels that the BN
// outputs of a block read lie in one run of the input, BN plus the rows the filter reaches over: 200 pixels for 128 outputs of a
// 3 x 3 filter on 35 x 35 maps.  Here K is walked in chunks of 16 channels with all taps inside, and the run is staged once per
// chunk; a tap is a constant shift of the LDS address, and a lane whose tap falls outside the image reads a slot of zeros (a bit
// per tap, known from the start).  Filters are operands straight from memory, one unit (16 k of one tap) ahead in registers, so
// the only barriers are those around the staging.
//
// What is left per unit is matrix work, TNW LDS reads per plane and three address instructions per 32 pixels (two terms: four
// more for the scaled filter operand).  Measured at batch 64, fp32 as three terms of bfloat16 (six products) -> two of half (three):
// 80 -> 192 channels 3 x 3 on 73 x 73 463 -> 306 us (308 TFLOP/s, 924 of half products), 32 -> 64 on 147 x 147 317 -> 233 us, 32 -> 32 on
// 149 x 149 203 -> 155 us, 48 -> 64 5 x 5 on 35 x 35 66 -> 48 us, 192 -> 192 1 x 7 on 17 x 17 55 -> 36 us.  In bfloat16, tap by tap -> on the window, the same layers in a pass: 225 -> 182 us, 216 -> 206
// (bound by 530 MB of activations), 158 -> 130.
#pragma once

#include "conv_pipe.h"

namespace ios {

// TMW x TNW MFMA tiles per wavefront, WM x WN wavefronts per block; P_IT: rounds of T / 2 pixels in which a block stages its window;
// NBUF: windows in LDS (2: one barrier per chunk, for tiles whose windows are small)
// TAPS: number of taps where it is known, 0 otherwise
template <int TERMS, bool HALF, int TMW, int TNW, int WM, int WN, int P_IT, int NBUF, int TAPS = 0>
struct ConvWindow {
    static_assert(TERMS == 1 || (TERMS == 2 && HALF), "one rounded term, or two terms of half");
    static constexpr int MT = 32;
    using M = Mfma<32>;
    static constexpr int BM = 32 * TMW * WM, BN = 32 * TNW * WN;
    static constexpr int T = 64 * WM * WN;
    static constexpr int THREADS = T;
    static constexpr int CPAD = 16;
    static constexpr bool FUSABLE = false;
    static constexpr int WAVES_PER_SIMD = TERMS == 1 ? 1 : TMW * TNW >= 3 ? 2 : TAPS > 0 || TNW == 2 ? 3 : 4;
    static constexpr int kTouches = 4;                 // lines of 128 bytes of the filters a thread requests at the start
    static constexpr int SPAN = P_IT * (T / 2);       // pixels of the input a block holds
    // slots of 16 bytes per plane and octet (eight consecutive channels), the last one zero; the octets of a pixel, which
    // neighbouring lanes store, fall into different banks
    static constexpr int S = SPAN + 4;
    static constexpr int BUF = 2 * TERMS * S;
    static constexpr int WORDS = std::max(NBUF * BUF * 4, WM * WN * tail_floats(TMW, TNW));
    static constexpr int SMEM_FLOATS = WORDS + (TERMS == 2 ? WM * WN : 0);   // (two terms: a word per wavefront)

    // Two terms: one limit for all pixels of the block (an output reads many of them), by the values of its first window.  Where that does
    // not serve all of them, the tile is computed again.  The code is there twice: a limit that changes inside the K loop costs it 30 to
    // 60 registers, a loop around it as many, for addresses and masks that are held for the second time.
    template <bool RES = false>
    __device__ static __forceinline__ void run(const ConvKernelArgs &a, float *smem, int tile, int g, int z) {
        // Inputs that need neither a ReLU nor channels masked: a test a round, and the copies that its two ways out take, cost as much as the
        // conversion (192 -> 192 1 x 7 on 17 x 17 at batch 64 in bfloat16: 290 cycles a round, 24.8 -> 21.1 us).  Not for two terms in windows of
        // two rounds, whose code comes out slower that way (160 -> 160 1 x 7 32.0 -> 34.1 us).
        constexpr bool KNOWN = TAPS > 0 && (TERMS == 1 || NBUF == 1);
        unsigned limit;
        if (KNOWN && a.pre_relu == 0 && (a.ICg & 3) == 0) limit = attempt<RES, true, KNOWN>(a, smem, tile, g, z, kNoLimit);
        else limit = attempt<RES, true, false>(a, smem, tile, g, z, kNoLimit);
        if (TERMS == 2 && __builtin_expect(limit != 0, 0)) attempt<RES, false, false>(a, smem, tile, g, z, limit);
    }

    // limit: kNoLimit for the first attempt.  Returns the limit for another one, or 0.
    template <bool RES, bool FIRST, bool PLAIN>
    __device__ static __forceinline__ unsigned attempt(const ConvKernelArgs &a, float *smem, int tile, int g, int z, unsigned limit) {
    constexpr int TM = TMW, TN = TNW, WTM = 32 * TMW, WTN = 32 * TNW;
    uintx4 *lds = reinterpret_cast<uintx4 *>(smem);
    int tid = threadIdx.x;
    if constexpr (TERMS == 2) asm volatile("" : "+v"(tid));   // (keeps the attempts from sharing what both derive from it)
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN;
    const int wm = wave / WN;
    const int lk = lane >> 5;
    const int lc = lane & 31;
    int tm, tn;
    xcd_tile(a, tile, tm, tn);
    const int m0 = tm * BM;
    int n0 = tn * BN, n_end = a.Npix;
    if (a.OH != a.H) {   // tiles of one image each (the host counts them so): the input pixels of two images do not follow each other
        const int per_image = (a.OHW + BN - 1) / BN;
        const int image = tn / per_image;
        n0 = image * a.OHW + (tn - image * per_image) * BN;
        n_end = (image + 1) * a.OHW;
    }
    const int taps = TAPS > 0 ? TAPS : a.Kq / a.ICgP;   // odd
    // K slice z of the grid: a range of chunks of 16 channels, all taps of each
    const int chunks_all = a.ICgP >> 4;
    const int per_slice = (chunks_all + a.split_k - 1) / a.split_k;
    const int ch_begin = z * per_slice, ch_end = min(chunks_all, ch_begin + per_slice);

    const __amdgpu_buffer_rsrc_t xr = buffer_of(a.x, a.x_bytes);
    // ---- filters: packed [g][k / 8][plane][OCgP] slots of 16 bytes, k = tap * ICgP + channel
    unsigned a_off[TM];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = m0 + wm * WTM + i * 32 + lc;
        a_off[i] = m < a.OCgP ? (((unsigned)g * ((unsigned)a.Kq >> 3) + (unsigned)lk) * TERMS * (unsigned)a.OCgP + (unsigned)m) * 16u : kOutOfRange;
    }
    const unsigned plane_bytes = (unsigned)a.OCgP * 16u;
    const unsigned tap_bytes = (unsigned)(a.ICgP >> 3) * TERMS * plane_bytes, chunk_bytes = 2u * TERMS * plane_bytes;

    // The filters of a pass fit no L2: what the block will read is requested at once, a word of every line, shared out over the
    // blocks of the XCD that read the same: the first kTouches * T lines for each of them, all of a tile's where enough of them share it (a tile of
    // 448 channels 3 x 3, two terms and 64 outputs has 8064; three blocks of 256 threads request 3072).  Requested two taps ahead only, each
    // of them waits for memory.  With filters that no cache
    // holds, bfloat16 at batch 64, 192 -> 192 1 x 7 on 17 x 17 took 25.7 us (20.6 with filters in the L2) and takes 20.2, 256 -> 256 3 x 3 on
    // 14 x 14 38.8 (26.8) -> 27.2, 448 -> 384 3 x 3 on 8 x 8 48.7 (32.3) -> 34.3; two terms at batch 7, 256 -> 256 38.5 -> 32.8.  It costs
    // 0.2 to 1 us where they are in the L2.
    unsigned touched[FIRST ? kTouches : 1];
    if constexpr (FIRST) {
        const int slot = tile >> 3;
        int share, mine;
        if (a.weights_major) {
            share = min(a.xcd_q, a.tile_div);
            mine = a.xcd_q <= a.tile_div ? slot : tn;
        } else {
            share = (int)fast_div((unsigned)a.xcd_q, a.div_tile);
            mine = (int)fast_div((unsigned)slot, a.div_tile);
        }
        constexpr int LINES = BM / 8;   // of 128 bytes, for eight consecutive k of a plane
        const int lines = a.split_k == 1 ? (a.Kq >> 3) * TERMS * LINES : 0, step = max(share, 1) * T;
        const __amdgpu_buffer_rsrc_t wr = buffer_of(a.wp, a.w_bytes);
        const unsigned base = (unsigned)g * ((unsigned)a.Kq >> 3) * TERMS * plane_bytes + (unsigned)m0 * 16u;
#pragma unroll
        for (int i = 0; i < kTouches; i++) {
            const int line = mine * T + tid + i * step;
            touched[i] = __builtin_amdgcn_raw_buffer_load_b32(wr, line < lines ? base + (unsigned)(line / LINES) * plane_bytes + (unsigned)(line % LINES) * 128u : kOutOfRange, 0, 0);
        }
    }

    // ---- window: first input pixel of the block: tap (0, 0) of output pixel n0
    auto input_of = [&](int n, int &oh, int &ow) {
        const int b = (int)fast_div((unsigned)n, a.div_ohw);
        const int r = n - b * a.OHW;
        oh = (int)fast_div((unsigned)r, a.div_ow);
        ow = r - oh * a.OW;
        return (b * a.H + oh - a.ph) * a.W + ow - a.pw;
    };
    int oh_, ow_;
    const int p0 = input_of(n0, oh_, ow_);
    // pixels from the first to the last that the block's outputs read: what lies behind, in the rounds of T / 2, is neither loaded nor
    // converted (a wavefront stages 32 neighbouring pixels a round)
    const int span = input_of(min(n0 + BN, n_end) - 1, oh_, ow_) - p0 + (taps / a.KW - 1) * a.W + a.KW;
    auto needed = [&](int i) { return wave * 32 + i * (T / 2) < span; };
    const int half = tid & 1;
    unsigned x_off = (unsigned)((p0 + (tid >> 1)) * a.x_ps + g * a.ICg + 8 * half) * 4u;   // may wrap below zero: beyond the extent
    const unsigned x_step = (unsigned)(T / 2) * (unsigned)a.x_ps * 4u;
    floatx4 b_reg[P_IT][2];
    int b_left;   // real channels of this thread's octet
    auto load_window = [&](int ch) {
        const int c0 = ch * 16;
        b_left = a.ICg - c0 - 8 * half;
        const unsigned dead = ch < ch_end ? 0u : kOutOfRange;
        const unsigned pad0 = ((unsigned)(b_left - 1) & kOutOfRange) | dead, pad1 = ((unsigned)(b_left - 5) & kOutOfRange) | dead;
#pragma unroll
        for (int i = 0; i < P_IT; i++) {
            const unsigned at = (x_off + (unsigned)c0 * 4u + (unsigned)i * x_step) | (needed(i) ? 0u : kOutOfRange);
            b_reg[i][0] = buffer_load_f32x4(xr, at | pad0);
            b_reg[i][1] = buffer_load_f32x4(xr, at | pad1, 16u);
        }
    };
    const bool ragged = (a.ICg & 3) != 0;
    InputWatch watch;   // two terms
    unsigned *words = reinterpret_cast<unsigned *>(smem) + WORDS;
    auto octet_of = [&](int i, float (&v)[8]) {   // of the window in registers
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = b_reg[i][j >> 2][j & 3];
        if (a.pre_relu != 0)
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = relu_above(0.f, v[j]);
        if (ragged)
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = j < b_left ? v[j] : 0.f;
    };
    auto store_window = [&](int buf) {
        uintx4 *at = lds + buf * BUF + half * S + (tid >> 1);
        const float scale = limit_scale(limit);
#pragma unroll
        for (int i = 0; i < P_IT; i++) {
            if (!needed(i)) break;
            float v[8];
            if constexpr (PLAIN) {
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = b_reg[i][j >> 2][j & 3];
            } else {
                octet_of(i, v);
            }
            if constexpr (TERMS == 2) {
                uintx4 hi, lo;
                watch.octet(octet_peak(v), limit);
                split_half2(v, scale, hi, lo);
                at[i * (T / 2)] = hi;
                at[i * (T / 2) + 2 * S] = lo;
            } else if constexpr (HALF) {
                const floatx8 f = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
                at[i * (T / 2)] = __builtin_bit_cast(uintx4, __builtin_convertvector(f, halfx8));
            } else {
                at[i * (T / 2)] = round_bf16x8(v);
            }
        }
    };
    // this lane's outputs: place of tap (0, 0) in the patch, and the taps that fall inside the image
    unsigned at0[TN], inside[TN];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const int n = n0 + wn * WTN + j * 32 + lc;
        int oh, ow;
        const int first = input_of(n < n_end ? n : n0, oh, ow);
        at0[j] = (unsigned)((first - p0) * 16 + lk * S * 16);
        unsigned mask = 0;
        int kh = 0, kw = 0;
        for (int t = 0; t < taps; t++) {
            const bool ok = n < n_end && (unsigned)(oh - a.ph + kh) < (unsigned)a.H && (unsigned)(ow - a.pw + kw) < (unsigned)a.W;
            mask |= (ok ? 1u : 0u) << t;
            const bool wrap = ++kw == a.KW;
            kw = wrap ? 0 : kw;
            kh += wrap ? 1 : 0;
        }
        inside[j] = mask;
    }
    if (tid < NBUF * TERMS) lds[(tid / TERMS) * BUF + (tid % TERMS) * 2 * S + S - 1] = uintx4{0, 0, 0, 0};
    constexpr unsigned kZero = (S - 1) * 16;

    typename M::acc_t acc[TM][TN];
    auto begin = [&] {   // behind the request for the first window
        if constexpr (TERMS == 2) {
            if constexpr (!FIRST) return;
            float most = 0.f;
#pragma unroll
            for (int i = 0; i < P_IT; i++) {
                float v[8];
                octet_of(i, v);
                most = needed(i) ? fmaxf(most, octet_peak(v)) : most;
            }
            limit = first_limit<WM * WN>(most, words);
        }
    };
    auto touches_end = [&] {
        if constexpr (FIRST)
#pragma unroll
            for (int i = 0; i < kTouches; i++) asm volatile("" ::"v"(touched[i]));
    };
    uintx4 av[2][TERMS][TM];
    // next filter operands to request
    int r_tap = 0, r_ch = ch_begin;
    unsigned r_at = (unsigned)ch_begin * chunk_bytes;
    auto load_filters = [&](uintx4 (&v)[TERMS][TM]) {
        const __amdgpu_buffer_rsrc_t wr = buffer_of(a.wp, r_ch < ch_end ? a.w_bytes : 0u);
#pragma unroll
        for (int p = 0; p < TERMS; p++)
#pragma unroll
            for (int i = 0; i < TM; i++) v[p][i] = __builtin_amdgcn_raw_buffer_load_b128(wr, a_off[i], r_at + (unsigned)p * plane_bytes, 0);
        const bool wrap = ++r_tap == taps;
        r_tap = wrap ? 0 : r_tap;
        r_ch += wrap ? 1 : 0;
        r_at = wrap ? (unsigned)r_ch * chunk_bytes : r_at + tap_bytes;
    };
    // With the number of taps known, the places of a lane's operands are computed once, and a unit is its loads, its LDS reads and its
    // matrix work; otherwise address arithmetic takes as long as half of that (192 -> 192 1 x 7 on 17 x 17 at batch 64: 2.6 us a chunk, 0.8 of
    // them with neither loads nor matrix work).  That layer with 64 x 256 outputs per block 40.0 -> 36.4 us with what follows, 96 -> 96 3 x 3 on
    // 35 x 35 (32 x 256) 52.8 -> 49.0, 80 -> 192 on 73 x 73 304 -> 289.
    unsigned place[TAPS > 0 ? TAPS : 1][TN];
    if constexpr (TAPS > 0) {
        int shift = 0, kw = 0;
#pragma unroll
        for (int t = 0; t < TAPS; t++) {
#pragma unroll
            for (int j = 0; j < TN; j++) place[t][j] = (inside[j] >> t & 1u) != 0 ? at0[j] + (unsigned)shift : kZero;
            const bool wrap = ++kw == a.KW;
            shift += wrap ? (a.W - a.KW + 1) * 16 : 16;
            kw = wrap ? 0 : kw;
        }
    }
    auto filters_at = [&](uintx4 (&v)[TERMS][TM], unsigned at, bool live) {
        const __amdgpu_buffer_rsrc_t wr = buffer_of(a.wp, live ? a.w_bytes : 0u);
#pragma unroll
        for (int p = 0; p < TERMS; p++)
#pragma unroll
            for (int i = 0; i < TM; i++) v[p][i] = __builtin_amdgcn_raw_buffer_load_b128(wr, a_off[i], (live ? at : 0u) + (unsigned)p * plane_bytes, 0);
    };
    // Filters are requested two taps ahead and the next window behind the third tap's: loads return in order, so whoever waits for filters
    // requested behind a window waits for the window.  SETS sets of registers take turns, tap t in set t % SETS; the first two taps of the
    // next chunk find sets 0 and 1 free.  (With the filters of a chunk in LDS, staged like the window, no wait is left inside a chunk, and it
    // was no faster: 36.4 against 35.4 us on the first of these layers.)
    constexpr int SETS = TAPS % 3 == 0 ? 3 : TAPS % 4 == 3 ? 4 : 5;
    static_assert(TAPS == 0 || (TAPS % SETS == 0) || (TAPS % SETS == SETS - 1), "the last taps leave the first sets alone");
    uintx4 fv[TAPS > 0 ? SETS : 1][TERMS][TM];
    auto known_chunk = [&](int ch, auto buffer) {
        constexpr int B = decltype(buffer)::value;
        store_window(B);
        __syncthreads();
        const char *buf = reinterpret_cast<const char *>(smem) + B * BUF * 16;
        const unsigned at = (unsigned)ch * chunk_bytes;
#pragma unroll
        for (int t = 0; t < TAPS; t++) {
            uintx4 bv[TERMS][TN];
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < TERMS; q++) bv[q][j] = reinterpret_cast<const uintx4 *>(buf + place[t][j])[q * 2 * S];
            if (t + 2 < TAPS) filters_at(fv[(t + 2) % SETS], at + (unsigned)(t + 2) * tap_bytes, true);
            else filters_at(fv[t + 2 - TAPS], at + chunk_bytes + (unsigned)(t + 2 - TAPS) * tap_bytes, ch + 1 < ch_end);
            if (t == 0) load_window(ch + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply_terms<TERMS, HALF>(acc, fv[t % SETS], bv);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (NBUF == 1) __syncthreads();
    };
    // tap of the unit at hand, its offset in the patch in bytes
    int u_tap = 0, u_kw = 0, u_shift = 0;
    auto unit = [&](const char *buf, const uintx4 (&fv)[TERMS][TM], uintx4 (&next)[TERMS][TM]) {
        uintx4 bv[TERMS][TN];
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const unsigned valid = (unsigned)((int)(inside[j] << (31 - u_tap)) >> 31);
            const unsigned at = ((at0[j] + (unsigned)u_shift) & valid) | (kZero & ~valid);
            const uintx4 *p = reinterpret_cast<const uintx4 *>(buf + at);
#pragma unroll
            for (int q = 0; q < TERMS; q++) bv[q][j] = p[q * 2 * S];
        }
        load_filters(next);
        const bool wrap = ++u_kw == a.KW;
        u_shift += wrap ? (a.W - a.KW + 1) * 16 : 16;
        u_kw = wrap ? 0 : u_kw;
        u_tap++;
        __builtin_amdgcn_sched_barrier(0);
        multiply_terms<TERMS, HALF>(acc, fv, bv);
        __builtin_amdgcn_sched_barrier(0);
    };
    // One chunk: its window from registers into LDS, the next one requested, then one unit of matrix work per tap, each with the
    // filters of the next unit requested first.  (The first three units lie outside the loop: inside it every wait for filters
    // would also wait for the window requested in front of it.)  P: the filter registers the chunk starts with; the number of taps
    // is odd, so the next chunk starts with the other ones.
    const char *bytes = reinterpret_cast<const char *>(smem);
    auto chunk = [&](int ch, auto parity) {
        constexpr int P = decltype(parity)::value;
        const int b = NBUF == 2 ? (ch & 1) : 0;
        store_window(b);
        __syncthreads();
        load_window(ch + 1);
        u_tap = 0; u_kw = 0; u_shift = 0;
        const char *buf = bytes + b * BUF * 16;
        unit(buf, av[P], av[P ^ 1]);
        unit(buf, av[P ^ 1], av[P]);
        for (int t = 3; t < taps; t += 2) {
            unit(buf, av[P], av[P ^ 1]);
            unit(buf, av[P ^ 1], av[P]);
        }
        unit(buf, av[P], av[P ^ 1]);
        if (NBUF == 1) __syncthreads();
    };
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < M::ACC; v++) acc[i][j][v] = 0.f;
    if constexpr (TAPS > 0) {
        filters_at(fv[0], (unsigned)ch_begin * chunk_bytes, true);
        filters_at(fv[1], (unsigned)ch_begin * chunk_bytes + tap_bytes, true);
        load_window(ch_begin);
        begin();
        touches_end();
        for (int ch = ch_begin; ch < ch_end; ch += 2) {
            known_chunk(ch, std::integral_constant<int, 0>{});
            if (ch + 1 >= ch_end) break;
            known_chunk(ch + 1, std::integral_constant<int, NBUF - 1>{});
        }
    } else {
        load_filters(av[0]);
        load_window(ch_begin);
        begin();
        touches_end();
        for (int ch = ch_begin; ch < ch_end; ch += 2) {
            chunk(ch, std::integral_constant<int, 0>{});
            if (ch + 1 >= ch_end) break;
            chunk(ch + 1, std::integral_constant<int, 1>{});
        }
    }
    TailConstants<TM> constants;
    tail_constants<MT, TERMS == 2>(a, constants, g, m0 + wm * WTM);
    bool scaled = false;
    if constexpr (TERMS == 2) {
        const unsigned state = block_or<WM * WN>((__ballot(watch.peak >= __uint_as_float(limit)) != 0 ? 1u : 0u) | (watch.below != 0 ? 2u : 0u), words);
        if (__builtin_expect((state & 1u) != 0 && limit != kMostLimit, 0)) return limit_for(block_peak<WM * WN>(watch.peak, words));
        InputRange<TN> in;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            in.limit[j] = limit;
            in.wild[j] = limit == kMostLimit;
        }
        in.octets = __builtin_expect(state != 0, 0) ? block_sum<WM * WN>(watch.below, words) : 0u;
        unscale_inputs(acc, in.limit);
        scaled = check_sums<MT>(a, acc, reinterpret_cast<floatx4 *>(smem + (wm * WN + wn) * tail_floats(TM, TN)), in, constants.least, g, m0 + wm * WTM, [&](int j) {
            const int n = n0 + wn * WTN + j * 32 + lc;
            return n < n_end ? n : -1;
        }, 0, a.Kq, ch_begin * 16, ch_end * 16);
    } else {
        __syncthreads();
    }
    tiled_tail<MT, BM, BN, TM, TN, WM, WN, RES, TERMS == 2>(a, smem, acc, tile, g, z, m0, n0, wm, wn, 0, constants, n_end, scaled);
    return 0;
    }   // attempt
};

// X(index, name, TMW, TNW, WM, WN, P_IT, NBUF).  A window of a 3 x 3 filter on wide maps takes 300 pixels beyond the outputs, so
// the tall-and-narrow blocks are for few channels on large maps; the 128-output blocks serve the smaller maps, those of eight and
// twelve wavefronts where there is a block or two for a compute unit.
#define IOS_WINDOW3_VARIANTS(X)                           \
    X(139, "x3_win_m64n256_w1x4", 2, 2, 1, 4, 5, 1)       \
    X(140, "x3_win_m64n128_w1x4_d", 2, 1, 1, 4, 2, 2)     \
    X(141, "x3_win_m32n256_w1x4", 1, 2, 1, 4, 5, 1)       \
    X(142, "x3_win_m96n128_w1x4_d", 3, 1, 1, 4, 2, 2)     \
    X(143, "x3_win_m64n128_w2x4_d", 1, 1, 2, 4, 1, 2)     \
    X(144, "x3_win_m64n256_w2x4", 1, 2, 2, 4, 3, 1)       \
    X(145, "x3_win_m96n128_w3x4_d", 1, 1, 3, 4, 1, 2)
#define IOS_WINDOW_BF16_VARIANTS(X)                      \
    X(146, "wb_win_m192n128_w2x2", 3, 2, 2, 2, 3, 1)     \
    X(147, "wb_win_m96n128_w1x4", 3, 1, 1, 4, 2, 1)      \
    X(148, "wb_win_m64n128_w1x4", 2, 1, 1, 4, 3, 1)      \
    X(149, "wb_win_m64n256_w1x4", 2, 2, 1, 4, 5, 1)      \
    X(150, "wb_win_m32n256_w1x4", 1, 2, 1, 4, 5, 1)
#define IOS_WINDOW_FP16_VARIANTS(X)                      \
    X(151, "wh_win_m192n128_w2x2", 3, 2, 2, 2, 3, 1)     \
    X(152, "wh_win_m96n128_w1x4", 3, 1, 1, 4, 2, 1)      \
    X(153, "wh_win_m64n128_w1x4", 2, 1, 1, 4, 3, 1)      \
    X(154, "wh_win_m64n256_w1x4", 2, 2, 1, 4, 5, 1)      \
    X(155, "wh_win_m32n256_w1x4", 1, 2, 1, 4, 5, 1)
// Rounds of a kernel for windows of at most three: loads of rounds that no output needs return zeros, but the L1 takes 16 cycles for each like
// for any other, and what a tap with one term waits for is the L1 (96 -> 96 3 x 3 on 35 x 35 at batch 64 52.2 -> 48.1 us, bfloat16 29.0 -> 27.2, with PLAIN).
constexpr int short_rounds(int rounds) { return std::min(rounds, 3); }
constexpr int kFirstWindowVariant = 139, kWindowVariants = 17, kNumConvVariants = 170;

// The window kernels in the order of the lists above: for any number of taps (conv_window.hip), for 7 and for 9 (conv_window7.hip,
// conv_window9.hip), the latter two also with windows of three rounds
extern const KernelPair kWindowKernels[], kWindow7Kernels[], kWindow9Kernels[], kWindow7ShortKernels[], kWindow9ShortKernels[];

}  // namespace ios
