// LDS-tiled convolution for large batches with both operands staged in LDS: ConvPipe.
//
// The GEMM view, K order and tails are those of conv_body.h; the operands are sixteen-bit ones: two terms of IEEE half that hold
// an fp32 value (TERMS = 2, fp32 accuracy, see split_half2) or one rounded term, bfloat16 or half (TERMS = 1, the
// reduced-precision modes), on v_mfma_f32_32x32x16.  ConvSplit3 reads its filters from global memory, once per wavefront: at 32 x 64
// outputs per wavefront the L1 delivers 64 bytes per cycle and compute unit for them alone, its limit.  Here a block reads its
// filter tile once, and a wavefront computes up to 64 x 64 or 96 x 32 outputs per operand read (with two terms 12 or 9 matrix
// instructions of 32 cycles for 8 LDS reads of 16 bytes per lane).
//
// A stage holds KU units of 16 k (a unit lies inside one filter tap).  One stage is two or more matrix times ahead in
// registers, the next one in LDS; one barrier per stage.  What a stage has to cover is the latency of its loads: with two terms one
// or two units do (12 matrix instructions of 32 cycles per wavefront and unit at 64 x 64), with one term it takes four (a one-unit
// stage is gone in 128 cycles).  Measured at batch 64 in fp32, three bfloat16 terms -> two terms of half: 288 -> 384 channels 3 x 3 stride 2 on
// 35 x 35 207 -> 149 us (247 TFLOP/s, with 64 x 64 per wavefront, two units), 768 -> 192 on 17 x 17 42 -> 34 us, 192 -> 64 on 35 x 35
// 20.7 -> 18.5 us (bound by its 80 MB).
#pragma once

#include "conv_body.h"

namespace ios {

// POINT: 1 x 1 filters without groups.  PLAIN: inputs that need neither a ReLU nor channels masked (pipe_plain).
template <int TERMS, bool HALF, int KU, int PD, int TMW, int TNW, int WM, int WN, bool POINT = false, bool PLAIN = false>
struct ConvPipe {
    static_assert(TERMS == 1 || (TERMS == 2 && HALF), "one rounded term, or two terms of half");
    static constexpr int MT = 32;
    using M = Mfma<32>;
    static constexpr int BM = 32 * TMW * WM, BN = 32 * TNW * WN, BK = 16 * KU;
    static constexpr int T = 64 * WM * WN;
    static constexpr int THREADS = T;
    static constexpr int CPAD = 16;
    static constexpr bool FUSABLE = false;
    // (stages of four units fill the LDS with two blocks: no fewer registers than three wavefronts leave, or the PLAIN form spills: 256 -> 256 3 x 3 on
    // 14 x 14 at batch 7 38.5 -> 33.0 us)
    static constexpr int WAVES_PER_SIMD = TERMS == 1 ? 1 : TMW * TNW >= 3 ? 2 : KU == 4 ? 3 : 4;
    static constexpr int OCT = 2 * KU;                 // octets (eight consecutive k) of a pixel or filter row in a stage
    static constexpr int B_IT = OCT * BN / T;          // pixels a thread stages, T / OCT apart
    static constexpr int A_SLOTS = OCT * TERMS * BM;   // slots of 16 bytes (eight 16-bit values)
    static constexpr int A_IT = (A_SLOTS + T - 1) / T;
    // inputs of one unit and plane: two slots per pixel; units are two slots out of step, so that the octets of a pixel, which
    // neighbouring lanes store, fall into different banks
    static constexpr int UNIT = 2 * BN + (KU > 1 ? 2 : 0);
    static constexpr int STAGE = A_SLOTS + KU * TERMS * UNIT;
    static constexpr int WORDS = std::max(2 * STAGE * 4, WM * WN * tail_floats(TMW, TNW));
    static constexpr int SMEM_FLOATS = WORDS + (TERMS == 2 ? WM * WN : 0);   // (two terms: a word per wavefront)
    static_assert(OCT * BN % T == 0 && T % OCT == 0, "input loader shape");

    // Two terms: one limit for the inputs of the tile, by those of its first stage.  Where that does not serve all of them, the tile is
    // computed again.  The code is there twice: as a loop the compiler holds addresses, masks and zeros for the second time, 40 to 100
    // registers.  The PLAIN form of the first attempt: what a tile with nothing beside it on its compute unit waits for is the sum of its
    // steps (768 -> 192 on 17 x 17, a block of 64 x 128, per 16 k: 230 cycles for the operands from LDS, 320 for the matrix instructions, 450 to
    // split an octet, 250 to store and for the barrier), and without the branches between them the split work lies under the matrix instructions.  That layer at batch 3 23.6 -> 21.7 us, at batch 64 31.8 -> 29.0; four such convolutions in a launch, 704 outputs,
    // batch 16 31.6 -> 29.2, batch 64 94.2 -> 92.2.  With one term the matrix work is a third of that and the two ways out of each test cost as much as the
    // conversion: passes of Inception-v3 in half at batch 7 660 -> 619 us, in bfloat16 at batch 64 2298 -> 2248.
    // A kernel holds one of the two forms: both in one take the registers of the larger for either (one term, 64 x 64 outputs, any filter 106
    // instead of 82, four wavefronts a SIMD instead of five).  Masked forms, both in one -> apart: 256 -> 256 3 x 3 behind a folded
    // ReLU on 14 x 14, half at batch 7, 26.1 -> 23.2 us; 768 -> 192 behind one on 17 x 17, bfloat16 at batch 64, 64 x 128 outputs 22.1 -> 20.9.
    template <bool RES = false>
    __device__ static __forceinline__ void run(const ConvKernelArgs &a, float *smem, int tile, int g, int z) {
        const unsigned limit = attempt<RES, true, PLAIN>(a, smem, tile, g, z, kNoLimit);
        if (TERMS == 2 && __builtin_expect(limit != 0, 0)) attempt<RES, false, false>(a, smem, tile, g, z, limit);
    }

    // limit: kNoLimit for the first attempt.  Returns the limit for another one, or 0.
    template <bool RES, bool FIRST, bool UNMASKED>
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
    const int n0 = tn * BN;
    const int k_begin = z * a.k_chunk;
    const int k_end = min(a.Kq, k_begin + a.k_chunk);
    const int stages = (k_end - k_begin + BK - 1) / BK;

    const __amdgpu_buffer_rsrc_t xr = buffer_of(a.x, a.x_bytes);
    const __amdgpu_buffer_rsrc_t wr = buffer_of(a.wp, a.w_bytes);
    // ---- filters: packed [g][k / 8][plane][OCgP] slots; slot s of a stage is (octet, plane, row) = (s / BM / TERMS, s / BM % TERMS, s % BM)
    unsigned a_off[A_IT];
    int a_oct[A_IT];
#pragma unroll
    for (int i = 0; i < A_IT; i++) {
        const int s = tid + i * T;
        const int row = s % BM, op = s / BM, m = m0 + row;
        a_oct[i] = op / TERMS;
        const bool ok = (A_SLOTS % T == 0 || s < A_SLOTS) && m < a.OCgP;
        a_off[i] = ok ? (((unsigned)g * ((unsigned)a.Kq >> 3) * TERMS + (unsigned)op) * (unsigned)a.OCgP + (unsigned)m) * 16u : kOutOfRange;
    }
    // ---- inputs: this thread's octet and pixels; the octets of a pixel go to neighbouring threads
    const int oct = tid % OCT;
    const int unit = KU == 1 ? 0 : oct >> 1;
    const int half = oct & 1;
    int ih0[B_IT], iw0[B_IT];
    unsigned x_off[B_IT], n_kill[B_IT];
#pragma unroll
    for (int i = 0; i < B_IT; i++) {
        const int n = n0 + tid / OCT + i * (T / OCT);
        n_kill[i] = n < a.Npix ? 0u : kOutOfRange;
        const int nn = n < a.Npix ? n : 0;
        const int b = (int)fast_div((unsigned)nn, a.div_ohw);
        const int r = nn - b * a.OHW;
        const int oh = (int)fast_div((unsigned)r, a.div_ow);
        const int ow = r - oh * a.OW;
        ih0[i] = oh * a.sh - a.ph;
        iw0[i] = ow * a.sw - a.pw;
        x_off[i] = (((unsigned)(b * a.H + ih0[i]) * (unsigned)a.W + (unsigned)iw0[i]) * (unsigned)a.x_ps + (unsigned)(g * a.ICg + 8 * half + (POINT ? 16 * unit : 0))) * 4u;
        if constexpr (POINT) x_off[i] |= n_kill[i] | ((unsigned)ih0[i] < (unsigned)a.H && (unsigned)iw0[i] < (unsigned)a.W ? 0u : kOutOfRange);
    }
    auto slot_of = [](int pixel, int octet) { return 2 * pixel + (octet ^ ((pixel >> 2) & 1)); };

    uintx4 a_reg[PD][A_IT];
    floatx4 b_reg[PD][B_IT][2];
    int b_left[PD];
    auto load_stage = [&](int st, uintx4 (&ar)[A_IT], floatx4 (&br)[B_IT][2], int &left) {
        const int k0 = k_begin + st * BK;
        if constexpr (POINT) {
            // Addresses stay, the descriptors move on to the stage and end where K does (stages past the end: at once).  Channels past the
            // end of a pixel's are masked by store_stage.
            const bool live = k0 < k_end;
            const unsigned w_stage = (unsigned)((k0 >> 3) * TERMS) * (unsigned)a.OCgP * 16u;
            const __amdgpu_buffer_rsrc_t xs = buffer_of(a.x + k0, live ? a.x_bytes - (unsigned)k0 * 4u : 0u);
            const __amdgpu_buffer_rsrc_t ws = buffer_of(a.wp + (w_stage >> 2), live ? a.w_bytes - w_stage : 0u);
#pragma unroll
            for (int i = 0; i < A_IT; i++) ar[i] = __builtin_amdgcn_raw_buffer_load_b128(ws, a_off[i], 0, 0);
#pragma unroll
            for (int i = 0; i < B_IT; i++) {
                br[i][0] = buffer_load_f32x4(xs, x_off[i]);
                br[i][1] = buffer_load_f32x4(xs, x_off[i], 16u);
            }
            left = a.ICg - k0;
            return;
        }
        const unsigned w_stage = (unsigned)((k0 >> 3) * TERMS) * (unsigned)a.OCgP * 16u;
#pragma unroll
        for (int i = 0; i < A_IT; i++) {
            const unsigned kill = k0 + 8 * a_oct[i] < k_end ? 0u : kOutOfRange;   // beyond the K range: zeros
            ar[i] = __builtin_amdgcn_raw_buffer_load_b128(wr, (a_off[i] + w_stage) | kill, 0, 0);
        }
        const int k = k0 + 16 * unit;
        const int tap = (int)__umulhi((unsigned)k, a.magic_icgp);
        const int c0 = k - tap * a.ICgP;
        const int kh = a.KW == 1 ? tap : (int)__umulhi((unsigned)tap, a.magic_kw);
        const int kw = tap - kh * a.KW;
        const unsigned dead = k < k_end ? 0u : kOutOfRange;
        const unsigned x_unit = (unsigned)((kh * a.W + kw) * a.x_ps + c0) * 4u;
        const int c_left = a.ICg - c0 - 8 * half;   // real channels from this octet on
        const unsigned pad0 = (unsigned)(c_left - 1) & kOutOfRange, pad1 = (unsigned)(c_left - 5) & kOutOfRange;   // sign bits
#pragma unroll
        for (int i = 0; i < B_IT; i++) {
            const unsigned in_h = (unsigned)(ih0[i] + kh) < (unsigned)a.H ? 1u : 0u;
            const unsigned in_w = (unsigned)(iw0[i] + kw) < (unsigned)a.W ? 1u : 0u;
            const unsigned at = (x_off[i] + x_unit) | (((in_h & in_w) ^ 1u) << 31) | n_kill[i] | dead;
            br[i][0] = buffer_load_f32x4(xr, at | pad0);
            br[i][1] = buffer_load_f32x4(xr, at | pad1, 16u);
        }
        left = c_left;
    };
    const bool ragged = (a.ICg & 3) != 0;
    InputWatch watch;   // two terms
    unsigned *words = reinterpret_cast<unsigned *>(smem) + WORDS;
    auto octet_of = [&](const floatx4 (&br)[2], int left, float (&v)[8]) {
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = br[j >> 2][j & 3];
        if (a.pre_relu != 0)
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = relu_above(0.f, v[j]);   // folded ReLU of the producer
        if (POINT ? left < BK : ragged) {
            const int mine = POINT ? left - 16 * unit - 8 * half : left;
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = j < mine ? v[j] : 0.f;
        }
    };
    auto store_filters = [&](int buf, const uintx4 (&ar)[A_IT]) {
        uintx4 *As = lds + buf * STAGE;
#pragma unroll
        for (int i = 0; i < A_IT; i++)
            if (A_SLOTS % T == 0 || tid + i * T < A_SLOTS) As[tid + i * T] = ar[i];
    };
    auto store_octet = [&](int buf, int i, const uintx4 &hi, const uintx4 &lo) {
        uintx4 *Bs = lds + buf * STAGE + A_SLOTS + unit * (TERMS * UNIT);
        const int slot = slot_of(tid / OCT + i * (T / OCT), half);
        Bs[slot] = hi;
        if constexpr (TERMS == 2) Bs[UNIT + slot] = lo;
    };
    auto convert = [&](const floatx4 (&br)[2], int left, uintx4 &hi, uintx4 &lo) {
        float v[8];
        if constexpr (UNMASKED) {
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = br[j >> 2][j & 3];
        } else {
            octet_of(br, left, v);
        }
        if constexpr (TERMS == 2) {
            watch.octet(octet_peak(v), limit);
            split_half2(v, limit_scale(limit), hi, lo);
        } else if constexpr (HALF) {
            const floatx8 f = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]};
            hi = __builtin_bit_cast(uintx4, __builtin_convertvector(f, halfx8));   // round to nearest even, overflow to infinity
        } else {
            hi = round_bf16x8(v);
        }
    };
    // (With tests between them octets are stored one by one: held until the last is converted, 161 -> 160 1 x 7 on 17 x 17 at batch 16 in
    // bfloat16, 64 x 128 outputs, takes 28.9 us instead of 24.2.)
    auto store_stage = [&](int buf, const uintx4 (&ar)[A_IT], const floatx4 (&br)[B_IT][2], int left) {
        uintx4 hi[UNMASKED ? B_IT : 1], lo[UNMASKED ? B_IT : 1];
        if constexpr (UNMASKED) {
#pragma unroll
            for (int i = 0; i < B_IT; i++) convert(br[i], left, hi[i], lo[i]);
        }
        store_filters(buf, ar);
#pragma unroll
        for (int i = 0; i < B_IT; i++) {
            if constexpr (!UNMASKED) convert(br[i], left, hi[0], lo[0]);
            store_octet(buf, i, hi[UNMASKED ? i : 0], lo[UNMASKED ? i : 0]);
        }
    };

    typename M::acc_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < M::ACC; v++) acc[i][j][v] = 0.f;

    // Register set s holds stage st with st % PD == s.  Iteration st: the matrix work of stage st from LDS buffer st & 1, the
    // registers of stage st + 1 into the other buffer, stage st + 1 + PD requested into the same registers.  The loop runs in
    // rounds of PD stages with a straight-line body; stages past the end are loaded as zeros.
#pragma unroll
    for (int s = 0; s < PD; s++) load_stage(s, a_reg[s], b_reg[s], b_left[s]);
    if constexpr (TERMS == 2) {
        if constexpr (FIRST) {
            float most = 0.f;
#pragma unroll
            for (int i = 0; i < B_IT; i++) {
                float v[8];
                octet_of(b_reg[0][i], b_left[0], v);
                most = fmaxf(most, octet_peak(v));
            }
            limit = first_limit<WM * WN>(most, words);
        }
    }
    store_stage(0, a_reg[0], b_reg[0], b_left[0]);
    load_stage(PD, a_reg[0], b_reg[0], b_left[0]);
    __syncthreads();
    // (otherwise the compiler waits for all loads in every round, for registers that hold loads only on the way in)
    if constexpr (UNMASKED) __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
    for (int st0 = 0; st0 < stages; st0 += PD) {
#pragma unroll
        for (int s = 0; s < PD; s++) {
            const int st = st0 + s;
            const int buf = st & 1;
            const uintx4 *Ab = lds + buf * STAGE + lk * (TERMS * BM) + wm * WTM + lc;
            const uintx4 *Bb = lds + buf * STAGE + A_SLOTS + slot_of(wn * WTN + lc, lk);   // (tiles are 32 pixels apart: the same exchange in all)
            // operands of the next unit are read ahead of a unit's matrix work, where registers allow it
            constexpr int TURN = UNMASKED && TERMS == 2 && KU > 1 && TMW * TNW != 2 ? 1 : 0;
            uintx4 av[TURN + 1][TERMS][TM], bv[TURN + 1][TERMS][TN];
            auto read_unit = [&](int u) {
#pragma unroll
                for (int p = 0; p < TERMS; p++) {
#pragma unroll
                    for (int i = 0; i < TM; i++) av[u & TURN][p][i] = Ab[(2 * u * TERMS + p) * BM + i * MT];
#pragma unroll
                    for (int j = 0; j < TN; j++) bv[u & TURN][p][j] = Bb[(u * TERMS + p) * UNIT + j * 2 * MT];
                }
            };
            const uintx4 (&ar)[A_IT] = a_reg[(s + 1) % PD];
            const floatx4 (&br)[B_IT][2] = b_reg[(s + 1) % PD];
            if constexpr (UNMASKED && TERMS == 2) {
                // The octets of the next stage are split between the matrix instructions of this one, a pair of values at a time.
                constexpr int SLOTS = 3 * TM * TN * KU, PIECES = 5 * B_IT;
                uintx4 hi[B_IT], lo[B_IT];
#pragma unroll
                for (int u = 0; u < KU; u++) {
                    if (TURN == 0 || u == 0) {
                        read_unit(u);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if (TURN == 1 && u + 1 < KU) read_unit(u + 1);
                    multiply_terms_between(acc, av[u & TURN], bv[u & TURN], [&](int n) {
                        const int slot = u * 3 * TM * TN + n;
#pragma unroll
                        for (int piece = slot * PIECES / SLOTS; piece < (slot + 1) * PIECES / SLOTS; piece++) {
                            const int i = piece / 5, q = piece % 5;
                            if (q < 4) {
                                unsigned h, l;
                                split_pair(br[i][q >> 1][2 * (q & 1)], br[i][q >> 1][2 * (q & 1) + 1], limit_scale(limit), h, l);
                                asm volatile("" : "+v"(h), "+v"(l));   // (here, and not where they are stored)
                                hi[i][q] = h;
                                lo[i][q] = l;
                            } else {
                                float v[8];
#pragma unroll
                                for (int j = 0; j < 8; j++) v[j] = br[i][j >> 2][j & 3];
                                watch.octet(octet_peak(v), limit);
                            }
                        }
                    });
                }
                store_filters(buf ^ 1, ar);
#pragma unroll
                for (int i = 0; i < B_IT; i++) store_octet(buf ^ 1, i, hi[i], lo[i]);
            } else {
#pragma unroll
                for (int u = 0; u < KU; u++) {
                    read_unit(u);
                    // all LDS reads of the unit are requested before its first matrix instruction
                    if (TERMS == 2) __builtin_amdgcn_sched_barrier(0);
                    multiply_terms<TERMS, HALF>(acc, av[0], bv[0]);
                }
                store_stage(buf ^ 1, ar, br, b_left[(s + 1) % PD]);
            }
            load_stage(st + 1 + PD, a_reg[(s + 1) % PD], b_reg[(s + 1) % PD], b_left[(s + 1) % PD]);
            __syncthreads();
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
        scaled = check_sums<MT>(a, acc, reinterpret_cast<floatx4 *>(smem + (wm * WN + wn) * tail_floats(TM, TN)), in, constants.least, g, m0 + wm * WTM,
                                [&](int j) {
            const int n = n0 + wn * WTN + j * 32 + lc;
            return n < a.Npix ? n : -1;
        }, k_begin, k_end, 0, a.ICgP);
    }
    tiled_tail<MT, BM, BN, TM, TN, WM, WN, RES, TERMS == 2>(a, smem, acc, tile, g, z, m0, n0, wm, wn, 0, constants, INT_MAX, scaled);
    return 0;
    }   // attempt
};

// X(index, name, KU, PD, TMW, TNW, WM, WN): two terms of half, three products
#define IOS_PIPE3_VARIANTS(X)                            \
    X(119, "x3p_m96n128_w1x4", 1, 2, 3, 1, 1, 4)         \
    X(120, "x3p_m64n128_w1x4", 1, 2, 2, 1, 1, 4)         \
    X(121, "x3p_m64n64_w2x2", 2, 1, 1, 1, 2, 2)          \
    X(122, "x3p_m128n128_w2x2_u2", 2, 1, 2, 2, 2, 2)     \
    X(123, "x3p_m64n128_w1x4_u2", 2, 1, 2, 1, 1, 4)      \
    X(124, "x3p_m128n64_w2x2_u2", 2, 1, 2, 1, 2, 2)      \
    X(125, "x3p_m64n64_w2x2_u4", 4, 1, 1, 1, 2, 2)       \
    X(126, "x3p_m32n128_w1x4_u2", 2, 1, 1, 1, 1, 4)
// one rounded term, bfloat16 (option precision=bf16)
#define IOS_PIPE_BF16_VARIANTS(X)                      \
    X(127, "wb_p_m128n128_w2x2", 4, 1, 2, 2, 2, 2)     \
    X(128, "wb_p_m64n128_w1x4", 4, 1, 2, 1, 1, 4)      \
    X(129, "wb_p_m96n128_w1x4", 4, 1, 3, 1, 1, 4)      \
    X(130, "wb_p_m32n256_w1x4", 2, 1, 1, 2, 1, 4)      \
    X(131, "wb_p_m128n64_w2x2", 4, 1, 2, 1, 2, 2)      \
    X(132, "wb_p_m64n64_w2x2", 4, 1, 1, 1, 2, 2)
// one rounded term, IEEE half (option precision=fp16)
#define IOS_PIPE_FP16_VARIANTS(X)                      \
    X(133, "wh_p_m128n128_w2x2", 4, 1, 2, 2, 2, 2)     \
    X(134, "wh_p_m64n128_w1x4", 4, 1, 2, 1, 1, 4)      \
    X(135, "wh_p_m96n128_w1x4", 4, 1, 3, 1, 1, 4)      \
    X(136, "wh_p_m32n256_w1x4", 2, 1, 1, 2, 1, 4)      \
    X(137, "wh_p_m128n64_w2x2", 4, 1, 2, 1, 2, 2)      \
    X(138, "wh_p_m64n64_w2x2", 4, 1, 1, 1, 2, 2)

constexpr int kFirstPipeVariant = 119;

// The kernels of conv_pipe.hip and their PLAIN forms of conv_pipe_plain.hip, in the order of the lists above; [0] any filter, [1] 1 x 1 filters
// without groups
extern const KernelPair kPipeKernels[][2], kPipePlainKernels[][2];

}  // namespace ios
