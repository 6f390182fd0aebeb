// Quantized products on the matrix cores for many activation rows (a prefill
// batch): the tiled form.
//
// A workgroup of WN x WK waves owns 16 RT WN weight rows and 16 MT activation
// rows; with WK > 1 its waves split K in ranges, each with its own window of
// activations, added at the end (few workgroups: more waves at work on each).
// Each wave owns RT tiles of 16 weight rows over all of the workgroup's
// activation rows and keeps its weights in registers (read, transposed and
// decoded as in mfma_direct.h, a step of four chunks ahead), so that a weight
// is decoded once per 16 MT activations; the activations are staged in LDS in
// the A operand's order, 128 values of K at a time, in two buffers with one
// barrier per window. A's operands are read from LDS once per RT products.
//
// Scales. Q4_K and Q6_K with fp16 activations (FOLD): the weight operand is
// code x 6-bit scale (Q4_K, an integer of at most 945, exact in fp16) or the
// two integers code x 16 (scale / 16) and code x (scale % 16) (Q6_K, in two
// products; both parts with the scale's sign, so that neither is larger than the
// scale: -1 as -16 + 15 would take the rounding of sixteen times its sum, 6.6e-7
// against 8e-8 where every scale is -1), so the matrix cores sum a whole 256-weight
// block before fp32 arithmetic: the block's d scales the tile once per 256 weights (twice
// in short rows, kFoldWhole). Q4_K's minimums are one more product per 256 weights, of the
// eight 6-bit minimums with the eight sub-blocks' activation sums, each sum as three bf16
// parts (24 bits).
// Otherwise every 32-weight block (Q6_K: each 16-weight scale group) is a product
// of its own, scaled in fp32 into the sums (fp32 activations: high and low fp16 parts
// as in mfma_direct.h, the power of two times the scale; Q4_K's minimum times the
// block's fp32 activation sum).
//
// Bound. With two waves per SIMD, waits: on Q4_K 4096->14336 at 512 rows, fp16 x, half
// of the waves' time goes to loads, LDS reads and the barrier, while VALU instructions
// issue for 0.40 of a SIMD's time, the matrix cores are busy for 0.31 and the LDS reads
// (1 KiB per two products) take about a third of their port's. A workgroup alone takes 2 to 11
// us a step of 256 values (mfma_tile.hip), so small products are bound by the length of
// K.
#pragma once

#include "mfma_direct.h"

namespace rq {

typedef __bf16 b8_t __attribute__((ext_vector_type(8)));

template <int FMT, int MT, bool XF32>
struct TileCfg {
    static constexpr bool FOLD = !XF32 && (FMT == Q4_K || FMT == Q6_K);
    static constexpr int XN = XF32 ? 2 : 1;                 // operands per activation tile
    static constexpr int WB = 4;                            // 32-value blocks per window
    static constexpr int ABYTES = WB * MT * XN * 1024;      // a window's operands
    static constexpr int GS = FMT == Q6_K ? 2 : 1;          // scale groups per block
    static constexpr int FBYTES = XF32 ? WB * MT * GS * 64 : 0;  // fp32 x: a power of two per (group, row)
    static constexpr int SBYTES = XF32 && FMT == Q4_K ? WB * MT * 64 : 0;  // fp32 x: activation sums per (block, row)
    static constexpr int BUF = ABYTES + FBYTES + SBYTES;
    static constexpr int SUMS = FOLD && FMT == Q4_K ? MT * 1024 : 0;  // Q4_K FOLD: the sums' operands, two buffers
    static constexpr int LDS = 2 * BUF + 2 * SUMS;          // per range of K
};

// Q4_K FOLD: eight 4-bit codes (stored XOR 8, weight i in bits 4i..4i+3) times a
// scale: the codes go into the mantissas of 1024 and 64 as in nibbles_to_h, and
// one packed fma by (sc, sc) + (-1024 sc, -64 sc) leaves code x sc exactly.
__device__ __forceinline__ void nibbles_scaled(uint32_t w, hv2_t sc, hv2_t off, uint32_t (&o)[4]) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const uint32_t sel = (uint32_t)t | 0x0c00u | ((uint32_t)t << 16) | 0x0c000000u;
        const uint32_t b = __builtin_amdgcn_perm(0u, w, sel);
        const hv2_t v = __builtin_bit_cast(hv2_t, (b & 0x00F0000Fu) ^ 0x54806408u);
        o[t] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(v, sc, off));
    }
}

// Rows from this length on fold whole 256-weight blocks, shorter ones halves: a chain of
// products rounds more than the fp32 additions it replaces, which few blocks do not make
// up for. Error against 64 bits in whole blocks / halves / a product per 32 weights, fp16
// x: Q4_K 1.12e-7 / 0.91e-7 / 1.06e-7 and Q6_K 1.22e-7 / 0.90e-7 / 1.07e-7 at 1,024
// columns; at 2,304 within 5 % of the last with activations of widely unlike magnitudes;
// at 4,096 1.2e-7 in whole blocks against 2.05e-7. Halves cost up to 2 %.
constexpr int kFoldWhole = 2560;

// Waves per SIMD the registers are bounded for: the smallest tile runs two
// workgroups per CU, the others one.
template <int RT, int MT, int WN, int WK, bool XF32>
constexpr int tile_waves() {
    return WN * WK / 4 * (RT * MT * (XF32 ? 2 : 1) <= 4 && WK == 1 ? 2 : 1);
}

template <int FMT, int RT, int MT, int WN, int WK, bool XF32>
__global__ void __launch_bounds__(64 * WN * WK) __attribute__((amdgpu_waves_per_eu(tile_waves<RT, MT, WN, WK, XF32>()))) matvec_mfma_tile(
    MvParams p, int M, uint32_t x_bytes, int n_tiles, int groups) {
    using C = TileCfg<FMT, MT, XF32>;
    constexpr int BPC = RtFmt<FMT>::BPC, WB = C::WB;
    constexpr int NB = 8;                        // 32-weight blocks per step: 256 values of K
    constexpr int SPL = NB / (4 * BPC);          // loads of four chunks per step (two for Q8_0)
    constexpr int WPS = NB / WB;                 // windows per step
    constexpr int FR = WB * MT / WN;             // operand fragments each wave stages per window
    constexpr bool LEAN = tile_waves<RT, MT, WN, WK, XF32>() > 2;  // (128 registers: shorter pipelines, more waves)
    constexpr int DW = RT == 1 && !LEAN ? 3 : 2;          // steps of weights in rotation (DW - 1 in flight)
    constexpr int XD = LEAN || (C::FOLD && RT * MT >= 16) ? 1 : 2;  // windows of activations in flight (one: registers)
    constexpr int PA = LEAN ? (XF32 ? 1 : 3) : XF32 ? 2 : RT * MT >= 16 ? 3 : 6;  // operands read from LDS ahead
    constexpr bool FXA = C::GS == 1 || (!LEAN && RT == 1);  // fp32 x: powers read ahead with the operands (Q6_K's two: registers)
    static_assert(WB * MT % WN == 0 && WPS == 2, "fragments divide over the waves; two windows a step");
    constexpr bool FOLD = C::FOLD;
    extern __shared__ uint4 smem[];
    // Workgroup -> (weight rows, activation rows): the groups of activation
    // rows that share weight rows sit on one XCD (workgroups go to the eight
    // XCDs in turn), so that its L2 serves all but the first.
    const int xcd = (int)blockIdx.x & 7, j8 = (int)blockIdx.x >> 3;
    const int nt = j8 / groups * 8 + xcd, m0 = (j8 % groups) * (16 * MT);
    if (nt >= n_tiles) return;  // (the grid is a whole number of eights)
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wave = wid % WN, wk = wid / WN;  // the wave's rows, its range of K
    const int mn = lane & 15, kq = lane >> 4;
    const int64_t row0 = ((int64_t)nt * WN + wave) * (16 * RT);
    uint8_t* const lds = reinterpret_cast<uint8_t*>(smem) + wk * C::LDS;  // this range's buffers
    const int nch = p.P.nch;
    const bool halves = FOLD && RT == 1 && p.K < kFoldWhole;
    const int loads = (nch + 3) / 4, total = (loads + SPL - 1) / SPL;
    // this wave's steps (every range runs as many rounds as the longest, for the
    // barriers: those past its end compute nothing)
    const int per = (total + WK - 1) / WK, s_begin = per * wk, s_end = total < s_begin + per ? total : s_begin + per;
    const int k_end = p.K < s_end * 256 ? p.K : s_end * 256;
    const __amdgpu_buffer_rsrc_t rs = planes_rsrc(p.P);
    const __amdgpu_buffer_rsrc_t xrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.x), (short)0, (int)x_bytes, 0x00020000);

    // ---- activations: fragment f = wave + W i of a window (block f / MT, tile
    // f % MT); lane (row mn, slice kq) takes eight values ----
    struct Frag {
        uint4 v[C::XN];
    };
    // (past the last activation row, the last row again: its sums are not written)
    uint32_t xoff[FR];
#pragma unroll
    for (int i = 0; i < FR; ++i) {
        const int m = m0 + 16 * ((wave + WN * i) % MT) + mn;
        xoff[i] = (uint32_t)(((int64_t)(m < M ? m : M - 1) * p.ldx + 8 * kq) * (XF32 ? 4 : 2));
    }
    auto load_x = [&](int win, Frag (&fr)[FR]) {
#pragma unroll
        for (int i = 0; i < FR; ++i) {
            const int k = win * (32 * WB) + 32 * ((wave + WN * i) / MT);  // (wave-uniform)
            if (k < k_end) {
#pragma unroll
                for (int h = 0; h < C::XN; ++h) {
                    const u32x4_t r = __builtin_amdgcn_raw_buffer_load_b128(xrs, xoff[i] + 16u * h, k * (XF32 ? 4 : 2), 0);
                    fr[i].v[h] = make_uint4(r[0], r[1], r[2], r[3]);
                }
            } else {
#pragma unroll
                for (int h = 0; h < C::XN; ++h) fr[i].v[h] = make_uint4(0, 0, 0, 0);
            }
        }
    };
    // Sums over a fragment's 32 values per row: with a matrix of ones as the A
    // operand, the product's every row holds them, the sum of row mn in lane mn
    // (fp32 x: times 1 / kSumScale).
    const h8_t ones = XF32 ? sum_operand() : h8_t{1, 1, 1, 1, 1, 1, 1, 1};
    auto store_x = [&](int win, const Frag (&fr)[FR]) {
        uint8_t* const buf = lds + (win & 1) * C::BUF;
        const f4_t z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < FR; ++i) {
            const int f = wave + WN * i, b = f / MT, t = f % MT;
            if constexpr (XF32) {
                float v[8];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = __builtin_bit_cast(float, word(fr[i].v[0], e));
                    v[4 + e] = __builtin_bit_cast(float, word(fr[i].v[1], e));
                }
                float am = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(v[e]));
                const int ks = block_shift(C::GS == 2 ? max_over_pair(am) : max_over_slices(am));
                uint32_t hi[4], lo[4];
                split_hi_lo(v, pow2f(ks), hi, lo);
                const uint4 h4 = make_uint4(hi[0], hi[1], hi[2], hi[3]), l4 = make_uint4(lo[0], lo[1], lo[2], lo[3]);
                *reinterpret_cast<uint4*>(buf + (2 * f) * 1024 + lane * 16) = h4;
                *reinterpret_cast<uint4*>(buf + (2 * f + 1) * 1024 + lane * 16) = l4;
                const float fx = pow2f(-ks);
                if (kq % (4 / C::GS) == 0)
                    *reinterpret_cast<float*>(buf + C::ABYTES + (C::GS * f + kq / (4 / C::GS)) * 64 + mn * 4) = fx;
                if constexpr (FMT == Q4_K) {
                    f4_t sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, __builtin_bit_cast(h8_t, h4), z, 0, 0, 0);
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, __builtin_bit_cast(h8_t, l4), sum, 0, 0, 0);
                    if (kq == 0) *reinterpret_cast<float*>(buf + C::ABYTES + C::FBYTES + f * 64 + mn * 4) = sum[0] * fx;
                }
            } else {
                *reinterpret_cast<uint4*>(buf + f * 1024 + lane * 16) = fr[i].v[0];
                if constexpr (FOLD && FMT == Q4_K) {
                    const f4_t d = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, __builtin_bit_cast(h8_t, fr[i].v[0]), z, 0, 0, 0);
                    const float sum = d[0];
                    // three bf16 parts; slice kq < 3 stores part kq of sub-block
                    // WB (win & 1) + b of the 256-value block (kq = 3: a fourth
                    // part, which the product's zero weights drop; it must only be
                    // finite where the sum is)
                    const uint32_t p0 = __builtin_bit_cast(uint32_t, sum) & 0xFFFF0000u;
                    const float r0 = sum - __builtin_bit_cast(float, p0);
                    const uint32_t p1 = __builtin_bit_cast(uint32_t, r0) & 0xFFFF0000u;
                    const float r1 = r0 - __builtin_bit_cast(float, p1);
                    const uint32_t part = kq == 0 ? p0 : kq == 1 ? p1 : __builtin_bit_cast(uint32_t, r1);
                    uint8_t* const sums = lds + 2 * C::BUF + ((win >> 1) & 1) * C::SUMS;
                    *reinterpret_cast<uint16_t*>(sums + t * 1024 + lane * 16 + (WB * (win & 1) + b) * 2) = (uint16_t)(part >> 16);
                }
            }
        }
    };

    f4_t acc[RT][MT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r][t] = f4_t{0.f, 0.f, 0.f, 0.f};

    // Window w's body stores window w + 1's activations (loaded XD windows
    // earlier) into the other buffer, then asks for window w + 1 + XD's and, in a
    // step's first window, for the weights of DW - 1 steps ahead. The sets of
    // weight registers rotate with the loop unrolled DW times, so that none is
    // copied while its loads are in flight.
    DirectStep<FMT> ring[DW][RT][SPL];
    Frag fr[XD][FR];
    DirectRow rows[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) rows[r] = direct_row(p.P, row0 + 16 * r, p.rows, lane);
    auto load_w = [&](int s, DirectStep<FMT> (&w)[RT][SPL]) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int q = 0; q < SPL; ++q)
                if (s < s_end && s * SPL + q < loads) load_direct_step<FMT>(rs, nch, rows[r], s * SPL + q, w[r][q]);
    };
#pragma unroll
    for (int i = 0; i < XD; ++i) load_x(s_begin * WPS + i, fr[i]);
#pragma unroll
    for (int u = 0; u < DW - 1; ++u) load_w(s_begin + u, ring[u]);
    store_x(s_begin * WPS, fr[0]);
    load_x(s_begin * WPS + XD, fr[0]);
    __syncthreads();
    auto step = [&](int s, const DirectStep<FMT> (&cur)[RT][SPL], DirectStep<FMT> (&ahead)[RT][SPL]) {
        DirectWords<FMT> wd[RT][SPL];
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int q = 0; q < SPL; ++q) direct_words<FMT>(cur[r][q], lane, wd[r][q]);
        f4_t D[FOLD ? RT : 1][FOLD ? MT : 1];
#pragma unroll
        for (int wi = 0; wi < WPS; ++wi) {
            const int win = s * WPS + wi;
            store_x(win + 1, fr[(wi + 1) % XD]);
            load_x(win + 1 + XD, fr[(wi + 1) % XD]);
            if (wi == 0) load_w(s + DW - 1, ahead);
            __builtin_amdgcn_sched_barrier(0);
            if (WK > 1 && s >= s_end) {  // (past this range: only the barriers)
                __syncthreads();
                continue;
            }
            const uint8_t* const buf = lds + (win & 1) * C::BUF;
            const f4_t z = {0.f, 0.f, 0.f, 0.f};
            // The window's operands in order (block, then activation tile): an
            // operand is read from LDS PA before its products, and a product's
            // scaled sums follow the next operand's products (written out, since
            // the compiler gathers a window's reads in front and its sums behind
            // and holds all of them in registers).
            struct Operand {
                h8_t a[C::XN];
                f4_t fx[FXA ? C::GS : 1], bs;
            };
            auto power = [&](int i, int h) { return *reinterpret_cast<const f4_t*>(buf + C::ABYTES + (i * C::GS + h) * 64 + kq * 16); };
            auto read = [&](int i) {
                Operand o;
#pragma unroll
                for (int h = 0; h < C::XN; ++h) o.a[h] = *reinterpret_cast<const h8_t*>(buf + (i * C::XN + h) * 1024 + lane * 16);
                if constexpr (XF32 && FXA) {
#pragma unroll
                    for (int h = 0; h < C::GS; ++h) o.fx[h] = power(i, h);
                }
                if constexpr (XF32 && FMT == Q4_K) o.bs = *reinterpret_cast<const f4_t*>(buf + C::ABYTES + C::FBYTES + i * 64 + kq * 16);
                return o;
            };
            Operand ops[PA + 1];
#pragma unroll
            for (int i = 0; i < PA; ++i) ops[i] = read(i);
            if constexpr (FOLD) {
                h8_t B[RT], B2[RT];
#pragma unroll
                for (int i = 0; i < WB * MT; ++i) {
                    const int b = wi * WB + i / MT, t = i % MT;
                    const Operand cu = ops[i % (PA + 1)];
                    if (i + PA < WB * MT) ops[(i + PA) % (PA + 1)] = read(i + PA);
                    if (t == 0) {
#pragma unroll
                        for (int r = 0; r < RT; ++r) {
                            const int c = b / BPC, sub = b % BPC;  // (FOLD formats: one load a step)
                            const DirectStep<FMT>& cw = cur[r][0];
                            uint32_t o[4];
                            if constexpr (FMT == Q4_K) {
                                uint32_t scv, mnv;
                                q4k_scale_min(cw.meta, b, scv, mnv);
                                const _Float16 sc = (_Float16)(float)scv;
                                const hv2_t s2 = {sc, sc};
                                const hv2_t off = s2 * (hv2_t){(_Float16)-1024.f, (_Float16)-64.f};
                                nibbles_scaled((sub ? wd[r][0].X1 : wd[r][0].X0)[0][c], s2, off, o);
                                B[r] = __builtin_bit_cast(h8_t, make_uint4(o[0], o[1], o[2], o[3]));
                            } else {
                                // the scale of this lane's slice: group 2 sub + kq / 2 of the chunk
                                const uint32_t scw = word(cw.meta, c) >> (16 * sub + 8 * (kq >> 1));
                                const _Float16 sv = (_Float16)(short)(int8_t)(scw & 0xffu);
                                const _Float16 sh = __builtin_elementwise_trunc(sv * (_Float16)0.0625f) * (_Float16)16.f;
                                const _Float16 sl = sv - sh;
                                const h8_t q = direct_operand<FMT>(wd[r][0], b, kq);
                                B[r] = q * (h8_t){sh, sh, sh, sh, sh, sh, sh, sh};
                                B2[r] = q * (h8_t){sl, sl, sl, sl, sl, sl, sl, sl};
                            }
                        }
                    }
#pragma unroll
                    for (int r = 0; r < RT; ++r) {
                        D[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cu.a[0], B[r], b == 0 ? z : D[r][t], 0, 0, 0);
                        if constexpr (FMT == Q6_K) D[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cu.a[0], B2[r], D[r][t], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                h8_t B[RT], B1[RT];  // (Q6_K: the first and the second scale group's)
                float s0[RT], s1[RT], p0[RT], p1[RT];
                f4_t d[RT], e[RT], pd[RT], pe[RT], pfx[C::GS], pbs;
                auto add = [&](int t) {  // the previous operand's products into its sums
#pragma unroll
                    for (int r = 0; r < RT; ++r) {
                        f4_t& ac = acc[r][t];
                        if constexpr (FMT == Q6_K) {
#pragma unroll
                            for (int j = 0; j < 4; ++j) ac[j] = fmaf(XF32 ? p1[r] * pfx[C::GS - 1][j] : p1[r], pe[r][j], ac[j]);
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            ac[j] = fmaf(XF32 ? p0[r] * pfx[0][j] : p0[r], pd[r][j], ac[j]);
                            if constexpr (FMT == Q4_K) ac[j] = fmaf(-p1[r], pbs[j], ac[j]);
                        }
                        pin(ac);
                    }
                };
#pragma unroll
                for (int i = 0; i < WB * MT; ++i) {
                    const int b = wi * WB + i / MT, t = i % MT;
                    const Operand cu = ops[i % (PA + 1)];
                    if (i + PA < WB * MT) ops[(i + PA) % (PA + 1)] = read(i + PA);
                    if (t == 0) {
#pragma unroll
                        for (int r = 0; r < RT; ++r) {
                            constexpr int BL = 4 * BPC;  // blocks per load
                            B[r] = direct_operand<FMT>(wd[r][b / BL], b % BL, kq);
                            if constexpr (FMT == Q6_K) {
                                B1[r] = group_operand(B[r], kq >= 2);
                                B[r] = group_operand(B[r], kq < 2);
                            }
                            direct_scales<FMT>(cur[r][b / BL], b % BL, 4 * SPL * s + b / BPC < nch, s0[r], s1[r]);
                            if constexpr (FMT == Q4_K) s1[r] *= kSumScale;
                        }
                    }
                    auto product = [&](const h8_t& Wt) {
                        f4_t v = __builtin_amdgcn_mfma_f32_16x16x32_f16(cu.a[0], Wt, z, 0, 0, 0);
                        if constexpr (XF32) v = __builtin_amdgcn_mfma_f32_16x16x32_f16(cu.a[C::XN - 1], Wt, v, 0, 0, 0);
                        return v;
                    };
#pragma unroll
                    for (int r = 0; r < RT; ++r) {
                        d[r] = product(B[r]);
                        if constexpr (FMT == Q6_K) e[r] = product(B1[r]);
                    }
                    if (i > 0) add((i - 1) % MT);
#pragma unroll
                    for (int r = 0; r < RT; ++r) {
                        pd[r] = d[r];
                        if constexpr (FMT == Q6_K) pe[r] = e[r];
                        p0[r] = s0[r];
                        p1[r] = s1[r];
                    }
#pragma unroll
                    for (int h = 0; h < C::GS; ++h) pfx[h] = XF32 && !FXA ? power(i, h) : cu.fx[FXA ? h : 0];
                    pbs = cu.bs;
                }
                add(MT - 1);
            }
            if constexpr (FOLD) {
                if (wi == 0 && halves) {  // (short rows: half a block's tile at a time)
#pragma unroll
                    for (int t = 0; t < MT; ++t)
#pragma unroll
                        for (int r = 0; r < RT; ++r) {
                            const float dd = half_lo(FMT == Q4_K ? cur[r][0].meta.x : cur[r][0].d);
#pragma unroll
                            for (int j = 0; j < 4; ++j) acc[r][t][j] = fmaf(dd, D[r][t][j], acc[r][t][j]);
                            D[r][t] = z;
                        }
                }
                if (wi == WPS - 1) {
                    // the 256-weight block's tile into the sums
                    b8_t Bm[FMT == Q4_K ? RT : 1];
                    if constexpr (FMT == Q4_K) {
#pragma unroll
                        for (int r = 0; r < RT; ++r) {
                            uint32_t mw[4];
#pragma unroll
                            for (int c = 0; c < 4; ++c) {
                                uint32_t sc0, mn0, sc1, mn1;
                                q4k_scale_min(cur[r][0].meta, 2 * c, sc0, mn0);
                                q4k_scale_min(cur[r][0].meta, 2 * c + 1, sc1, mn1);
                                // small integers are exact in bf16: the high halves of their fp32 patterns
                                mw[c] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, (float)mn1),
                                                              __builtin_bit_cast(uint32_t, (float)mn0), 0x07060302u);
                                mw[c] = kq < 3 ? mw[c] : 0u;
                            }
                            Bm[r] = __builtin_bit_cast(b8_t, make_uint4(mw[0], mw[1], mw[2], mw[3]));
                        }
                    }
                    const uint8_t* const sums = lds + 2 * C::BUF + (s & 1) * C::SUMS;
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
                        b8_t Am;
                        if constexpr (FMT == Q4_K) Am = *reinterpret_cast<const b8_t*>(sums + t * 1024 + lane * 16);
#pragma unroll
                        for (int r = 0; r < RT; ++r) {
                            const float dd = half_lo(FMT == Q4_K ? cur[r][0].meta.x : cur[r][0].d);
#pragma unroll
                            for (int j = 0; j < 4; ++j) acc[r][t][j] = fmaf(dd, D[r][t][j], acc[r][t][j]);
                            if constexpr (FMT == Q4_K) {
                                const f4_t dm = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Am, Bm[r], z, 0, 0, 0);
                                const float dmin = half_hi(cur[r][0].meta.x);
#pragma unroll
                                for (int j = 0; j < 4; ++j) acc[r][t][j] = fmaf(-dmin, dm[j], acc[r][t][j]);
                            }
                        }
                    }
                }
            }
            __syncthreads();
        }
    };
    for (int s = 0; s < per; s += DW)
#pragma unroll
        for (int u = 0; u < DW; ++u)
            if (s + u < per) step(s_begin + s + u, ring[u], ring[(u + DW - 1) % DW]);

    // the ranges' tiles, added in order
    if constexpr (WK > 1) {
        f4_t* const red = reinterpret_cast<f4_t*>(smem);
        constexpr int NT = RT * MT;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int t = 0; t < MT; ++t) red[(wid * NT + r * MT + t) * 64 + lane] = acc[r][t];
        __syncthreads();
        // wave (rows, range wk) writes every WK-th tile
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            if (i % WK != wk) continue;
            f4_t v = red[(wave * NT + i) * 64 + lane];
#pragma unroll
            for (int w = 1; w < WK; ++w) {
                const f4_t o = red[((w * WN + wave) * NT + i) * 64 + lane];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] += o[j];
            }
            const int64_t row = row0 + 16 * (i / MT) + mn;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int m = m0 + 16 * (i % MT) + 4 * kq + j;
                if (row < p.rows && m < M) p.y[(int64_t)m * p.ldy + row] = v[j];
            }
        }
        return;
    }

#pragma unroll
    for (int r = 0; r < RT; ++r) {
        const int64_t row = row0 + 16 * r + mn;
        if (row >= p.rows) continue;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int m = m0 + 16 * t + 4 * kq + j;
                if (m < M) p.y[(int64_t)m * p.ldy + row] = acc[r][t][j];
            }
    }
}

}  // namespace rq
