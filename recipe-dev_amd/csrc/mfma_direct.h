// Quantized products on the matrix cores, fp32 activations: the form whose
// waves read their activations straight from the caches.
//
// A wave owns RT tiles of 16 weight rows, MT tiles of 16 activation rows and a
// range of K; the waves of a workgroup split K between them and add their
// tiles in LDS in wave order at the end, so there is no barrier in the loop
// and results are deterministic. Weights are read as in the streaming form
// (mfma_rt.h): 16 rows x 4 chunks x 16 bytes per load instruction, one step of
// four chunks ahead, transposed to the B operand's order by lane swaps in
// registers. A lane (row m, slice kq) loads the eight activations its A
// operand holds, PD operands ahead.
//
// fp32 activations become two fp16 operands per 32-value block: the block (Q6_K:
// each of its two 16-value scale groups) is scaled by the power of two 2^k that
// brings its largest magnitude into [2^14, 2^15) and split into a high and a low
// part (x = hi + lo to 2^-22 of the value); its scale times 2^-k multiplies the
// sum of the two products in fp32. Up to eight activation rows (PACK), the high parts are
// rows 0-7 of one A operand and the low parts rows 8-15: the same count of
// matrix-core products as fp16 activations, the two halves added at the end.
//
// 2^-k is known in the lanes of activation row m = lane & 15, and the product
// leaves row 4 kq + j in register j of lane (n, kq): three row rotations bring
// lane j of 16-lane row kq the power of row 4 kq + j, and the multiplications
// by it take it through a row broadcast (DPP).
//
// Bound. VALU issue: 0.75 of a SIMD's time on Q6_K 14336->4096 at 77 rows, 0.59 on
// Q4_K 4096x4096 at five, most of it the conversions of the activations, which every
// row tile's workgroup repeats (about 45 instructions per eight values); at few rows
// also the round trips of a wave's two or four steps. The weights' bytes take a fifth
// of the time. Measured against the staged form this replaces (kernel us, fp32 x): Q4_K
// 4096x4096 at 5 rows 83.8 -> 12.2 (780 GB/s), Q6_K 14336->4096 at 77 rows
// 3363 -> 106 (85 TFLOP/s).
#pragma once

#include <hip/hip_ext.h>

#include "halfcode.h"
#include "kernels.h"
#include "mfma_rt.h"

namespace rq {

// The exponent k that brings a block's largest magnitude `amax` into
// [2^14, 2^15) (fp16 holds up to 65504), 0 for a zero or non-finite block,
// within [-126, 126] so that 2^-k is a normal fp32.
__device__ __forceinline__ int block_shift(float amax) {
    if (!(amax > 0.f) || !(amax <= 3.402823466e38f)) return 0;
    const int k = 15 - __builtin_amdgcn_frexp_expf(amax);
    return k < -126 ? -126 : (k > 126 ? 126 : k);
}

__device__ __forceinline__ float pow2f(int k) { return __builtin_bit_cast(float, (uint32_t)(127 + k) << 23); }

typedef float f2_t __attribute__((ext_vector_type(2)));

// Eight scaled values v * 2^k as fp16 high parts and the fp16 roundings of what
// is left.
__device__ __forceinline__ void split_hi_lo(const float (&v)[8], float scale, uint32_t (&hi)[4], uint32_t (&lo)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float a = v[2 * e] * scale, b = v[2 * e + 1] * scale;
        const hv2_t h = __builtin_convertvector((f2_t){a, b}, hv2_t);
        const hv2_t l = __builtin_convertvector((f2_t){a - (float)h.x, b - (float)h.y}, hv2_t);
        hi[e] = __builtin_bit_cast(uint32_t, h);
        lo[e] = __builtin_bit_cast(uint32_t, l);
    }
}

// A copy of a value that the compiler does not know to be one: of a swap whose
// two operands are the same value it takes both results to be equal, which
// they are not.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// Keeps a tile's arithmetic where it stands: sums that only the end of a loop's
// body reads would otherwise all be moved there, with every product they take
// held in registers until then.
__device__ __forceinline__ void pin(f4_t& v) { asm volatile("" : "+v"(v)); }

// The largest of a value over slices 0 and 1, or 2 and 3 (the lanes 16 apart that
// hold one scale group of Q6_K), in both.
__device__ __forceinline__ float max_over_pair(float v) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = opaque(a);
    swap_bit4(a, b);
    return fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}
// A value of each pair, first and second, in all four lanes.
__device__ __forceinline__ void both_pairs(float v, float& first, float& second) {
    uint32_t a = __builtin_bit_cast(uint32_t, v), b = opaque(a);
    swap_bit5(a, b);
    first = __builtin_bit_cast(float, a);
    second = __builtin_bit_cast(float, b);
}
__device__ __forceinline__ float max_over_slices(float v) {
    float a, b;
    both_pairs(max_over_pair(v), a, b);
    return fmaxf(a, b);
}

// Lane i of 16-lane row kq takes lane (i + 4 kq) mod 16 of a value that every
// row holds alike, so that lane j < 4 has the value of lane 4 kq + j.
__device__ __forceinline__ float rotate_to_rows(float v) {
    const int s = __builtin_bit_cast(int, v);
    int r = s;
    r = __builtin_amdgcn_update_dpp(r, s, 0x12C, 0x2, 0xF, false);  // row 1: row_ror:12
    r = __builtin_amdgcn_update_dpp(r, s, 0x128, 0x4, 0xF, false);  // row 2: row_ror:8
    r = __builtin_amdgcn_update_dpp(r, s, 0x124, 0x8, 0xF, false);  // row 3: row_ror:4
    return __builtin_bit_cast(float, r);
}
// The same of a value that rows 0 and 1, and rows 2 and 3, hold alike, for each pair's
// (rows 1 and 3 turn by 12 before the exchange, rows 2 and 3 by 8 after it).
__device__ __forceinline__ void rotate_pairs_to_rows(float v, float& first, float& second) {
    const int s = __builtin_bit_cast(int, v);
    v = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(s, s, 0x12C, 0xA, 0xF, false));  // row_ror:12
    both_pairs(v, first, second);
    const int a = __builtin_bit_cast(int, first), b = __builtin_bit_cast(int, second);
    first = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(a, a, 0x128, 0xC, 0xF, false));  // row_ror:8
    second = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(b, b, 0x128, 0xC, 0xF, false));
}
template <int J>
__device__ __forceinline__ float row_bcast(float v) {
    const int s = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(s, s, 0x150 + J, 0xF, 0xF, false));  // row_newbcast:J
}

// One step (four chunks) of one 16-row tile: code words as loaded, and the
// scales of row n = lane & 15.
template <int FMT>
struct DirectStep {
    uint32_t w[Traits<FMT>::QP][1][4];
    uint4 meta;
    uint32_t d;  // Q6_K: the quad's fp16 d
};

// A lane's loads of a tile: row n = lane & 15 (the last row again past the
// weight's end: its sums are not written), chunk lane >> 4 of each step. The
// step's own offset is wave-uniform and goes into the loads' scalar offset.
// Every address lies in the row: a row's scale bytes are whole quads, and the
// chunks past its last are read as the last again (their activations are zeros).
struct DirectRow {
    uint32_t at;  // the row's byte offset
    int chunk;
};
__device__ __forceinline__ DirectRow direct_row(const Planes& P, int64_t row0, int64_t rows, int lane) {
    const int64_t row = row0 + (lane & 15);
    return DirectRow{(uint32_t)(row < rows ? row : rows - 1) * (uint32_t)P.row_bytes, lane >> 4};
}

// Step s (chunks 4 s .. 4 s + 3, s below the count of steps) of a tile.
template <int FMT>
__device__ __forceinline__ void load_direct_step(__amdgpu_buffer_rsrc_t rs, int nch, const DirectRow& row, int s,
                                                 DirectStep<FMT>& t) {
    constexpr int QP = Traits<FMT>::QP, QB = RtFmt<FMT>::QB;
    const int c0 = 4 * s, within = c0 & 63;
    const int rest = nch - (c0 & ~63), nb = rest > 64 ? 64 : rest;
    const int gbase = (c0 >> 6) * (int)full_group_bytes<FMT>();
    int chunk = row.chunk;
    if constexpr (FMT == Q8_0 || FMT == Q4_0)  // (the others have whole quads)
        if (nch - c0 < 4) chunk = chunk < nch - c0 ? chunk : nch - c0 - 1;
    const uint32_t off = row.at + 16u * (uint32_t)chunk;
#pragma unroll
    for (int part = 0; part < QP; ++part) {
        const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rs, off, gbase + (part * nb + within) * 16, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) t.w[part][0][j] = v[j];
    }
    const int meta = gbase + QP * nb * 16, quad = within >> 2;
    if constexpr (QB == 16) {
        const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(rs, row.at, meta + quad * 16, 0);
        t.meta = make_uint4(v[0], v[1], v[2], v[3]);
    } else {
        const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(rs, row.at, meta + quad * 8, 0);
        t.meta = make_uint4(v[0], v[1], 0u, 0u);
    }
    t.d = 0u;
    if constexpr (FMT == Q6_K) t.d = __builtin_amdgcn_raw_buffer_load_b16(rs, row.at, meta + (nb >> 2) * 16 + quad * 2, 0);
}

// The B-operand words of a step, transposed from the loaded words (RB = 16 of
// mfma_rt.h): word kq of chunk c for lane (row n, kq) at [c].
template <int FMT>
struct DirectWords {
    uint32_t X0[1][4], X1[1][4], X2[1][4], X3[1][4];
};
template <int FMT>
__device__ __forceinline__ void direct_words(const DirectStep<FMT>& t, int lane, DirectWords<FMT>& o) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if constexpr (FMT == Q8_0) {
            o.X0[0][j] = t.w[j >> 1][0][2 * (j & 1)];
            o.X1[0][j] = t.w[j >> 1][0][2 * (j & 1) + 1];
        } else {
            o.X0[0][j] = t.w[0][0][j];
            o.X1[0][j] = t.w[1][0][j];
            if constexpr (FMT == Q6_K) {
                o.X2[0][j] = t.w[2][0][j >> 1];
                o.X3[0][j] = t.w[2][0][2 + (j >> 1)];
            }
        }
    }
    transpose_words<16>(o.X0, lane);
    transpose_words<16>(o.X1, lane);
    if constexpr (FMT == Q6_K) {
        transpose_words<16>(o.X2, lane);
        transpose_words<16>(o.X3, lane);
    }
}

// Block b (chunk c = b / BPC of the step, sub-block b % BPC) as the B operand.
template <int FMT>
__device__ __forceinline__ h8_t direct_operand(const DirectWords<FMT>& w, int b, int kq) {
    constexpr int BPC = RtFmt<FMT>::BPC;
    const int c = b / BPC, sub = b % BPC;
    uint32_t o[4];
    if constexpr (FMT == Q4_0 || FMT == Q4_K) {
        nibbles_to_h((sub ? w.X1 : w.X0)[0][c] ^ 0x88888888u, FMT == Q4_0 ? 0xD480E408u : 0xD400E400u, o);
    } else if constexpr (FMT == Q8_0) {
        bytes_to_h(w.X0[0][c], o[0], o[1]);
        bytes_to_h(w.X1[0][c], o[2], o[3]);
    } else {
        q6_to_h((sub ? w.X1 : w.X0)[0][c] ^ 0x88888888u, ((sub ? w.X3 : w.X2)[0][c] >> (2 * (kq & 1))) & 0x33333333u, o);
    }
    return __builtin_bit_cast(h8_t, make_uint4(o[0], o[1], o[2], o[3]));
}

// Q6_K: a block's weights with those of the other scale group (first: slices 0 and
// 1) zero. A product per group, each scaled on its own: the second group's sum as
// the whole block's less the first's would keep the first's rounding, however small
// its scale (one value of 1e5 in a group of scale 0 beside one of scale 100, 4096
// columns: error against 64 bits 6e-5 instead of 3e-7).
__device__ __forceinline__ h8_t group_operand(const h8_t& B, bool mine) {
    const uint4 o = __builtin_bit_cast(uint4, B);
    return __builtin_bit_cast(h8_t, make_uint4(mine ? o.x : 0u, mine ? o.y : 0u, mine ? o.z : 0u, mine ? o.w : 0u));
}

// Sub-block `b` (0..7) of a Q4_K superblock: its six-bit scale and minimum, for
// an index known at compile time (one funnel shift per 24-bit field).
__device__ __forceinline__ void q4k_scale_min(const uint4& meta, int b, uint32_t& sc, uint32_t& mn) {
    const int p = b >> 1;
    const uint32_t f = p == 0   ? meta.y
                       : p == 1 ? __builtin_amdgcn_alignbit(meta.z, meta.y, 24)
                       : p == 2 ? __builtin_amdgcn_alignbit(meta.w, meta.z, 16)
                                : meta.w >> 8;
    sc = bfe(f, 12 * (b & 1), 6);
    mn = bfe(f, 12 * (b & 1) + 6, 6);
}

// Row n's scales of block b of a step: s0 (Q6_K: the first 16-value group's),
// s1 (Q4_K: the minimum; Q6_K: the second group's). Chunks
// past the row's end scale by zero (the bytes there are not the row's).
template <int FMT>
__device__ __forceinline__ void direct_scales(const DirectStep<FMT>& t, int b, bool chunk_ok, float& s0, float& s1) {
    constexpr int BPC = RtFmt<FMT>::BPC;
    const int c = b / BPC, sub = b % BPC;
    s1 = 0.f;
    if constexpr (FMT == Q4_K) {
        uint32_t sc, mn;
        q4k_scale_min(t.meta, b, sc, mn);
        s0 = half_lo(t.meta.x) * (float)sc;
        s1 = half_hi(t.meta.x) * (float)mn;
    } else if constexpr (FMT == Q4_0) {
        const uint32_t dw = word(t.meta, c);
        s0 = sub ? half_hi(dw) : half_lo(dw);
        s0 = chunk_ok ? s0 : 0.f;
    } else if constexpr (FMT == Q8_0) {
        const uint32_t dw = word(t.meta, c >> 1);
        s0 = (c & 1) ? half_hi(dw) : half_lo(dw);
        s0 = chunk_ok ? s0 : 0.f;
    } else {
        const uint32_t scw = word(t.meta, c);
        const float dd = half_lo(t.d);
        s0 = dd * (float)(int8_t)((scw >> (16 * sub)) & 0xffu);
        s1 = dd * (float)(int8_t)((scw >> (16 * sub + 8)) & 0xffu);
    }
}

// Q4_K: a block's activations are summed as 2^-6 of their sum (exactly: a product
// with this operand), and the minimum multiplies as 2^6 of itself, so that the sum of
// 32 values of up to fp32's largest does not overflow before a small minimum scales it.
constexpr float kSumScale = 64.f;
__device__ __forceinline__ h8_t sum_operand() {
    constexpr _Float16 u = (_Float16)(1.f / kSumScale);
    return h8_t{u, u, u, u, u, u, u, u};
}

constexpr int kDirectMaxWaves = 8;

template <int FMT, int RT, int MT, bool PACK>
__global__ void __launch_bounds__(64 * kDirectMaxWaves) matvec_mfma_direct(MvParams p, int M, uint32_t x_bytes, int WK,
                                                                                   int groups) {
    static_assert(!PACK || MT == 1, "packed rows are one operand tile");
    constexpr int BPC = RtFmt<FMT>::BPC, NB = 4 * BPC, CW = Traits<FMT>::CW;
    constexpr int ROWS = PACK ? 8 : 16 * MT;   // activation rows of a workgroup
    constexpr int NI = NB * MT;                // A operands per step, block-major
    constexpr int PD = MT == 1 ? NB : 4;       // A operands in flight
    static_assert(NI % PD == 0, "the ring of operands divides a step");
    extern __shared__ uint4 smem[];
    const int lane = threadIdx.x & 63;
    const int wk = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int mn = lane & 15, kq = lane >> 4;
    // workgroup: row tiles blockIdx.x / groups, activation rows blockIdx.x % groups
    // (neighbours read the same weights at about the same time)
    const int tile = (int)blockIdx.x / groups;
    const int64_t row0 = (int64_t)tile * (16 * RT);
    const int m0 = ((int)blockIdx.x - tile * groups) * ROWS;
    const int nch = p.P.nch;
    const int total = (nch + 3) / 4;
    const int s_begin = (int)((int64_t)total * wk / WK), s_end = (int)((int64_t)total * (wk + 1) / WK);
    const __amdgpu_buffer_rsrc_t rs = planes_rsrc(p.P);
    const __amdgpu_buffer_rsrc_t xrs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.x), (short)0, (int)x_bytes, 0x00020000);
    // byte offset of this lane's eight values of step 0, block 0, per activation
    // tile (past the last row, the last row again: its sums are not written)
    uint32_t xoff[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int m = m0 + (PACK ? (mn & 7) : 16 * t + mn);
        xoff[t] = (uint32_t)(((int64_t)(m < M ? m : M - 1) * p.ldx + 8 * kq) * 4);
    }
    struct AItem {
        uint4 v[2];
    };
    auto load_a = [&](int s, int i, AItem& a) {
        const int b = i / MT, t = i % MT;
        const int k = s * (4 * CW) + 32 * b;  // (wave-uniform)
        if (s < s_end && k < p.K) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const u32x4_t r = __builtin_amdgcn_raw_buffer_load_b128(xrs, xoff[t] + 16u * h, k * 4, 0);
                a.v[h] = make_uint4(r[0], r[1], r[2], r[3]);
            }
        } else {
            a.v[0] = a.v[1] = make_uint4(0, 0, 0, 0);
        }
    };

    f4_t acc[RT][MT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r][t] = f4_t{0.f, 0.f, 0.f, 0.f};

    DirectRow rows[RT];
    DirectStep<FMT> cur[RT], nxt[RT];
    AItem ring[PD];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        rows[r] = direct_row(p.P, row0 + 16 * r, p.rows, lane);
        if (s_begin < s_end) load_direct_step<FMT>(rs, nch, rows[r], s_begin, cur[r]);
    }
#pragma unroll
    for (int i = 0; i < PD; ++i) load_a(s_begin + i / NI, i % NI, ring[i]);
    for (int s = s_begin; s < s_end; ++s) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
            if (s + 1 < s_end) load_direct_step<FMT>(rs, nch, rows[r], s + 1, nxt[r]);
        DirectWords<FMT> wd[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) direct_words<FMT>(cur[r], lane, wd[r]);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            h8_t B[RT], B1[RT];  // (Q6_K: the first and the second scale group's)
            float s0[RT], s1[RT];
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                B[r] = direct_operand<FMT>(wd[r], b, kq);
                if constexpr (FMT == Q6_K) {
                    B1[r] = group_operand(B[r], kq >= 2);
                    B[r] = group_operand(B[r], kq < 2);
                }
                direct_scales<FMT>(cur[r], b, 4 * s + b / BPC < nch, s0[r], s1[r]);
                if constexpr (FMT == Q4_K) s1[r] *= kSumScale;
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const int i = b * MT + t;
                const AItem a = ring[i % PD];
                load_a(s + (i + PD) / NI, (i + PD) % NI, ring[i % PD]);
                float v[8];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = __builtin_bit_cast(float, word(a.v[0], e));
                    v[4 + e] = __builtin_bit_cast(float, word(a.v[1], e));
                }
                // the block's (Q6_K: each scale group's) largest magnitude (a NaN
                // takes the zero shift's way through the split, as an infinity does)
                float am = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) am = fmaxf(am, fabsf(v[e]));
                uint32_t hi[4], lo[4];
                float f[4], g[4];  // the inverse powers of rows 4 kq + j (g: the second group's)
                auto rows_of = [](float fx, float (&o)[4]) {
                    o[0] = row_bcast<0>(fx);
                    o[1] = row_bcast<1>(fx);
                    o[2] = row_bcast<2>(fx);
                    o[3] = row_bcast<3>(fx);
                };
                const int ks = block_shift(FMT == Q6_K ? max_over_pair(am) : max_over_slices(am));
                split_hi_lo(v, pow2f(ks), hi, lo);
                if constexpr (FMT == Q6_K) {
                    float f0, f1;
                    rotate_pairs_to_rows(pow2f(-ks), f0, f1);
                    rows_of(f0, f);
                    rows_of(f1, g);
                } else {
                    rows_of(rotate_to_rows(pow2f(-ks)), f);
                }
                h8_t A[2];
                if constexpr (PACK) {
                    const bool low = mn >= 8;
                    A[0] = __builtin_bit_cast(h8_t, make_uint4(low ? lo[0] : hi[0], low ? lo[1] : hi[1], low ? lo[2] : hi[2],
                                                               low ? lo[3] : hi[3]));
                } else {
                    A[0] = __builtin_bit_cast(h8_t, make_uint4(hi[0], hi[1], hi[2], hi[3]));
                    A[1] = __builtin_bit_cast(h8_t, make_uint4(lo[0], lo[1], lo[2], lo[3]));
                }
                const f4_t z = {0.f, 0.f, 0.f, 0.f};
                auto product = [&](const h8_t& W) {
                    f4_t D = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[0], W, z, 0, 0, 0);
                    if constexpr (!PACK) D = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[1], W, D, 0, 0, 0);
                    return D;
                };
                f4_t bs = z;
                if constexpr (FMT == Q4_K) {  // the block's activation sums
                    bs = product(sum_operand());
#pragma unroll
                    for (int j = 0; j < 4; ++j) bs[j] *= f[j];
                }
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    const f4_t D = product(B[r]);
                    f4_t& ac = acc[r][t];
                    if constexpr (FMT == Q6_K) {
                        const f4_t D1 = product(B1[r]);
#pragma unroll
                        for (int j = 0; j < 4; ++j) ac[j] = fmaf(s1[r] * g[j], D1[j], ac[j]);
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) ac[j] = fmaf(s0[r] * f[j], D[j], ac[j]);
                    if constexpr (FMT == Q4_K) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) ac[j] = fmaf(-s1[r], bs[j], ac[j]);
                    }
                    pin(ac);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) cur[r] = nxt[r];
    }

    // the waves' tiles, added in wave order
    f4_t* red = reinterpret_cast<f4_t*>(smem);
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) red[(wk * (RT * MT) + r * MT + t) * 64 + lane] = acc[r][t];
    __syncthreads();
    for (int it = wk; it < RT * MT; it += WK) {
        f4_t v = red[it * 64 + lane];
        for (int w = 1; w < WK; ++w) {
            const f4_t o = red[(w * (RT * MT) + it) * 64 + lane];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] += o[j];
        }
        if constexpr (PACK) {  // high and low parts of row m: operand rows m and m + 8
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float part = v[j];  // (a bit cast of a vector's element would read element 0)
                uint32_t a = __builtin_bit_cast(uint32_t, part), b = opaque(a);
                swap_bit5(a, b);
                v[j] = __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
            }
        }
        const int64_t row = row0 + 16 * (it / MT) + mn;
        if (row < p.rows && (!PACK || kq < 2)) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int m = m0 + 16 * (it % MT) + 4 * kq + j;
                if (m < M) p.y[(int64_t)m * p.ldy + row] = v[j];
            }
        }
    }
}

}  // namespace rq
