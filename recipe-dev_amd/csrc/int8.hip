// recipe's int(8) sum on gfx950: the default precision profile's `sum = "int8"`
// with a 32-input step and the llama.cpp profile's 256-input step.
//
// The activation column of each position is rounded, in the workgroup's LDS,
// to Q8 records: per `step` inputs one fp32 step d and a signed byte per input
// (amd-nv-cpu.ll:1304-1500). Weight codes come from the repacked layout
// (layout.h) and dot the record bytes in v_dot4_i32_i8; every integer is exact,
// so the integer work is free to take any order, and the fp32 tail runs in
// recipe's order so each output carries recipe's bits.
//
// Reference: contraction_forward_gemv_wave_body on a backend with int8 dots
// (amd-nv-cpu.ll:1231-2241) and its slice helpers (build.rs:743-915).
// recipe's GPU backends run 32 lanes per output (NVIDIA warps, gfx11/gfx12
// wave32). Here each wave64 runs two outputs on its two 32-lane halves: lane l
// of a half holds exactly the partial sums recipe's lane l holds, and
// lane exchanges within the half (lane_xor) repeat recipe's butterfly.
//
// fp32 order per output (this file is built with -ffp-contract=off, and fmaf
// stands where recipe's state madd is):
//   16-value slices (Q4_K and Q6_K at a 32 step; Q8_0 and Q4_0 at either step):
//     lane l adds slices l, l+32, ... from +0; the lanes meet at offsets 16..1.
//       Q4_K  d8 * ((d*sc)*dot - (dmin*m)*sum)
//       Q6_K  d * (d8 * (sc * (dot - 32 sum)))
//       Q8_0, Q4_0  d8 * ((d*dot) + 0*sum), Q4_0's dot less 8 sum
//   Q4_K at a 256 step: acc = fma(dot_b, d*d8, acc), accmin = fma(min_b, dmin*d8,
//     accmin) per block in order (per quarter of the block for positions before
//     the last M % 4, unless the tail rule makes the last position whole); the
//     output is acc - accmin.
//   Q6_K at a 256 step: eight chains f_l = fma(d8*d, i_l, f_l) per block, added
//     as ((f0 + f4) + (f2 + f6)) + ((f1 + f5) + (f3 + f7)).
#include <hip/hip_runtime.h>

#include "chunk.h"
#include <stdlib.h>

#include "kernels.h"

namespace rq {

namespace {

constexpr int kI8Threads = 512;                  // eight waves
constexpr int kI8Rows = 2 * (kI8Threads / 64);   // outputs per workgroup: two per wave

// Extreme selection of recipe's Q8 records (amd-nv-cpu.ll:1422-1470): the
// partner replaces the running extreme when its magnitude is larger, or equal
// with a larger signed value. Scanning values in any order from +0 with this
// rule yields the value recipe's 32-lane butterfly leaves: the maximum under
// (magnitude, signed value), zeros and NaNs never replacing +0.
__device__ __forceinline__ bool extreme_wins(float p, float e) {
    const float ap = fabsf(p), ae = fabsf(e);
    return ap > ae || (ap == ae && p > e);
}

// inverse = -127 / extreme and d = 1 / inverse, both correctly rounded; an
// all-zero step has inverse 0 and d 0 (amd-nv-cpu.ll:1447-1456).
__device__ __forceinline__ void step_of(float e, float& inverse, float& d) {
    const bool nonzero = fabsf(e) > 0.f;
    const float inverse_raw = -127.f / (nonzero ? e : 1.f);
    const float d_raw = 1.f / inverse_raw;
    inverse = nonzero ? inverse_raw : 0.f;
    d = nonzero ? d_raw : 0.f;
}

// The 32 inputs of one record from a 16-byte aligned row.
__device__ __forceinline__ void load_record(const float* __restrict__ xr, float4 (&xv)[8]) {
#pragma unroll
    for (int q = 0; q < 8; ++q) xv[q] = reinterpret_cast<const float4*>(xr)[q];
}

// A code: clamp(round-half-even(x * inverse), -128, 127) (amd-nv-cpu.ll:1484-1490).
__device__ __forceinline__ int record_code(float x, float inverse) {
    return (int)fminf(fmaxf(__builtin_rintf(x * inverse), -128.f), 127.f);
}

// The 32 codes of a record in registers, written to LDS.
__device__ __forceinline__ void record_codes(const float4 (&xv)[8], float inverse, int8_t* out) {
    uint32_t w[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const float f[4] = {xv[q].x, xv[q].y, xv[q].z, xv[q].w};
        uint32_t word = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) word |= ((uint32_t)record_code(f[k], inverse) & 0xffu) << (8 * k);
        w[q] = word;
    }
    reinterpret_cast<uint4*>(out)[0] = make_uint4(w[0], w[1], w[2], w[3]);
    reinterpret_cast<uint4*>(out)[1] = make_uint4(w[4], w[5], w[6], w[7]);
}

// Record r at a 32 step from its 32 inputs in registers: the extreme, the
// step d[r] and the codes.
__device__ __forceinline__ void record_from_registers(const float4 (&xv)[8], float* d, int8_t* codes, int r) {
    float e = 0.f;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        if (extreme_wins(xv[q].x, e)) e = xv[q].x;
        if (extreme_wins(xv[q].y, e)) e = xv[q].y;
        if (extreme_wins(xv[q].z, e)) e = xv[q].z;
        if (extreme_wins(xv[q].w, e)) e = xv[q].w;
    }
    float inverse, dd;
    step_of(e, inverse, dd);
    record_codes(xv, inverse, codes + r * 32);
    d[r] = dd;
}

// The value of lane ^ OFF (OFF < 32, within the lane's 32-lane half), through
// DPP and the 16-lane swap rather than the LDS crossbar: quad permutations
// for 1 and 2, row shifts by 4 either way for 4, a row rotation by 8 for 8,
// v_permlane16_swap for 16. Each lane then adds exactly the partner
// __shfl_xor would give it, so the butterflies keep their bits.
template <int OFF>
__device__ __forceinline__ float lane_xor(float v) {
    const int iv = __builtin_bit_cast(int, v);
    if constexpr (OFF == 1) return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, iv, 0xB1, 0xf, 0xf, false));
    if constexpr (OFF == 2) return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, iv, 0x4E, 0xf, 0xf, false));
    if constexpr (OFF == 4) {
        const int up = __builtin_amdgcn_update_dpp(0, iv, 0x114, 0xf, 0xf, false);    // row_shr:4 (lane - 4)
        const int down = __builtin_amdgcn_update_dpp(0, iv, 0x104, 0xf, 0xf, false);  // row_shl:4 (lane + 4)
        return __builtin_bit_cast(float, (threadIdx.x & 4) ? up : down);
    }
    if constexpr (OFF == 8) return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, iv, 0x128, 0xf, 0xf, false));
    if constexpr (OFF == 16) {
        float a = v, b = v;
        asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
        return (threadIdx.x & 16) ? a : b;
    }
    static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8 || OFF == 16, "lane_xor: 1, 2, 4, 8 or 16");
    return v;
}

// LDS of one activation row's records: codes[K], d[K/32] and spare words.
__host__ __device__ inline int i8_row_bytes(int K) {
    const int tail = (K >> 5) + ((K + 255) >> 8);
    return K + ((tail + 3) & ~3) * 4;
}

// The Q8 records of MR activation rows (16-byte aligned) from row m0 on, the last of
// the M rows again past it, into LDS, row r at r * i8_row_bytes(K). All rows' records
// are spread over the workgroup at once. Ends with a barrier.
// Step 32: one thread per record scans its 32 inputs. Step 256: recipe's lane v keeps
// the first largest magnitude among input v of the step's 32-value blocks
// (amd-nv-cpu.ll:1408-1440): 32 lanes per step each hold those inputs, take the extreme
// over the lanes by exchanges and code what they hold. With one thread per (step, lane), then one per
// step over 32 LDS reads, then one per record, a row's records took about 3 us of a
// workgroup: Q4_K 1111x2048 at two rows 6.6 -> 4.8 us, Q6_K 14336 x 4096 at
// eight rows, a workgroup a row, 78 -> 61.
template <int MR>
__device__ __forceinline__ void q8_record_rows(const float* __restrict__ x, int64_t ldx, int m0, int M, int K, int step,
                                               uint8_t* lds, int tid) {
    const int blocks = K >> 5, stride = i8_row_bytes(K);
    auto row_of = [&](int r) { return x + (int64_t)(m0 + r < M ? m0 + r : M - 1) * ldx; };
    if (step == 32) {
        for (int i = tid; i < MR * blocks; i += kI8Threads) {
            const int r = MR == 1 ? 0 : i / blocks, b = i - r * blocks;
            float4 xv[8];
            load_record(row_of(r) + b * 32, xv);
            record_from_registers(xv, reinterpret_cast<float*>(lds + r * stride + K), reinterpret_cast<int8_t*>(lds + r * stride), b);
        }
        __syncthreads();
        return;
    }
    constexpr int U = 4, HALVES = kI8Threads / 32;  // steps a half-wave loads at once; half-waves
    const int groups = (blocks + 7) >> 3, items = MR * groups, v = tid & 31;
    const bool whole = (blocks & 7) == 0;
    for (int i0 = tid >> 6 << 1; i0 < items; i0 += U * HALVES) {  // (wave-uniform: the exchanges need every lane)
        float xv[U][8];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (i0 + u * HALVES >= items) break;
            const int i = min(i0 + u * HALVES + ((tid >> 5) & 1), items - 1), r = MR == 1 ? 0 : i / groups, g = i - r * groups;
            const float* const at = row_of(r) + g * 256 + v;
            if (whole) {
#pragma unroll
                for (int b = 0; b < 8; ++b) xv[u][b] = at[b * 32];
            } else {
#pragma unroll
                for (int b = 0; b < 8; ++b) xv[u][b] = g * 8 + b < blocks ? at[b * 32] : 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (i0 + u * HALVES >= items) break;
            const int i = i0 + u * HALVES + ((tid >> 5) & 1), r = MR == 1 ? 0 : i / groups, g = i - r * groups;
            float e = 0.f;
#pragma unroll
            for (int b = 0; b < 8; ++b)  // (zeros past the row's end never win)
                if (fabsf(xv[u][b]) > fabsf(e)) e = xv[u][b];
            float o = lane_xor<16>(e);
            if (extreme_wins(o, e)) e = o;
            o = lane_xor<8>(e);
            if (extreme_wins(o, e)) e = o;
            o = lane_xor<4>(e);
            if (extreme_wins(o, e)) e = o;
            o = lane_xor<2>(e);
            if (extreme_wins(o, e)) e = o;
            o = lane_xor<1>(e);
            if (extreme_wins(o, e)) e = o;
            float inverse, dd;
            step_of(e, inverse, dd);
            if (i >= items) continue;
            int8_t* const codes = reinterpret_cast<int8_t*>(lds + r * stride) + g * 256 + v;
#pragma unroll
            for (int b = 0; b < 8; ++b)
                if (whole || g * 8 + b < blocks) codes[b * 32] = (int8_t)record_code(xv[u][b], inverse);
            if (v < 8 && g * 8 + v < blocks) reinterpret_cast<float*>(lds + r * stride + K)[g * 8 + v] = dd;
        }
    }
    __syncthreads();
}

// Four consecutive 4-bit fields of word n (its low half, or its high half when
// `hi`) as four bytes, field k in byte k.
__device__ __forceinline__ uint32_t spread(uint32_t n, bool hi) {
    const uint32_t a = n & 0x0F0F0F0Fu, b = (n >> 4) & 0x0F0F0F0Fu;
    return __builtin_amdgcn_perm(b, a, hi ? 0x07030602u : 0x05010400u);
}
// Four stored nibbles (XOR 8, layout.h) as the codes q = nibble ^ 8, one per byte.
__device__ __forceinline__ uint32_t nib_codes(uint32_t n, bool hi) { return spread(n, hi) ^ 0x08080808u; }

__device__ __forceinline__ float f16_at(const uint8_t* p) {
    return (float)*reinterpret_cast<const _Float16*>(p);
}

__device__ __forceinline__ int code_sum(const uint4& c) {
    int s = sdot4(0x01010101u, c.x, 0);
    s = sdot4(0x01010101u, c.y, s);
    s = sdot4(0x01010101u, c.z, s);
    return sdot4(0x01010101u, c.w, s);
}

__device__ __forceinline__ int dot4w(uint32_t q0, uint32_t q1, uint32_t q2, uint32_t q3, const uint4& c) {
    int s = sdot4(q0, c.x, 0);
    s = sdot4(q1, c.y, s);
    s = sdot4(q2, c.z, s);
    return sdot4(q3, c.w, s);
}

// get_scale_min_k4 of sub-block g from the superblock's meta words (the
// chunk fields of q4k_field).
__device__ __forceinline__ void q4k_scale_min(const uint4& meta, int g, int& sc, int& m) {
    const uint32_t f = q4k_field(meta, g >> 1);
    sc = (int)bfe(f, 12 * (g & 1), 6);
    m = (int)bfe(f, 12 * (g & 1) + 6, 6);
}

// The dot of 16 stored nibbles (two words, XOR 8) with a slice's record bytes.
__device__ __forceinline__ int q4_dot(uint32_t n0, uint32_t n1, const uint4& c) {
    return dot4w(nib_codes(n0, false), nib_codes(n0, true), nib_codes(n1, false), nib_codes(n1, true), c);
}

// Q6_K slice t (0..3) of a chunk: codes q = l | h << 4, four per word.
__device__ __forceinline__ void q6_words(const ChunkData<Q6_K>& D, int t, uint32_t q[4]) {
    const uint4& lo = D.q[t >> 1];
    const uint32_t n0 = (t & 1) ? lo.z : lo.x, n1 = (t & 1) ? lo.w : lo.y;
    const uint32_t H = word(D.q[2], t);
    const uint32_t h0 = H & 0x33333333u, h1 = (H >> 2) & 0x33333333u;
    q[0] = nib_codes(n0, false) | (spread(h0, false) << 4);
    q[1] = nib_codes(n0, true) | (spread(h0, true) << 4);
    q[2] = nib_codes(n1, false) | (spread(h1, false) << 4);
    q[3] = nib_codes(n1, true) | (spread(h1, true) << 4);
}

__device__ __forceinline__ uint4 record_bytes(const int8_t* xc, int s) {
    return *reinterpret_cast<const uint4*>(xc + s * 16);
}

// Slices per chunk: a chunk is 64 weights (four 16-value slices) except
// Q8_0's 32 (two).
template <int FMT>
constexpr int chunk_slices() {
    return FMT == Q8_0 ? 2 : 4;
}

// The fp32 values of chunk c's slices (build.rs:776-804, 845-848, 909-912),
// slice t of the chunk being slice c * chunk_slices + t of the row.
template <int FMT>
__device__ __forceinline__ void chunk_values(const ChunkData<FMT>& D, int c, const int8_t* xc, const float* xd,
                                             float v[chunk_slices<FMT>()]) {
    if constexpr (FMT == Q4_K) {
        const float d = half_lo(D.meta.x), dmin = half_hi(D.meta.x);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int s = 4 * c + t, j = t >> 1, h = t & 1;
            const int g = 2 * (c & 3) + j;
            const uint4 x = record_bytes(xc, s);
            int sc, m;
            q4k_scale_min(D.meta, g, sc, m);
            const float group_d = d * (float)sc;
            const float group_dmin = dmin * (float)m;
            const float dot_scaled = group_d * (float)q4_dot(word(D.q[j], 2 * h), word(D.q[j], 2 * h + 1), x);
            const float minimum_scaled = group_dmin * (float)code_sum(x);
            const float value = dot_scaled - minimum_scaled;
            v[t] = xd[(c >> 2) * 8 + g] * value;
        }
    } else if constexpr (FMT == Q6_K) {
        const float d = half_lo(D.meta.y);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int s = 4 * c + t;
            const uint4 x = record_bytes(xc, s);
            uint32_t q[4];
            q6_words(D, t, q);
            const int dot_signed = dot4w(q[0], q[1], q[2], q[3], x) - code_sum(x) * 32;
            const float scaled = (float)sbfe(D.meta.x, 8 * t, 8) * (float)dot_signed;
            const float value = xd[s >> 1] * scaled;
            v[t] = d * value;
        }
    } else if constexpr (FMT == Q8_0) {
        const float d = half_lo(D.meta.x);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const uint4 x = record_bytes(xc, 2 * c + t);
            const uint4& w = D.q[t];
            const int sum = code_sum(x);
            const float minimum = 0.f;
            const float dot_scaled = d * (float)dot4w(w.x, w.y, w.z, w.w, x);
            const float minimum_scaled = minimum * (float)sum;
            const float value = dot_scaled + minimum_scaled;
            v[t] = xd[c] * value;
        }
    } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int s = 4 * c + t, j = t >> 1, h = t & 1;
            const uint4 x = record_bytes(xc, s);
            const float d = j ? half_hi(D.meta.x) : half_lo(D.meta.x);
            const int sum = code_sum(x);
            const int dot = q4_dot(word(D.q[j], 2 * h), word(D.q[j], 2 * h + 1), x) - sum * 8;
            const float minimum = 0.f;
            const float dot_scaled = d * (float)dot;
            const float minimum_scaled = minimum * (float)sum;
            const float value = dot_scaled + minimum_scaled;
            v[t] = xd[2 * c + j] * value;
        }
    }
}

struct I8Launch {
    Planes P;
    int64_t rows;
    int K;
    const float* x;
    int64_t ldx;
    float* y;
    int64_t ldy;
    int M;
    int step;
    int tail;
};

// LDS: the records' codes (K bytes), steps (K/32 floats) and ceil(K/256) spare
// words, then per wave two rows of 256 slice values.
__device__ __forceinline__ void stage_records(const I8Launch& p, int step, int8_t*& xc, float*& xd, float*& rowbuf) {
    extern __shared__ __align__(16) uint8_t i8_lds[];
    xc = reinterpret_cast<int8_t*>(i8_lds);
    xd = reinterpret_cast<float*>(i8_lds + p.K);
    const int tail_floats = (p.K >> 5) + ((p.K + 255) >> 8);
    rowbuf = xd + ((tail_floats + 3) & ~3) + ((int)threadIdx.x >> 6) * 512;
    q8_record_rows<1>(p.x, p.ldx, (int)blockIdx.y, p.M, p.K, step, i8_lds, (int)threadIdx.x);
}

// Exact int sums over the four lanes of a quad (one 256-value block).
__device__ __forceinline__ int quad_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false);  // lane ^ 1
    return v + __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, false);  // lane ^ 2
}
__device__ __forceinline__ int lane_int(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float lane_float(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// 16-value slices. Each wave takes two rows at a time, lane i decoding chunk
// i of each 64-chunk pass; the pass's slice values go to the wave's LDS rows,
// where recipe's lane l (lanes 0-31 for the first row, 32-63 for the second)
// adds slices l, l+32, ... in order; the halves' butterflies end each row.
template <int FMT>
__global__ __launch_bounds__(kI8Threads) void int8_slices_kernel(I8Launch p) {
    constexpr int CS = chunk_slices<FMT>();
    int8_t* xc;
    float* xd;
    float* rowbuf;
    const int tid = (int)threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int64_t row0 = (int64_t)blockIdx.x * kI8Rows + 2 * wave;
    const bool live = row0 < p.rows, two = row0 + 1 < p.rows;
    const int slices = p.K >> 4, nch = p.P.nch;
    // At a 32 step with at most one record per thread, the inputs of the
    // thread's record are loaded first and the first pass's weights after
    // them, so that waiting for the inputs leaves the weight loads in flight
    // (the counter of outstanding loads drains in order).
    const int blocks = p.K >> 5;
    const bool early = p.step == 32 && blocks <= kI8Threads;
    ChunkData<FMT> A, B;
    bool have = false;
    if (early) {
        extern __shared__ __align__(16) uint8_t i8_lds[];
        xc = reinterpret_cast<int8_t*>(i8_lds);
        xd = reinterpret_cast<float*>(i8_lds + p.K);
        const int tail_floats = (p.K >> 5) + ((p.K + 255) >> 8);
        rowbuf = xd + ((tail_floats + 3) & ~3) + wave * 512;
        float4 xv[8];
        if (tid < blocks) load_record(p.x + (int64_t)blockIdx.y * p.ldx + tid * 32, xv);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        if (live && lane < nch) {
            load_chunk<FMT>(p.P, row0, lane, A);
            if (two) load_chunk<FMT>(p.P, row0 + 1, lane, B);
            have = true;
        }
        if (tid < blocks) record_from_registers(xv, xd, xc, tid);
        __syncthreads();
    } else {
        stage_records(p, p.step, xc, xd, rowbuf);
    }
    if (!live) return;
    const int mine = lane >> 5;  // which of the two rows this lane sums
    float acc = 0.f;
    for (int c0 = 0; c0 < nch; c0 += 64) {
        const int c = c0 + lane;
        if (c < nch && !(have && c0 == 0)) {
            load_chunk<FMT>(p.P, row0, c, A);
            if (two) load_chunk<FMT>(p.P, row0 + 1, c, B);
        }
        if (c < nch) {
            float va[CS], vb[CS] = {};
            chunk_values<FMT>(A, c, xc, xd, va);
            if (two) chunk_values<FMT>(B, c, xc, xd, vb);
#pragma unroll
            for (int t = 0; t < CS; ++t) {
                rowbuf[lane * CS + t] = va[t];
                rowbuf[256 + lane * CS + t] = vb[t];
            }
        }
        __builtin_amdgcn_wave_barrier();
        const int base = c0 * CS;  // first slice of the pass
        const float* mybuf = rowbuf + 256 * mine;
        const int l = lane & 31;
#pragma unroll
        for (int j = 0; j < 2 * CS; ++j) {
            const int s = base + l + 32 * j;
            if (s < slices) acc = acc + mybuf[l + 32 * j];
        }
        __builtin_amdgcn_wave_barrier();
    }
    acc = acc + lane_xor<16>(acc);
    acc = acc + lane_xor<8>(acc);
    acc = acc + lane_xor<4>(acc);
    acc = acc + lane_xor<2>(acc);
    acc = acc + lane_xor<1>(acc);
    if ((lane & 31) == 0 && (mine == 0 || two)) p.y[(int64_t)blockIdx.y * p.ldy + row0 + mine] = acc;
}

// Batches: MR activation rows per workgroup, whose records stand in LDS side by side;
// each wave reads and unpacks its two weight rows once for all of them. Every output sees
// the operations of the one-row kernel in their order. Step 32, us at 4 / 8 rows with a
// workgroup per activation row -> four rows a workgroup: Q4_K 4096->14336 27.7 / 52.5 ->
// 22.3 / 36.2, Q6_K 33.5 / 62.0 -> 21.2 / 32.3, Q4_0 33.2 / 61.6 -> 24.4 / 35.5; Q8_0
// 5120x5120 14.3 / 25.9 -> 13.1 (two rows) / 20.5. Bound by VALU issue (0.68 of a SIMD's
// time on Q4_K 4096->14336 at four rows) and by the records' LDS reads and the sums'
// round trip, whose bank conflicts alone take a quarter of a CU's time.
template <int MR>
__device__ __forceinline__ float* stage_record_rows(const I8Launch& p, int step, uint8_t* lds) {
    q8_record_rows<MR>(p.x, p.ldx, (int)blockIdx.y * MR, p.M, p.K, step, lds, (int)threadIdx.x);
    return reinterpret_cast<float*>(lds + MR * i8_row_bytes(p.K)) + ((int)threadIdx.x >> 6) * 512;
}

template <int FMT, int MR>
__global__ __launch_bounds__(kI8Threads) void int8_slices_rows_kernel(I8Launch p) {
    constexpr int CS = chunk_slices<FMT>();
    extern __shared__ __align__(16) uint8_t i8_lds[];
    float* const rowbuf = stage_record_rows<MR>(p, p.step, i8_lds);
    const int stride = i8_row_bytes(p.K), wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    const int64_t row0 = (int64_t)blockIdx.x * kI8Rows + 2 * wave;
    if (row0 >= p.rows) return;
    const bool two = row0 + 1 < p.rows;
    const int slices = p.K >> 4, nch = p.P.nch, mine = lane >> 5, l = lane & 31;
    float acc[MR];
#pragma unroll
    for (int r = 0; r < MR; ++r) acc[r] = 0.f;
    for (int c0 = 0; c0 < nch; c0 += 64) {
        const int c = c0 + lane;
        ChunkData<FMT> A, B;
        if (c < nch) {
            load_chunk<FMT>(p.P, row0, c, A);
            if (two) load_chunk<FMT>(p.P, row0 + 1, c, B);
        }
        const int base = c0 * CS;  // first slice of the pass
        const float* mybuf = rowbuf + 256 * mine;
#pragma unroll
        for (int r = 0; r < MR; ++r) {
            if (c < nch) {
                const int8_t* xc = reinterpret_cast<const int8_t*>(i8_lds + r * stride);
                const float* xd = reinterpret_cast<const float*>(i8_lds + r * stride + p.K);
                float va[CS], vb[CS] = {};
                chunk_values<FMT>(A, c, xc, xd, va);
                if (two) chunk_values<FMT>(B, c, xc, xd, vb);
#pragma unroll
                for (int t = 0; t < CS; ++t) {
                    rowbuf[lane * CS + t] = va[t];
                    rowbuf[256 + lane * CS + t] = vb[t];
                }
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int j = 0; j < 2 * CS; ++j) {
                const int s = base + l + 32 * j;
                if (s < slices) acc[r] = acc[r] + mybuf[l + 32 * j];
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
#pragma unroll
    for (int r = 0; r < MR; ++r) {
        float v = acc[r];
        v = v + lane_xor<16>(v);
        v = v + lane_xor<8>(v);
        v = v + lane_xor<4>(v);
        v = v + lane_xor<2>(v);
        v = v + lane_xor<1>(v);
        const int m = (int)blockIdx.y * MR + r;
        if (l == 0 && (mine == 0 || two) && m < p.M) p.y[(int64_t)m * p.ldy + row0 + mine] = v;
    }
}

// Q4_K at a 256 step (amd-nv-cpu.ll:1545-1733). Lane i decodes chunk i of a
// pass: quarter i%4 of block i/4, whose two sub-blocks give the quarter's
// exact ints (scale times dot, minimum times code sum). Each pass leaves, per
// row and block, the four quarters' ints and the block's two scales in the
// wave's LDS row (ten words per block); lanes 0 and 1 (first row) and 32 and
// 33 (second row) then run the acc and accmin fma chains in block order.
__device__ __forceinline__ void q4k256_ints(const ChunkData<Q4_K>& D, int c, const int8_t* xc, const float* xd,
                                            float* out) {
    int dq = 0, mq = 0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int g = 2 * (c & 3) + j;
        int sc, m;
        q4k_scale_min(D.meta, g, sc, m);
        const uint4 x0 = record_bytes(xc, 4 * c + 2 * j), x1 = record_bytes(xc, 4 * c + 2 * j + 1);
        dq += sc * (q4_dot(word(D.q[j], 0), word(D.q[j], 1), x0) + q4_dot(word(D.q[j], 2), word(D.q[j], 3), x1));
        mq += m * (code_sum(x0) + code_sum(x1));
    }
    float* blk = out + (c & 63) / 4 * 10;
    blk[2 * (c & 3)] = __builtin_bit_cast(float, dq);
    blk[2 * (c & 3) + 1] = __builtin_bit_cast(float, mq);
    if ((c & 3) == 0) {
        const float d8 = xd[(c >> 2) * 8];
        blk[8] = half_lo(D.meta.x) * d8;
        blk[9] = half_hi(D.meta.x) * d8;
    }
}

__global__ __launch_bounds__(kI8Threads) void int8_q4k256_kernel(I8Launch p) {
    int8_t* xc;
    float* xd;
    float* rowbuf;
    stage_records(p, 256, xc, xd, rowbuf);
    const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    const int64_t row0 = (int64_t)blockIdx.x * kI8Rows + 2 * wave;
    if (row0 >= p.rows) return;
    const bool two = row0 + 1 < p.rows;
    const int m = (int)blockIdx.y;
    const bool whole = m >= p.M - (p.M & 3) || (p.tail && m == p.M - 1);
    const int nch = p.P.nch;
    const int chain = lane & 1;                        // 0: acc, 1: accmin
    const float* mine = rowbuf + 256 * (lane >> 5);  // the row this lane's chain belongs to
    float acc = 0.f;
    for (int c0 = 0; c0 < nch; c0 += 64) {
        const int c = c0 + lane;
        ChunkData<Q4_K> A, B;
        if (c < nch) {
            load_chunk<Q4_K>(p.P, row0, c, A);
            if (two) load_chunk<Q4_K>(p.P, row0 + 1, c, B);
            q4k256_ints(A, c, xc, xd, rowbuf);
            if (two) q4k256_ints(B, c, xc, xd, rowbuf + 256);
        }
        __builtin_amdgcn_wave_barrier();
        if ((lane & 31) < 2) {
            const int blocks = min(16, (nch - c0) >> 2);
            for (int b = 0; b < blocks; ++b) {
                const float* blk = mine + b * 10;
                const float s = blk[8 + chain];
                if (whole) {
                    const int w = (__builtin_bit_cast(int, blk[chain]) + __builtin_bit_cast(int, blk[2 + chain])) +
                                  (__builtin_bit_cast(int, blk[4 + chain]) + __builtin_bit_cast(int, blk[6 + chain]));
                    acc = fmaf((float)w, s, acc);
                } else {
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc = fmaf((float)__builtin_bit_cast(int, blk[2 * q + chain]), s, acc);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    const float other = lane_xor<1>(acc);
    if (lane == 0) p.y[(int64_t)m * p.ldy + row0] = acc - other;
    if (lane == 32 && two) p.y[(int64_t)m * p.ldy + row0 + 1] = acc - other;
}

// Q6_K at a 256 step (amd-nv-cpu.ll:1836-2031, build.rs:871-884). Lane i
// decodes chunk i of a pass: quarter i%4 of block i/4, slices 4(i%4)+t. Chain
// k takes word k%4 of the slices with parity k/4 (the four-value words at 4k
// of every 32-value group) and -32 times the scaled code sums of group k. The
// quads' exact sums give each block's eight chain ints, left with the block's
// scale in the wave's LDS row (nine words per block); lanes 0-7 (first row)
// and 32-39 (second row) each run one chain's fmas in block order.
__device__ __forceinline__ void q6k256_ints(const ChunkData<Q6_K>& D, int c, const int8_t* xc, const float* xd,
                                            float* out) {
    const int qq = c & 3;
    int I[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int G0 = 0, G1 = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const uint4 x = record_bytes(xc, 4 * c + t);
        const int sc = sbfe(D.meta.x, 8 * t, 8);
        uint32_t q[4];
        q6_words(D, t, q);
        I[(t & 1) * 4 + 0] += sc * sdot4(q[0], x.x, 0);
        I[(t & 1) * 4 + 1] += sc * sdot4(q[1], x.y, 0);
        I[(t & 1) * 4 + 2] += sc * sdot4(q[2], x.z, 0);
        I[(t & 1) * 4 + 3] += sc * sdot4(q[3], x.w, 0);
        const int g = -32 * (sc * code_sum(x));
        if (t < 2)
            G0 += g;
        else
            G1 += g;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        I[k] += (k == 2 * qq ? G0 : 0) + (k == 2 * qq + 1 ? G1 : 0);
        I[k] = quad_sum(I[k]);
    }
    if (qq == 0) {
        float* blk = out + (c & 63) / 4 * 9;
#pragma unroll
        for (int k = 0; k < 8; ++k) blk[k] = __builtin_bit_cast(float, I[k]);
        blk[8] = xd[(c >> 2) * 8] * half_lo(D.meta.y);
    }
}

__global__ __launch_bounds__(kI8Threads) void int8_q6k256_kernel(I8Launch p) {
    int8_t* xc;
    float* xd;
    float* rowbuf;
    stage_records(p, 256, xc, xd, rowbuf);
    const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    const int64_t row0 = (int64_t)blockIdx.x * kI8Rows + 2 * wave;
    if (row0 >= p.rows) return;
    const bool two = row0 + 1 < p.rows;
    const int nch = p.P.nch;
    const int chain = lane & 7;
    const float* mine = rowbuf + 256 * (lane >> 5);
    float f = 0.f;
    for (int c0 = 0; c0 < nch; c0 += 64) {
        const int c = c0 + lane;
        ChunkData<Q6_K> A, B;
        if (c < nch) {  // whole quads: nch is a multiple of four
            load_chunk<Q6_K>(p.P, row0, c, A);
            if (two) load_chunk<Q6_K>(p.P, row0 + 1, c, B);
            q6k256_ints(A, c, xc, xd, rowbuf);
            if (two) q6k256_ints(B, c, xc, xd, rowbuf + 256);
        }
        __builtin_amdgcn_wave_barrier();
        if ((lane & 31) < 8) {
            const int blocks = min(16, (nch - c0) >> 2);
            for (int b = 0; b < blocks; ++b) {
                const float* blk = mine + b * 9;
                f = fmaf(blk[8], (float)__builtin_bit_cast(int, blk[chain]), f);
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    const float t = f + lane_xor<4>(f);
    const float u = t + lane_xor<2>(t);
    const float total = u + lane_xor<1>(u);
    if (lane == 0) p.y[(int64_t)blockIdx.y * p.ldy + row0] = total;
    if (lane == 32 && two) p.y[(int64_t)blockIdx.y * p.ldy + row0 + 1] = total;
}

// Batches at a 256 step (Q4_K, Q6_K): MR activation rows per workgroup. A wave reads its
// two weight rows once for all of them, and the serial chains of every (activation row,
// weight row) run side by side in one pass over the blocks: sixteen lanes of Q4_K's, 64
// of Q6_K's at four rows, where the one-row kernels keep four and sixteen busy for the
// same round trips. Every chain sees the one-row kernels' operations in their order.
// Bound by the staged codes' LDS reads and the chains. Us at 4 / 8 rows:
// Q4_K 4096->14336 31 / 58 -> 26.4 / 43.6, Q6_K 32 / 61 -> 23 / 37.
template <int FMT>
constexpr int block_words() {  // a block's ints and scales in LDS
    return FMT == Q4_K ? 10 : 9;
}
template <int FMT>
constexpr int slot_pitch() {  // words of 16 blocks, such that the slots' chains read different banks
    return FMT == Q4_K ? 162 : 152;
}
template <int FMT>
constexpr int block_wave_bytes(int mr) {
    return 2 * mr * slot_pitch<FMT>() * 4;
}
template <int FMT, int MR>
__global__ __launch_bounds__(kI8Threads) void int8_blocks_rows_kernel(I8Launch p) {
    constexpr int BW = block_words<FMT>(), SP = slot_pitch<FMT>(), CH = FMT == Q4_K ? 2 : 8;
    extern __shared__ __align__(16) uint8_t i8_lds[];
    stage_record_rows<MR>(p, 256, i8_lds);
    const int stride = i8_row_bytes(p.K), wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    float* const buf = reinterpret_cast<float*>(i8_lds + MR * stride) + wave * (2 * MR * SP);
    const int64_t row0 = (int64_t)blockIdx.x * kI8Rows + 2 * wave;
    if (row0 >= p.rows) return;
    const bool two = row0 + 1 < p.rows;
    const int nch = p.P.nch;
    // this lane's chain: activation row m0 + slot / 2, weight row row0 + slot % 2
    const int chain = lane % CH, slot = lane / CH, m = (int)blockIdx.y * MR + (slot >> 1);
    const bool whole = m >= p.M - (p.M & 3) || (p.tail && m == p.M - 1);
    const float* const mine = buf + slot * SP;
    float acc = 0.f;
    for (int c0 = 0; c0 < nch; c0 += 64) {
        const int c = c0 + lane;
        if (c < nch) {  // whole quads: nch is a multiple of four
            ChunkData<FMT> D[2];
            load_chunk<FMT>(p.P, row0, c, D[0]);
            load_chunk<FMT>(p.P, two ? row0 + 1 : row0, c, D[1]);
#pragma unroll
            for (int r = 0; r < MR; ++r) {
                const int8_t* xc = reinterpret_cast<const int8_t*>(i8_lds + r * stride);
                const float* xd = reinterpret_cast<const float*>(i8_lds + r * stride + p.K);
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    if constexpr (FMT == Q4_K) q4k256_ints(D[w], c, xc, xd, buf + (2 * r + w) * SP);
                    else q6k256_ints(D[w], c, xc, xd, buf + (2 * r + w) * SP);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
        if (slot < 2 * MR) {
            const int blocks = min(16, (nch - c0) >> 2);
#pragma unroll 4
            for (int b = 0; b < blocks; ++b) {
                const float* blk = mine + b * BW;
                if constexpr (FMT == Q4_K) {
                    const float s = blk[8 + chain];
                    int q[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) q[i] = __builtin_bit_cast(int, blk[2 * i + chain]);
                    if (whole) {
                        acc = fmaf((float)((q[0] + q[1]) + (q[2] + q[3])), s, acc);
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc = fmaf((float)q[i], s, acc);
                    }
                } else {
                    acc = fmaf(blk[8], (float)__builtin_bit_cast(int, blk[chain]), acc);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    float v;
    if constexpr (FMT == Q4_K) {
        v = acc - lane_xor<1>(acc);
    } else {
        const float t = acc + lane_xor<4>(acc);
        const float u = t + lane_xor<2>(t);
        v = u + lane_xor<1>(u);
    }
    if (chain == 0 && slot < 2 * MR && m < p.M && (two || !(slot & 1))) p.y[(int64_t)m * p.ldy + row0 + (slot & 1)] = v;
}

// The records of one row, staged as the products stage them, then copied out.
__global__ __launch_bounds__(kI8Threads) void q8_records_kernel(const float* x, int K, int step, float* d,
                                                                int8_t* codes) {
    extern __shared__ __align__(16) uint8_t i8_lds[];
    int8_t* xc = reinterpret_cast<int8_t*>(i8_lds);
    float* xd = reinterpret_cast<float*>(i8_lds + K);
    q8_record_rows<1>(x, 0, 0, 1, K, step, i8_lds, (int)threadIdx.x);
    for (int i = (int)threadIdx.x; i < K; i += kI8Threads) codes[i] = xc[i];
    for (int i = (int)threadIdx.x; i < (K >> 5); i += kI8Threads) d[i] = xd[i];
}

}  // namespace

// codes, steps, spare words (rounded up to 16 bytes), then 2 KiB of
// slice values per wave.
size_t int8_lds_bytes(int64_t cols) {
    const size_t tail = (size_t)(cols / 32) + (size_t)((cols + 255) / 256);
    return (size_t)cols + ((tail + 3) & ~size_t(3)) * 4 + (size_t)(kI8Threads / 64) * 2048;
}

// Activation rows per workgroup of a batch: one, two or four, whichever costs least. A
// CU's workgroups (two at least: fewer take as long) cost w of a one-row workgroup's time
// each, w as measured on batches of 15 rows and more (us, one / two / four rows a
// workgroup, step 32: Q4_K 4096->14336 at 64 rows 378 / 358 / 264, Q6_K 548 / 415 / 295;
// four cost more on longer rows, whose records leave room for fewer workgroups). One-row
// workgroups of Q8_0 wait for memory once the weight outgrows the eight L2s of 4 MB (486 /
// 310 / 220). Last groups may have places empty: Q6_K 25600x1024 at three rows 39.9 / 39.9 /
// 28.9, Q8_0 14336x4096 at five 37.8 / 31.1 / 30.2. Over 4,088 batches the choice takes
// 0.7 % more than the best of the three on average and is behind one row a workgroup by
// more than 3 % in 61 (12 % at most). The records and the waves' buffers stay within 64 KiB
// of LDS. RQMV_I8_ROWS=1/2/4 overrides it for tuning.
static int int8_rows(int fmt, int step, int M, int64_t rows, int K, size_t weight_bytes, int cus, size_t (*wave_bytes)(int)) {
    auto fits = [&](int mr) { return (size_t)mr * i8_row_bytes(K) + (size_t)(kI8Threads / 64) * wave_bytes(mr) <= 65536; };
    int mr = 1;
    const char* env = getenv("RQMV_I8_ROWS");
    if (env && *env) {
        mr = atoi(env) >= 4 ? 4 : atoi(env) >= 2 ? 2 : 1;
        while (mr > 1 && !fits(mr)) mr >>= 1;
        return mr;
    }
    const bool s32 = step == 32;
    float two = 0.f, four = 0.f;
    switch (fmt) {
        case Q4_0: two = s32 ? 1.92f : 1.90f, four = s32 ? 3.00f : 3.10f; break;
        case Q4_K: two = s32 ? 1.85f : 1.50f, four = s32 ? 2.70f : 2.75f; break;
        case Q8_0: two = s32 ? 1.65f : 1.70f, four = s32 ? 2.75f : 3.00f; break;
        default: two = s32 ? 1.52f : 1.62f, four = s32 ? 2.15f : 2.70f; break;
    }
    if (fmt == Q8_0 && weight_bytes > (24u << 20)) two *= 0.77f, four *= 0.69f;
    four *= 1.f + 0.1f * ((float)K / 4096.f - 1.f);
    const int64_t tiles = (rows + kI8Rows - 1) / kI8Rows;
    auto cost = [&](int n, float w) {
        const int64_t per_cu = (tiles * ((M + n - 1) / n) + cus - 1) / cus;
        return w * (float)(per_cu > 2 ? per_cu : 2);
    };
    float best = cost(1, 1.f);
    if (M >= 2 && fits(2) && cost(2, two) < best) mr = 2, best = cost(2, two);
    if (M >= 3 && fits(4) && cost(4, four) < best) mr = 4;
    return mr;
}

template <int FMT>
static hipError_t launch_blocks(const I8Launch& p, int cus, hipStream_t stream) {
    auto wave_bytes = [](int mr) -> size_t { return block_wave_bytes<FMT>(mr); };
    const int mr = int8_rows(FMT, 256, p.M, p.rows, p.K, p.P.bytes, cus, wave_bytes);
    const dim3 grid((unsigned)((p.rows + kI8Rows - 1) / kI8Rows), (unsigned)((p.M + mr - 1) / mr));
    size_t lds = int8_lds_bytes(p.K);
    void (*kernel)(I8Launch) = FMT == Q4_K ? int8_q4k256_kernel : int8_q6k256_kernel;
    if (mr > 1) {
        lds = (size_t)mr * i8_row_bytes(p.K) + (size_t)(kI8Threads / 64) * wave_bytes(mr);
        kernel = mr == 4 ? int8_blocks_rows_kernel<FMT, 4> : int8_blocks_rows_kernel<FMT, 2>;
    }
    hipLaunchKernelGGL(kernel, grid, dim3(kI8Threads), lds, stream, p);
    return hipGetLastError();
}

template <int FMT>
static hipError_t launch_slices(const I8Launch& p, int cus, hipStream_t stream) {
    const int mr = int8_rows(FMT, p.step, p.M, p.rows, p.K, p.P.bytes, cus, [](int) -> size_t { return 2048; });
    const dim3 grid((unsigned)((p.rows + kI8Rows - 1) / kI8Rows), (unsigned)((p.M + mr - 1) / mr));
    size_t lds = int8_lds_bytes(p.K);
    auto kernel = int8_slices_kernel<FMT>;
    if (mr > 1) {
        lds = (size_t)mr * i8_row_bytes(p.K) + (size_t)(kI8Threads / 64) * 2048;
        kernel = mr == 4 ? int8_slices_rows_kernel<FMT, 4> : int8_slices_rows_kernel<FMT, 2>;
    }
    hipLaunchKernelGGL(kernel, grid, dim3(kI8Threads), lds, stream, p);
    return hipGetLastError();
}

hipError_t launch_matvec_int8(int fmt, const Planes& P, int64_t rows, int K, const float* x, int M, int64_t ldx,
                              float* y, int64_t ldy, int step, int tail, int cus, hipStream_t stream) {
    I8Launch p{P, rows, K, x, ldx, y, ldy, M, step, tail};
    if (step == 256 && fmt == Q4_K) return launch_blocks<Q4_K>(p, cus, stream);
    if (step == 256 && fmt == Q6_K) return launch_blocks<Q6_K>(p, cus, stream);
    switch (fmt) {
        case Q4_K: return launch_slices<Q4_K>(p, cus, stream);
        case Q6_K: return launch_slices<Q6_K>(p, cus, stream);
        case Q8_0: return launch_slices<Q8_0>(p, cus, stream);
        case Q4_0: return launch_slices<Q4_0>(p, cus, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_q8_records(const float* x, int K, int step, float* d, int8_t* codes, hipStream_t stream) {
    hipLaunchKernelGGL(q8_records_kernel, dim3(1), dim3(kI8Threads), int8_lds_bytes(K), stream, x, K, step, d, codes);
    return hipGetLastError();
}

}  // namespace rq
