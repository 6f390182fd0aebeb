// Quantized products on the matrix cores for fp32 activations: launch planning
// of mfma_direct.h. Built without the matrix-core VGPR form.
#include "mfma_direct.h"

namespace rq {

static int env_or(const char* name, int fallback) {
    const char* v = getenv(name);
    return v && *v ? atoi(v) : fallback;
}

template <int FMT, int RT, int MT, bool PACK>
static hipError_t launch_direct_one(const MvParams& p, int M, uint32_t x_bytes, int WK, hipStream_t stream,
                                    hipEvent_t ev0, hipEvent_t ev1) {
    const int rows = PACK ? 8 : 16 * MT;
    const int groups = (M + rows - 1) / rows;
    const int64_t wgs = (p.rows + 16 * RT - 1) / (16 * RT) * groups;
    if (wgs > 0x7FFFFFFF) return hipErrorInvalidValue;
    const dim3 grid((unsigned)wgs);
    const size_t lds = (size_t)WK * RT * MT * 64 * sizeof(f4_t);  // (at most 48 KiB)
    auto kernel = matvec_mfma_direct<FMT, RT, MT, PACK>;
    if (ev0 || ev1)
        hipExtLaunchKernelGGL(kernel, grid, dim3(64 * WK), (uint32_t)lds, stream, ev0, ev1, 0u, p, M, x_bytes, WK, groups);
    else
        hipLaunchKernelGGL(kernel, grid, dim3(64 * WK), lds, stream, p, M, x_bytes, WK, groups);
    return hipGetLastError();
}

// Shape. Up to eight activation rows take the packed operand; above, up to three
// tiles of 16 rows per wave (a fourth cost more than a further group wherever it was
// timed: Q4_K 14336->1024 at 64 rows 110 us as one group of four, 62 as two of two), in
// groups as even as they come. Two row tiles per wave share the activations' loads and
// conversions once there is more than one row tile and group per CU (us, fp32 x, one
// against two row tiles per wave: Q4_K 4096->14336 at 5 / 16 / 32 rows 36.2 / 42.9 / 67.3 ->
// 27.2 / 28.6 / 40.3, Q8_0 5120x5120 at 16 / 32 rows 29.1 / 46.0 -> 20.3 / 30.5; with 256
// row tiles one is better: Q4_K 4096x4096 at 5 / 16 rows 12.8 / 14.1 against 15.4 / 15.6).
// Eight waves split K, or four from three workgroups per two CUs on (Q4_K 4096->14336 at
// 5 rows 29.3 -> 27.2). RQMV_DIRECT_RT and RQMV_DIRECT_WK override them for tuning.
struct DirectShape {
    int rt, mt, wk;
    int64_t wgs;
};
static DirectShape direct_shape(int M, int64_t rows, int cus) {
    const int tiles = (M + 15) / 16, groups = M <= 8 ? 1 : (tiles + 2) / 3;
    const int64_t row_tiles = (rows + 15) / 16;
    DirectShape s;
    s.mt = (tiles + groups - 1) / groups;
    s.rt = env_or("RQMV_DIRECT_RT", row_tiles * groups > cus ? 2 : 1) == 2 ? 2 : 1;
    s.wgs = (row_tiles + s.rt - 1) / s.rt * groups;
    const int wk = env_or("RQMV_DIRECT_WK", s.wgs >= (int64_t)3 * cus / 2 ? 4 : 8);
    s.wk = wk < 1 ? 1 : wk > kDirectMaxWaves ? kDirectMaxWaves : wk;
    return s;
}

// Estimated time (us), for the choice between this form and the tiled one: 3 us and,
// for every workgroup a CU takes, what a step of 256 values costs times the steps of its
// waves (all of them as many as the longest; where some have none, half of those: the
// others run the faster). Fitted to 1,918 products of 17 to 512 rows (within 7 to 9 % of
// the estimates, root mean square), less 2 %, so that ties go to this form; activation
// rows that only repeat the last cost half of the others.
float direct_us(int fmt, int M, int64_t rows, int64_t cols, int cus) {
    struct Cost {
        float one;        // us a step and activation tile, one row tile per wave
        float two, tile;  // us a step, and a step and activation tile, two row tiles per wave
    };
    const Cost c = fmt == Q4_0   ? Cost{0.45f, 0.27f, 0.41f}
                   : fmt == Q4_K ? Cost{0.47f, 0.37f, 0.40f}
                   : fmt == Q8_0 ? Cost{0.50f, 0.28f, 0.47f}
                                 : Cost{0.51f, 0.60f, 0.41f};
    const DirectShape s = direct_shape(M, rows, cus);
    const int groups = (M + 16 * s.mt - 1) / (16 * s.mt);
    const float tiles = 0.5f * ((float)s.mt + (float)M / (16.f * (float)groups));
    const int64_t unit = fmt == Q8_0 ? 128 : 256, steps = (cols + unit - 1) / unit;
    const float longest = steps < s.wk ? 0.5f * (float)(steps + s.wk) : (float)((steps + s.wk - 1) / s.wk * s.wk);
    const float each = longest * (float)unit / 256.f;
    return 3.f + (float)((s.wgs + cus - 1) / cus) * each * (s.rt == 1 ? c.one * tiles : c.two + c.tile * tiles);
}

template <int FMT>
static hipError_t launch_direct(const MvParams& p, int M, uint32_t x_bytes, int cus, hipStream_t stream, hipEvent_t ev0,
                                hipEvent_t ev1) {
    const DirectShape s = direct_shape(M, p.rows, cus);
#define RQ_DIRECT(MT, PACK)                                                                         \
    return s.rt == 2 ? launch_direct_one<FMT, 2, MT, PACK>(p, M, x_bytes, s.wk, stream, ev0, ev1)   \
                   : launch_direct_one<FMT, 1, MT, PACK>(p, M, x_bytes, s.wk, stream, ev0, ev1)
    if (M <= 8) RQ_DIRECT(1, true);
    switch (s.mt) {
        case 1: RQ_DIRECT(1, false);
        case 2: RQ_DIRECT(2, false);
        default: RQ_DIRECT(3, false);
    }
#undef RQ_DIRECT
}

hipError_t launch_matvec_f32(int fmt, const MvParams& p, int M, int cus, hipStream_t stream, hipEvent_t ev0,
                             hipEvent_t ev1) {
    const int64_t x_bytes = ((int64_t)(M - 1) * p.ldx + p.K) * 4;
    if (M < 1 || x_bytes >= (int64_t)kOobOffset) return hipErrorInvalidValue;
    switch (fmt) {
        case Q4_0: return launch_direct<Q4_0>(p, M, (uint32_t)x_bytes, cus, stream, ev0, ev1);
        case Q4_K: return launch_direct<Q4_K>(p, M, (uint32_t)x_bytes, cus, stream, ev0, ev1);
        case Q8_0: return launch_direct<Q8_0>(p, M, (uint32_t)x_bytes, cus, stream, ev0, ev1);
        case Q6_K: return launch_direct<Q6_K>(p, M, (uint32_t)x_bytes, cus, stream, ev0, ev1);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace rq
