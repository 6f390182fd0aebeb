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
    const size_t lds = (size_t)WK * RT * MT * 64 * sizeof(f4_t);  // (at most 64 KiB)
    auto kernel = matvec_mfma_direct<FMT, RT, MT, PACK>;
    if (ev0 || ev1)
        hipExtLaunchKernelGGL(kernel, grid, dim3(64 * WK), (uint32_t)lds, stream, ev0, ev1, 0u, p, M, x_bytes, WK, groups);
    else
        hipLaunchKernelGGL(kernel, grid, dim3(64 * WK), lds, stream, p, M, x_bytes, WK, groups);
    return hipGetLastError();
}

// Shape. Up to eight activation rows take the packed operand; above, up to four
// tiles of 16 rows per wave, in groups as even as they come. Two row tiles per
// wave share the activations' loads and conversions once there is more than one
// row tile per CU (kernel us, fp32 x, one against two row tiles per wave: Q4_K
// 4096->14336 at 5 / 16 / 32 rows 36.2 / 42.9 / 67.3 -> 27.2 / 28.6 / 40.3, Q8_0
// 5120x5120 at 16 / 32 rows 29.1 / 46.0 -> 20.3 / 30.5; with 256 row tiles one
// is better: Q4_K 4096x4096 at 5 / 16 rows 12.8 / 14.1 against 15.4 / 15.6).
// Eight waves split K, or four where the workgroups alone fill the chip three
// times over (Q4_K 4096->14336 at 5 rows 29.3 -> 27.2). RQMV_DIRECT_RT and
// RQMV_DIRECT_WK override them for tuning.
template <int FMT>
static hipError_t launch_direct(const MvParams& p, int M, uint32_t x_bytes, int cus, hipStream_t stream, hipEvent_t ev0,
                                hipEvent_t ev1) {
    const int tiles = (M + 15) / 16, groups = (tiles + 3) / 4, mt = (tiles + groups - 1) / groups;
    const int64_t row_tiles = (p.rows + 15) / 16;
    const int rt = env_or("RQMV_DIRECT_RT", row_tiles * groups > cus ? 2 : 1) == 2 ? 2 : 1;
    int wk = env_or("RQMV_DIRECT_WK", (row_tiles + rt - 1) / rt * groups >= (int64_t)3 * cus / 2 ? 4 : 8);
    wk = wk < 1 ? 1 : wk > kDirectMaxWaves ? kDirectMaxWaves : wk;
#define RQ_DIRECT(MT, PACK)                                                                         \
    return rt == 2 ? launch_direct_one<FMT, 2, MT, PACK>(p, M, x_bytes, wk, stream, ev0, ev1)       \
                   : launch_direct_one<FMT, 1, MT, PACK>(p, M, x_bytes, wk, stream, ev0, ev1)
    if (M <= 8) RQ_DIRECT(1, true);
    switch (mt) {
        case 1: RQ_DIRECT(1, false);
        case 2: RQ_DIRECT(2, false);
        case 3: RQ_DIRECT(3, false);
        default: RQ_DIRECT(4, false);
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
