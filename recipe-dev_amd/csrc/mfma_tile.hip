// Launch planning of the tiled matrix-core products (mfma_tile.h).
#include "mfma_tile.h"

namespace rq {

template <int FMT, int RT, int MT, int WN, int WK, bool XF32>
static hipError_t launch_tile_one(const MvParams& p, int M, uint32_t x_bytes, hipStream_t stream, hipEvent_t ev0,
                                  hipEvent_t ev1) {
    const int64_t n_tiles = (p.rows + 16 * RT * WN - 1) / (16 * RT * WN);
    const int groups = (M + 16 * MT - 1) / (16 * MT);
    const int64_t wgs = (n_tiles + 7) / 8 * 8 * groups;
    if (wgs > 0x7FFFFFFF) return hipErrorInvalidValue;
    constexpr size_t lds = (size_t)WK * TileCfg<FMT, MT, XF32>::LDS;
    static_assert(lds <= 160 * 1024 && (WK == 1 || lds >= (size_t)WN * WK * RT * MT * 1024), "LDS holds the windows and the tiles");
    auto kernel = matvec_mfma_tile<FMT, RT, MT, WN, WK, XF32>;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    if (ev0 || ev1)
        hipExtLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(64 * WN * WK), (uint32_t)lds, stream, ev0, ev1, 0u, p, M,
                              x_bytes, (int)n_tiles, groups);
    else
        hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(64 * WN * WK), lds, stream, p, M, x_bytes, (int)n_tiles, groups);
    return hipGetLastError();
}

// The shapes, and what a step of 256 values of K takes a workgroup in each (us,
// measured with one workgroup per CU at most, less a launch's 4 us): the plan takes
// the shape whose steps, times the rounds of workgroups over the chip, are fewest.
// Kernel us at the shape the plan takes, against the streaming form in launches of
// 32 rows (fp16 x) or the direct form (fp32 x):
//   fp16 x  Q4_K 4096->14336 at 64 / 512 rows 50.6 / 393 -> 29.2 / 114 (528 TFLOP/s)
//           Q4_0 4096->14336 at 512 rows -> 97.4 (617 TFLOP/s)
//           Q6_K 14336->4096 at 128 / 512 rows 161 / 642 -> 78.8 / 173
//           Q8_0 5120x5120 at 64 / 512 rows 41.5 / 341 -> 31.2 / 85.8
//   fp32 x  Q4_K 4096->14336 at 64 / 512 rows 122 / 439 -> 52.7 / 234
//           Q6_K 14336->4096 at 64 / 512 rows 112 / 473 -> 90.2 / 335
// With few workgroups, several ranges of K per workgroup (x2, x4) make up for the
// rows they take from it: Q6_K 14336->4096 at 64 rows 175 -> 79.5 (fp16 x).
struct TileShape {
    int id, rt, mt, wn, wk;  // mt for fp16 x, half of it for fp32 x
    float step[2][4];        // us per step: [fp32 x][Q4_0, Q4_K, Q8_0, Q6_K]
};
constexpr TileShape kTileShapes[] = {
    {11, 1, 4, 8, 1, {{2.15f, 2.2f, 2.8f, 3.0f}, {2.75f, 2.7f, 3.25f, 3.7f}}},
    {12, 1, 8, 8, 1, {{3.0f, 3.05f, 3.5f, 3.9f}, {3.9f, 4.5f, 4.55f, 5.4f}}},
    {22, 2, 8, 8, 1, {{5.8f, 6.8f, 6.9f, 9.5f}, {5.9f, 7.0f, 6.9f, 10.5f}}},
    {15, 1, 4, 4, 2, {{2.9f, 3.0f, 3.4f, 3.6f}, {3.5f, 3.8f, 4.15f, 4.45f}}},
    {14, 1, 4, 2, 4, {{4.7f, 5.2f, 5.4f, 5.4f}, {5.8f, 6.6f, 5.6f, 6.5f}}},
};

static int fmt_slot(int fmt) { return fmt == Q4_0 ? 0 : fmt == Q4_K ? 1 : fmt == Q8_0 ? 2 : 3; }

// The best shape for a product and its estimated time (us). Shape 11's workgroups run
// two to a CU, where a round of them takes 0.82 of two. RQMV_TILE names a shape instead.
static const TileShape& tile_plan(int fmt, bool f32, int64_t M, int64_t rows, int64_t cols, int cus, float* us) {
    const char* env = getenv("RQMV_TILE");
    const int want = env && *env ? atoi(env) : 0;
    const TileShape* best = nullptr;
    for (const TileShape& s : kTileShapes) {
        const int64_t bn = 16 * s.rt * s.wn, bm = 16 * (f32 ? s.mt / 2 : s.mt);
        const int64_t wgs = (rows + bn - 1) / bn * ((M + bm - 1) / bm);
        const int64_t steps = ((cols + 255) / 256 + s.wk - 1) / s.wk, rounds = (wgs + cus - 1) / cus;
        const float share = s.id == 11 && rounds > 1 ? 0.82f : 1.f;
        const float t = 4.f + s.step[f32][fmt_slot(fmt)] * (float)steps * (float)rounds * share;
        if (s.id == want || (!best || (t < *us && best->id != want))) {
            best = &s;
            *us = t;
        }
    }
    return *best;
}

template <int FMT, bool XF32>
static hipError_t launch_tile_fmt(int shape, const MvParams& p, int M, uint32_t x_bytes, hipStream_t stream,
                                  hipEvent_t ev0, hipEvent_t ev1) {
    constexpr int L = XF32 ? 4 : 8, S = XF32 ? 2 : 4;  // activation tiles of the shapes' mt 8 and 4
#define RQ_SHAPE(RT, MT, WN, WK) launch_tile_one<FMT, RT, MT, WN, WK, XF32>(p, M, x_bytes, stream, ev0, ev1)
    switch (shape) {
        case 11: return RQ_SHAPE(1, S, 8, 1);
        case 12: return RQ_SHAPE(1, L, 8, 1);
        case 22: return RQ_SHAPE(2, L, 8, 1);
        case 15: return RQ_SHAPE(1, S, 4, 2);
        default: return RQ_SHAPE(1, S, 2, 4);
    }
#undef RQ_SHAPE
}

// Against the other forms, by the same measure. The streaming form (fp16 x) takes 32
// rows a launch and per launch 3 us and the larger of 0.65 us (Q8_0 0.9) a step of 256
// values and 1.6 ns a step and row tile (Q4_K 4096->14336 25 us, Q8_0 5120x5120 21,
// Q6_K 5120->25600 55); up to 32 rows it is always ahead (Q4_K 4096x4096 at 20 rows 13.9
// against 19.2). The direct form (fp32 x) is ahead up to 16 rows; above, it takes the
// larger of 0.9 us a step and 3.6 ns a step and row tile (2.5 with two row tiles per
// wave) for one or two activation tiles per wave, and where the rows fall into groups
// of three tiles 3.5 ns a group (Q6_K 14336->4096 at 77 rows 106 against 120); otherwise
// it is behind. RQMV_TILE=0 keeps every product off the tiled form.
bool tile_takes(int fmt, int xtype, int M, int64_t rows, int64_t cols, int cus) {
    const char* env = getenv("RQMV_TILE");
    if (env && *env) return *env != '0';
    float us = 0.f;
    const bool f32 = xtype == X_F32;
    if (M <= 16 || (!f32 && M <= 32)) return false;
    tile_plan(fmt, f32, M, rows, cols, cus, &us);
    const float steps = (float)((cols + 255) / 256), units = steps * (float)((rows + 15) / 16);
    if (f32) {
        const int tiles = (M + 15) / 16, groups = (tiles + 3) / 4;
        if (M > 32 && (groups == 1 || (tiles + groups - 1) / groups != 3)) return true;
        const float b = (M > 32 ? 3.5e-3f * (float)groups : (rows + 15) / 16 > cus ? 2.5e-3f : 3.6e-3f) * units;
        return us < 4.f + (0.9f * steps > b ? 0.9f * steps : b);
    }
    const float a = (fmt == Q8_0 ? 0.9f : 0.65f) * steps, b = 1.6e-3f * units;
    return us < (float)((M + 31) / 32) * (3.f + (a > b ? a : b));
}

hipError_t launch_matvec_tile(int fmt, int xtype, int M, const MvParams& p, int cus, hipStream_t stream, hipEvent_t ev0,
                              hipEvent_t ev1) {
    const bool f32 = xtype == X_F32;
    const int64_t x_bytes = ((int64_t)(M - 1) * p.ldx + p.K) * (f32 ? 4 : 2);
    if (M < 1 || x_bytes >= (int64_t)kOobOffset) return hipErrorInvalidValue;
    float us = 0.f;
    const int shape = tile_plan(fmt, f32, M, p.rows, p.K, cus, &us).id;
#define RQ_TILE(FMT)                                                                              \
    return f32 ? launch_tile_fmt<FMT, true>(shape, p, M, (uint32_t)x_bytes, stream, ev0, ev1)     \
               : launch_tile_fmt<FMT, false>(shape, p, M, (uint32_t)x_bytes, stream, ev0, ev1)
    switch (fmt) {
        case Q4_0: RQ_TILE(Q4_0);
        case Q4_K: RQ_TILE(Q4_K);
        case Q8_0: RQ_TILE(Q8_0);
        case Q6_K: RQ_TILE(Q6_K);
        default: return hipErrorInvalidValue;
    }
#undef RQ_TILE
}

}  // namespace rq
