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

// The shapes, and what a step of 256 values of K and a round of workgroups over the
// chip take in each (us; 0: not built, since its registers spill and no product was
// fastest in it). Fitted to 3,847 products of 256 to 25,600 rows, 1,024 to 14,336
// columns and 17 to 512 activation rows, each timed in every shape (within 5 to 9 % of
// the estimates, root mean square). The plan takes the shape whose rounds cost the
// fewest; over the same products its choice, this form or the other, takes 0.4 % more
// than the best of all on average, 20 % at most.
// us a product at the shape the plan takes, against the streaming form in launches of
// 32 rows (fp16 x) or the direct form (fp32 x):
//   fp16 x  Q4_K 4096->14336 at 64 / 512 rows 48.5 / 381 -> 28.5 / 108 (557 TFLOP/s)
//           Q4_0 4096->14336 at 512 rows 332 -> 96.3 (624 TFLOP/s)
//           Q6_K 14336->4096 at 128 / 512 rows 157 / 608 -> 82 / 161
//           Q8_0 5120x5120 at 64 / 512 rows 41.5 / 341 -> 30.3 / 82.1
//   fp32 x  Q4_K 4096->14336 at 64 / 512 rows 79 / 498 -> 48 / 242
//           Q6_K 14336->4096 at 512 rows 589 -> 323
// With few workgroups, several ranges of K per workgroup (x2, x4) make up for the
// rows they take from it: Q6_K 14336->4096 at 64 rows 159 -> 79 (fp16 x).
struct TileShape {
    int id, rt, mt, wn, wk;  // mt for fp16 x, half of it for fp32 x
    float step[2][4];        // us per step: [fp32 x][Q4_0, Q4_K, Q8_0, Q6_K]
    float round;             // us per round
};
constexpr TileShape kTileShapes[] = {
    {11, 1, 4, 8, 1, {{2.02f, 2.06f, 2.51f, 2.70f}, {2.38f, 2.72f, 2.89f, 3.60f}}, 0.6f},
    {12, 1, 8, 8, 1, {{3.06f, 3.08f, 3.44f, 3.82f}, {3.62f, 4.41f, 4.09f, 5.36f}}, 2.8f},
    {22, 2, 8, 8, 1, {{5.26f, 5.81f, 6.02f, 0.00f}, {5.60f, 6.93f, 6.45f, 10.87f}}, 2.6f},
    {15, 1, 4, 4, 2, {{2.49f, 2.78f, 2.98f, 3.28f}, {3.07f, 3.52f, 3.52f, 4.17f}}, 2.5f},
    {14, 1, 4, 2, 4, {{3.73f, 4.33f, 4.21f, 4.60f}, {4.70f, 5.34f, 5.18f, 5.74f}}, 3.1f},
};

static int fmt_slot(int fmt) { return fmt == Q4_0 ? 0 : fmt == Q4_K ? 1 : fmt == Q8_0 ? 2 : 3; }

// The best shape for a product and its estimated time (us). Rounds are those of the XCD
// with the most workgroups (an XCD takes every eighth tile of rows). Of several, each
// takes 1.04 of one alone, in shape 11, whose workgroups run two to a CU, 0.87 (fp16 x) or
// 0.79. RQMV_TILE names a shape instead.
static const TileShape& tile_plan(int fmt, bool f32, int64_t M, int64_t rows, int64_t cols, int cus, float* us) {
    const char* env = getenv("RQMV_TILE");
    const int want = env && *env ? atoi(env) : 0;
    const TileShape* best = nullptr;
    for (const TileShape& s : kTileShapes) {
        const float step = s.step[f32][fmt_slot(fmt)];
        if (step == 0.f || (!f32 && fmt == Q4_K && s.rt == 2 && cols < kFoldWhole)) continue;  // (that shape folds whole blocks)
        const int64_t bn = 16 * s.rt * s.wn, bm = 16 * (f32 ? s.mt / 2 : s.mt);
        const int64_t wgs = ((rows + bn - 1) / bn + 7) / 8 * 8 * ((M + bm - 1) / bm);
        const int64_t steps = ((cols + 255) / 256 + s.wk - 1) / s.wk, rounds = (wgs + cus - 1) / cus;
        const float each = rounds == 1 ? 1.f : s.id != 11 ? 1.04f : f32 ? 0.79f : 0.87f;
        const float t = 1.5f + (float)rounds * each * (step * (float)steps + s.round);
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
        case 22:
            if constexpr (FMT == Q6_K && !XF32) return hipErrorInvalidValue;  // (not built: the plan never names it)
            else return RQ_SHAPE(2, L, 8, 1);
        case 15: return RQ_SHAPE(1, S, 4, 2);
        default: return RQ_SHAPE(1, S, 2, 4);
    }
#undef RQ_SHAPE
}

// Against the other form, by the same measure (stream_us, direct_us). The streaming
// form (fp16 x) is always ahead up to 32 rows (Q4_K 4096x4096 at 20 rows 13.9 against
// 19.2), the direct form (fp32 x) up to 16. RQMV_TILE=0 keeps every product off the
// tiled form.
bool tile_takes(int fmt, int xtype, int M, int64_t rows, int64_t cols, int cus) {
    const char* env = getenv("RQMV_TILE");
    if (env && *env) return *env != '0';
    const bool f32 = xtype == X_F32;
    if (M <= 16 || (!f32 && M <= 32)) return false;
    float us = 0.f;
    tile_plan(fmt, f32, M, rows, cols, cus, &us);
    return us < (f32 ? direct_us(fmt, M, rows, cols, cus) : stream_us(fmt, M, rows, cols, cus));
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
