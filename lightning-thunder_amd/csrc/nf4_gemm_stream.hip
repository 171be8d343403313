// Which tile the kernel of nf4_gemm_stream.h uses for a call, and its launch.
#include "nf4_gemv.h"

namespace nf4 {
namespace stream {
hipError_t launch_bf16(const MatmulArgs& a, const StreamPlan& p, hipStream_t stream);
hipError_t launch_bf16_dq(const MatmulArgs& a, const StreamPlan& p, hipStream_t stream);
hipError_t launch_f16(const MatmulArgs& a, const StreamPlan& p, hipStream_t stream);
hipError_t launch_f16_dq(const MatmulArgs& a, const StreamPlan& p, hipStream_t stream);
}  // namespace stream
namespace {

// The rule is a model of the kernel's time in us: rounds of 256 workgroups (one per CU), each the 64-k steps of its
// longest k group at 0.45..1 us (by the rows of x per tile; up to 30 % less on a sparsely filled chip); partial tiles that meet
// in the workspace cost by their size and number.  Over M = 1..128 at fifteen shapes from [600, 1088] to [128256, 4096] its
// choice takes 0.6 % longer than the best of all choices on average, 9 % at most.  (M <= 16 is judged as 32 rows: the two
// differ by 0.02 us per step, and a call's sums are then added in one order whether its rows come alone or with others.)
float step_us(int bm) { return bm <= 32 ? 0.47f : bm == 64 ? 0.67f : 1.0f; }
float model_us(int64_t wgs, int64_t steps, int bm, int rows, int splits) {
    const int64_t rounds = (wgs + 255) / 256;
    const float fill = (float)wgs / (float)(rounds * 256);
    const float merge = splits == 1 ? 0.0f : 1.0f + (float)(rows * bm) / 32768.0f * (float)(5 + splits);
    return (float)rounds * ((float)steps * step_us(bm) * (0.7f + 0.3f * fill) + 1.0f) + merge;
}

size_t plan_bytes(const StreamPlan& p) {
    if (p.splits == 1) return 0;
    return GEMV_COUNTER_REGION_BYTES + (size_t)p.m_tiles * p.n_tiles * p.splits * p.wn * 32 * (p.bm < 32 ? 32 : p.bm) * sizeof(float);
}

}  // namespace

bool stream_possible(int64_t M, int64_t N, int64_t K) {
    // 32-bit offsets: of x, of a tile's codes, of a weight's blocks
    return M >= 1 && M < (1 << 20) && N >= 1 && K >= 64 && K % 64 == 0 && K < (1 << 24) && N <= INT32_MAX &&
           N * (K / 64) < ((int64_t)1 << 31) && M * K * 2 < ((int64_t)1 << 32);
}

// More than 128 rows of x: while tiles of 128 x 256 fill the chip once at most.  Measured against the kernel of
// nf4_gemm_wide.hip (its own tiles and pieces; graph replay, cold weights, us, wide / here), M = 130, 512, 2048: [1024, 4096] 25.4 / 10.6,
// 26.1 / 13.6, 34.6 / 28.9; [4096, 4096] 28.7 / 18.6, 35.6 / 27.7, 76.8 / 74.1 (256 tiles); [4096, 14336] 52.5 / 41.4, 80.4 / 72.9, 224.5 /
// 218.3; [14336, 4096] 50.0 / 40.9, 73.4 / 65.8 (224 tiles), 216.6 / 253.6.  Beyond one round that kernel's 256-row tiles expand every
// weight half as often: [28672, 4096] M = 256 75.1 / 65.3 (224 tiles), M = 384 112.5 / 118.1 (336).  With few k steps and a nearly
// full chip the two are level ([32000, 1024] M = 130..256, 250 tiles: 25.8, 25.5, 26.7 / 25.8, 26.0, 27.4).
bool stream_served(int64_t M, int64_t N, int64_t K) {
    if (!stream_possible(M, N, K)) return false;
    const int64_t tiles = ((M + 127) / 128) * ((N + 255) / 256);
    return M <= 128 || tiles <= (K >= 2048 ? 256 : 128);
}

// Of these, nf4hip_gemm leaves to that kernel what it takes in 256-row tiles cut along K (at most 128 of them, K >= 14336) when its
// model is ahead: the 128-row tiles here expand every weight twice as often and often have no split left to fill the chip with.
// Over 80 such shapes the choice takes 0.2 % longer than the better of the two on average, 6 % at most (always here: 7 %, 36 %); wide /
// here: M = 986 [4384, 27520] 243 / 330, M = 1343 [4864, 26560] 358 / 413, M = 2005 [3236, 20224] 271 / 295, M = 315 [8768, 27648] 250 / 206.
bool stream_serves_gemm(int64_t M, int64_t N, int64_t K) {
    if (!stream_served(M, N, K)) return false;
    return M <= 128 || !gemm_wide_cuts_long_tiles(M, N, K) || stream_us(M, N, K) <= gemm_wide_us(M, N, K);
}

namespace {

StreamPlan plan_and_time(int64_t M, int64_t N, int64_t K, int max_splits, float& best_us) {
    StreamPlan best{};
    best_us = 0.0f;
    const int64_t ksteps = K / 64, units = (ksteps + 3) / 4;
    for (int bm = 32; bm <= 128; bm *= 2) {
        const int64_t m_tiles = (M + bm - 1) / bm;
        for (int wn = bm == 128 ? 8 : bm == 64 ? 4 : 2; wn <= 8; wn *= 2) {
            const int64_t n_tiles = (N + 32 * wn - 1) / (32 * wn);
            const int wk = 8 / wn;
            for (int s = 1; s <= max_splits; ++s) {
                if (s > 1 && (m_tiles * n_tiles * s > 256 || units < s * wk)) break;  // one round, nobody idle
                const int64_t steps = 4 * ((units + wk * s - 1) / (wk * s));
                const float us = model_us(m_tiles * n_tiles * s, steps < ksteps ? steps : ksteps, bm, 32 * wn, s);
                if (!best.bm || us < best_us) {
                    best = StreamPlan{bm, wn, s, (int)m_tiles, (int)n_tiles};
                    best_us = us;
                }
            }
        }
        if (bm >= M) break;
    }
    if (M <= 16 && best.bm == 32) best.bm = 16;
    return best;
}

}  // namespace

StreamPlan stream_plan(int64_t M, int64_t N, int64_t K, int max_splits) {
    float us;
    return plan_and_time(M, N, K, max_splits, us);
}

// (5 us: what the model leaves out because every choice has it, the start of a launch and its last stores.  Measured / modelled
// at M = 130, 512, 2048: [1024, 4096] 10.6, 13.6, 28.9 / 10.8, 13.5, 27.4; [4096, 4096] 18.6, 27.7, 74.1 / 18.7, 27.4, 70.0; [4096, 14336]
// 41.4, 72.9, 218.3 / 43.5, 72.0, 230.0; [14336, 4096] at 130 and 512 40.9, 65.8 / 44.5, 67.6.)
float stream_us(int64_t M, int64_t N, int64_t K) {
    float us;
    plan_and_time(M, N, K, STREAM_MAX_SPLITS, us);
    return us + 5.0f;
}

size_t stream_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    return stream_possible(M, N, K) ? plan_bytes(stream_plan(M, N, K, STREAM_MAX_SPLITS)) : 0;
}

hipError_t launch_stream(const MatmulArgs& a, bool f16, hipStream_t stream) {
    StreamPlan p = stream_plan(a.M, a.N, a.K, STREAM_MAX_SPLITS);
    if (plan_bytes(p) > a.workspace_bytes) p = stream_plan(a.M, a.N, a.K, 1);
    if (f16) return a.nested.q ? stream::launch_f16_dq(a, p, stream) : stream::launch_f16(a, p, stream);
    return a.nested.q ? stream::launch_bf16_dq(a, p, stream) : stream::launch_bf16(a, p, stream);
}

}  // namespace nf4
