// The rule that picks the kernel of an M > 16 projection no measured ladder names: tw4_gemm_plan. Every candidate's time is
// predicted from the sizes alone and the fastest is taken. Host code: a call plans its kernel at the first use of its (M, N, K), and
// prompt lengths are mostly new, so a plan has to cost less than a launch (2-5 us; the same search in Python took 80-340).
//
// The terms follow the kernels' structure, so one row of coefficients per configuration covers every shape:
//   units U = (output tiles x K splits) dealt to the CUs: the busiest runs ceil(U / CUs) of them, `occ` at a time;
//   a unit costs (its steps along K) x (time of a step on a full CU, or alone; in between in a straight line);
//   a K split adds the wait for the last arriver, its fp32 partial tile and the traffic of all of them;
//   every launch has a fixed cost, every further unit of a CU a prologue and an epilogue;
//   the bytes all units move together: weights from memory, x and weights of every tile through L2, SwiGLU's results.
// The coefficients are microseconds on MI355X (256 CUs), fitted with `python bench.py fit` (non-negative least squares on relative
// errors) to 34,000 timed calls, weights streamed from HBM: 28 (K, N) from 1024 x 4096 to 5120 x 34816, N = 1032 and 7288
// among them, x 35 M from 17 to 4096 (profiles/gemm_rule_sweep.jsonl). The choice is 1.2 % slower than the fastest timed
// candidate on average, within 6 % at 95 of 100 sizes, 16 % at worst; 1.5, 8 and 26 % (a library product at M = 3500) over seven shapes
// left out of the fit. Against the fixed ladder these sizes had before any rule (8 wavefronts of the decode kernel up to M = 64, the
// x-ring GEMM to 1024, dequantize + hipBLASLt above) it takes 0.72 of the time on average: Qwen3-14B gate_up at M = 40 132 us
// against 40, Qwen3-8B-sized qkv (K 4096, N 6144) at M = 512 43 against 32.
#include <algorithm>
#include <initializer_list>

#include "tw4_common.h"

namespace tw4 {

struct PlanCost {
    double launch;        // per call
    double full, alone;   // a step of a unit on a CU with `occ` units, with one
    double unit;          // a further unit of the busiest CU
    double split, part;   // a K split: the wait, per 10^4 partial sums of a tile's splits
    double weights;       // per MB of packed weights
    double partials;      // per MB of partial sums of the whole call
    double x, tiles;      // per MB of x and of weights that all tiles read
    double act;           // SwiGLU: per MB of gate and up
};
// tw4_gemm_tiled (mt, nt, warps_n, warps_m, warps_k, ring), occ workgroups per CU; a step is 64 k
struct PlanTiled {
    int mt, nt, wn, wm, wk, ring, occ;
    PlanCost c;
};
// tw4_gemm's x ring (mt, nt, warps_n, warps_k, stages); a step is warps_k groups. Its weights skip LDS, so it starts sooner: short
// K ranges and small N.
struct PlanRing {
    int mt, nt, wn, wk, stages, occ;
    PlanCost c;
};
// the matrix-core decode kernel (warps_k, unroll, ntile), M <= 64; a step is a group of one of its warps_k wavefronts, and costs
// (full | alone) + (full | alone)_tile per batch tile of 16 tokens (2 or 4 of them)
struct PlanMma {
    int wk, unroll, ntile, max_m;
    double launch, full, alone, full_tile, alone_tile, unit, tile, weights, x, act;
};

constexpr double kPlanTiledPflops = 1.24;  // long calls run at the clock the card's power allows
constexpr PlanTiled kPlanTiled[] = {
    {2, 2, 2, 1, 2, 4, 4, {4.263, 0.2843, 0.157, 0.1535, 0.2202, 1.43, 0.07071, 0.1459, 0, 0.06634, 0.5368}},  // 32 x 64
    {2, 3, 2, 1, 2, 4, 4, {4.099, 0.3899, 0.186, 0.2415, 0.4852, 1.223, 0.06283, 0.1606, 0, 0.06364, 0.529}},  // 32 x 96
    {3, 2, 2, 1, 2, 4, 4, {4.001, 0.3749, 0.1726, 0.5309, 0.4221, 1.31, 0.0922, 0.1369, 0.02105, 0, 0.4379}},  // 48 x 64
    {3, 3, 2, 1, 2, 4, 3, {4.36, 0.3825, 0.2071, 0.6481, 0.4521, 0.8755, 0.06646, 0.1665, 0.01771, 0.02311, 0.5183}},  // 48 x 96
    {4, 2, 2, 1, 2, 4, 3, {4.066, 0.3364, 0.1825, 0.5995, 0.4119, 1.053, 0.07531, 0.1742, 0.01586, 0.01754, 0.4282}},  // 64 x 64
    {4, 3, 2, 1, 2, 4, 3, {4.858, 0.429, 0.215, 0.7439, 0.1847, 0.727, 0.06086, 0.1735, 0.01349, 0.04131, 0.4575}},  // 64 x 96
    {5, 2, 2, 1, 2, 4, 2, {4.363, 0.2999, 0.2058, 0.7892, 0.2221, 0.9259, 0.08093, 0.1876, 0.01165, 0, 0.4016}},  // 80 x 64
    {5, 3, 2, 1, 2, 4, 2, {4.825, 0.3388, 0.245, 1.443, 0.3586, 0.8735, 0.04941, 0.1701, 0.01239, 0.05689, 0.4433}},  // 80 x 96
    {5, 4, 2, 1, 2, 4, 2, {5.418, 0.4351, 0.2935, 1.75, 0.2735, 0.9584, 0.04272, 0.1683, 0.01934, 0.03908, 0.4106}},  // 80 x 128
    {8, 2, 2, 1, 2, 4, 2, {5.049, 0.4184, 0.2512, 1.612, 0, 0.8086, 0.0276, 0.2331, 0.008498, 0.03748, 0.4059}},  // 128 x 64
    {8, 3, 2, 1, 2, 4, 1, {6.235, 0.3184, 0, 5.066, 0, 0.3184, 0.04632, 0.256, 0.01242, 0.007974, 0.5946}},  // 128 x 96
    {8, 4, 2, 1, 2, 4, 1, {6.997, 0.3431, 0, 5.842, 0, 0.3484, 0.01823, 0.2542, 0.006154, 0.1048, 0.5239}},  // 128 x 128
    {8, 4, 4, 1, 1, 3, 2, {7.718, 0.8805, 0.4976, 3.692, 0, 0.4335, 0.04006, 0.2131, 0, 0.1692, 0.1435}},  // 128 x 256
    {8, 6, 2, 1, 2, 4, 1, {8.902, 0.4914, 0, 7.638, 0, 1.137, 0.05522, 0.2284, 0.0397, 0.006301, 0.5254}},  // 128 x 192
    {8, 6, 2, 2, 1, 3, 1, {9.728, 0.7085, 0, 10.48, 0, 0, 0.04363, 0.5105, 0.02484, 0.2178, 0.09126}},  // 256 x 192
};
constexpr PlanRing kPlanRing[] = {
    {2, 1, 4, 2, 2, 4, {3.225, 1.33, 0.5999, 0.3716, 0.6888, 1.331, 0.03114, 0.2026, 0, 0.0334, 0.2522}},  // 32 x 64
    {2, 2, 4, 2, 2, 2, {3.644, 1.302, 0.8649, 0.8988, 0.5723, 0.9686, 0.02168, 0.2249, 0, 0.0143, 0.183}},  // 32 x 128
    {4, 2, 4, 2, 2, 2, {4.176, 2.372, 1.196, 2.578, 0.6866, 0.4721, 0.01123, 0.2186, 0.01059, 0, 0.06145}},  // 64 x 128
};
constexpr PlanMma kPlanMma[] = {
    {4, 1, 1, 48, 2.25, 0, 0, 0.4057, 0.19, 0, 0.1539, 0, 0.06696, 0},
    {4, 1, 2, 48, 2.47, 0, 0.1014, 0.4363, 0.2535, 0.5073, 0.1103, 0, 0.06571, 0.453},
    {4, 1, 3, 64, 2.59, 0.3685, 0.1419, 0.4001, 0.3175, 0.5103, 0.1105, 0, 0.06497, 0.6496},
    {4, 1, 6, 64, 3.442, 0.7838, 0.3092, 0.7079, 0.3663, 0, 0.579, 0, 0.06583, 1.868},
};
// dequantize + hipBLASLt, from M = 1536 on (below, a fused kernel was the fastest at all but one of the timed sizes): launches, per 10^6
// weights (the dequantized matrix out and in), per 10^9 products, per round of 256 x 256 tiles and 10^3 k (its last round nearly
// empty costs a whole one), per 10^6 results, and those of the separate SwiGLU. At ragged M the library's time varies most (24576 x
// 4096 at M = 3000 618 us, as at 4096, against 509 fused): there it has to be that much faster.
constexpr double kPlanRagged = 1.03;
constexpr double kPlanDense[6] = {10.4, 0.6708, 1.142, 2.327, 0.2666, 1.306};
constexpr int kPlanDenseRows = 1536;
constexpr int kPlanRingRows = 256;
constexpr int kPlanSplits[] = {1, 2, 3, 4, 6, 8, 12, 16};

static int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The busiest CU's steps at the full rate and at the lone one, for n units at most `occ` at a time.
struct PlanLoad {
    double full, alone;
    int64_t more;
};
static PlanLoad plan_load(int64_t units, int cus, int occ, double steps) {
    const int64_t n = cdiv(units, cus), rounds = n / occ, left = n % occ;
    const double share = left && occ > 1 ? static_cast<double>(left - 1) / (occ - 1) : 0.0;
    return {(rounds + share) * steps, left ? (1.0 - share) * steps : 0.0, n - 1};
}

}  // namespace tw4

using namespace tw4;

extern "C" int tw4_gemm_plan(int M, int N, int K, int act, int cus, int* out) {
    TW4_REQUIRE(out, -TW4_EINVAL, "gemm_plan: null pointer");
    TW4_REQUIRE(M >= 1 && N >= 8 && N % 8 == 0 && K >= 128 && K % 128 == 0 && cus >= 1, -TW4_EINVAL,
                "gemm_plan: M >= 1, N %% 8 == 0, K %% 128 == 0 (M %d, N %d, K %d, %d CUs)", M, N, K, cus);
    const int64_t groups = K / 128;
    const double m = M, n = N, k = K, chip = 256.0 / cus;  // the call's share of the coefficients' memory rates
    const double weights_mb = n * k / 2e6 * chip, act_mb = act ? m * n * 2 / 1e6 * chip : 0.0;
    const double floor = 2.0 * m * n * k / (kPlanTiledPflops * 1e9) * chip;
    int ints = 0;
    double best = 1e300;
    auto offer = [&](double t, std::initializer_list<int> entry) {
        if (!(t < best)) return;
        best = t;
        ints = 0;
        for (const int v : entry) out[ints++] = v;
    };
    auto tile_cost = [&](const PlanCost& c, int occ, int bm, int bn, int64_t tiles, int64_t steps, int splits) {
        const PlanLoad l = plan_load(tiles * splits, cus, occ, static_cast<double>(steps));
        const double mb = static_cast<double>(cdiv(M, bm)), partial = static_cast<double>(splits) * bm * bn;
        double t = c.launch + c.full * l.full + c.alone * l.alone + c.unit * l.more + c.weights * weights_mb + c.act * act_mb +
                   (c.x * static_cast<double>(tiles) * (M < bm ? M : bm) * k * 2 / 1e6 + c.tiles * mb * n * k / 2e6) * chip;
        if (splits > 1) t += c.split + c.part * partial / 1e4 + c.partials * static_cast<double>(tiles) * partial * 4 / 1e6 * chip;
        return t;
    };
    // K splits within the default workspace, and only where the tiles alone do not fill the GPU twice
    auto split_ok = [&](int64_t tiles, int splits, int bm, int bn) {
        return splits == 1 || (splits <= groups && tiles < 2 * cus && tiles <= TW4_AUTO_SPLIT_COUNTERS &&
                               tiles * splits * bm * bn <= TW4_AUTO_SPLIT_FLOATS);
    };
    if (M >= kPlanDenseRows) {
        const double* d = kPlanDense;
        const double rounds = static_cast<double>(cdiv(cdiv(M, 256) * cdiv(N, 256), cus));
        const double t = d[0] + d[3] * rounds * k / 1e3 +
                         (d[1] * n * k / 1e6 + d[2] * m * n * k / 1e9 + d[4] * m * n / 1e6 + (act ? d[5] * m * n / 1e6 : 0.0)) * chip;
        offer(M % 256 ? kPlanRagged * t : t, {0});
    }
    if (static_cast<int64_t>(M) * K < (1LL << 31) && ((N + 15LL) & ~15LL) * K < (1LL << 33))  // tw4_gemm_tiled's limits
        for (const PlanTiled& p : kPlanTiled) {
            const int bm = 16 * p.mt * p.wm, bn = 16 * p.nt * p.wn;
            const int64_t tiles = cdiv(M, bm) * cdiv(N, bn);
            for (const int s : kPlanSplits)
                if (split_ok(tiles, s, bm, bn)) {
                    const double t = tile_cost(p.c, p.occ, bm, bn, tiles, 2 * cdiv(groups, s), s);
                    offer(std::max(floor, t) + 1e-3 * t, {3, p.mt, p.nt, p.wn, p.wm, p.wk, p.ring, s});  // at the floor: the least
                }
        }
    if (M <= kPlanRingRows || !ints)  // past it only where nothing else takes the sizes
        for (const PlanRing& p : kPlanRing) {
            const int bm = 16 * p.mt, bn = 16 * p.nt * p.wn;
            const int64_t tiles = cdiv(M, bm) * cdiv(N, bn), steps = cdiv(groups, p.wk);
            for (const int s : kPlanSplits)
                if (s <= steps && split_ok(tiles, s, bm, bn))
                    offer(tile_cost(p.c, p.occ, bm, bn, tiles, cdiv(steps, s), s), {2, p.mt, p.nt, p.wn, p.wk, p.stages, s});
        }
    for (const PlanMma& p : kPlanMma) {
        if (M > p.max_m) continue;
        const int64_t units = cdiv(cdiv(N, 16), p.ntile);
        const PlanLoad l = plan_load(units, cus, 2, static_cast<double>(cdiv(groups, p.wk)));
        const double mt = M <= 32 ? 2 : 4;
        offer(p.launch + (p.full + p.full_tile * mt) * l.full + (p.alone + p.alone_tile * mt) * l.alone + p.unit * l.more +
                  p.tile * mt + p.weights * weights_mb + p.x * static_cast<double>(units) * m * k * 2 / 1e6 * chip + p.act * act_mb,
              {1, p.wk, p.unroll, p.ntile});
    }
    return ints;
}
