// RMSNorm and residual-add + RMSNorm of the decoder layer around the W4A16 projections, fp16 rows
// of K values (K % 512 == 0, K <= 8192), fp32 math:
//
//   tw4_rms_norm:      y = fp16(x rstd w),                  rstd = rsqrt(mean(x^2) + eps)
//   tw4_add_rms_norm:  s = x + r (fp32); r <- fp16(s); x <- fp16(s rstd w),  rstd from s (in place)
//
// A workgroup per row (four for the shortest), W wavefronts of J chunks per lane (8 halves, 16 bytes: chunks W 64 j + 64 wave + lane of the row),
// all loaded before any math and kept in registers for the second pass. The sum of squares follows the fixed order of
// norm_rstd (per chunk, per quant group of 16 chunks, then over the groups), the same order as the decode kernels' fused
// norm prologue, so a fused projection sees the very bits this kernel writes.
// A decode batch is a few rows and latency-bound: one chunk per lane (two from K = 5120) leaves two dependent round trips to
// memory and one chunk's arithmetic, where a wavefront per row ran all K / 512 chunks' one after another. us before ->
// after, add + norm (norm alone): K 4096 M = 1 2.7 -> 1.9 (2.5 -> 1.8), M = 8 3.4 -> 2.1 (3.0 -> 2.0), M = 512 4.4 -> 3.5;
// K 2048 M = 5 2.3 -> 1.9; K 5120 M = 40 3.9 -> 2.3; K 8192 M = 8 5.3 -> 2.4. The launch itself takes 1.8.
// From kTallRows rows on the rows alone fill the GPU and the kernel is bound by memory: fewer wavefronts per row with more
// loads in flight each. add + norm at M = 2048, that form / the short one / a wavefront per row: K 2560 5.5 / 5.7 / 5.6,
// K 4096 7.5 / 7.6 / 8.1, K 5120 10.9 / 11.6 / 10.8; over M = 1024 .. 8192 that form takes 0.75-1.0 of a wavefront per row's time
// from K = 1536 on (two odd ones: norm alone at K 5120, M = 2048 1.07, K 3072, M = 3000 1.06), and the short form is level
// with it at M = 1023. Rows of K <= 1024 are one or two chunks per lane: from kManyRows rows on a workgroup per row is bound by
// dispatching them, and four rows share one, a wavefront each (add + norm at K 1024, M = 1024: 3.7 -> 3.5).
#include "tw4_common.h"

namespace tw4 {

constexpr int kNormMaxGroups = 64;  // K <= 8192
constexpr int kTallRows = 1024, kManyRows = 640;

// ROWS > 1: that many rows per workgroup, a wavefront each (W = 1).
template <bool ADD, int W, int J, int ROWS>
__global__ void __launch_bounds__(64 * W * ROWS) rms_norm_kernel(h1* x, h1* r, const h1* __restrict__ w, h1* y, int M, int K,
                                                                 float eps) {  // y may be x: every store follows every load
    static_assert(W == 1 || ROWS == 1, "a row is one workgroup's or one wavefront's");
    __shared__ float sums[ROWS][ROWS == 1 ? kNormMaxGroups : 4 * J];
    const int lane = threadIdx.x & 63, wave = ROWS == 1 ? threadIdx.x >> 6 : 0;
    const int sub = ROWS == 1 ? 0 : threadIdx.x >> 6, row = blockIdx.x * ROWS + sub;
    if (ROWS > 1 && row >= M) return;  // whole wavefronts; no workgroup barrier below for them
    float* gsum = sums[sub];
    const int64_t base = static_cast<int64_t>(row) * (K >> 3);
    u4* xr = reinterpret_cast<u4*>(x) + base;
    u4* rr = reinterpret_cast<u4*>(r) + base;
    const u4* wr = reinterpret_cast<const u4*>(w);
    u4 xv[J], rv[J], wv[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int c = 64 * (W * j + wave) + lane;
        xv[j] = xr[c];
        if constexpr (ADD) rv[j] = rr[c];
        wv[j] = wr[c];
    }
    float s[J][8];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        chunk_to_f32(xv[j], s[j]);
        if constexpr (ADD) {
            float b[8];
            chunk_to_f32(rv[j], b);
#pragma unroll
            for (int i = 0; i < 8; ++i) s[j][i] += b[i];
        }
        const float q = row16_sum(sumsq8(s[j]));  // quant group 4 (W j + wave) + lane / 16
        if ((lane & 15) == 0) gsum[4 * (W * j + wave) + (lane >> 4)] = q;
    }
    if constexpr (ROWS == 1) {
        __syncthreads();
    } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    const float rstd = norm_rstd(gsum, K >> 7, K, eps, lane);
    u4* yr = reinterpret_cast<u4*>(y) + base;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int c = 64 * (W * j + wave) + lane;
        float g[8];
        if constexpr (ADD) rr[c] = f32_to_chunk(s[j]);
        chunk_to_f32(wv[j], g);
#pragma unroll
        for (int i = 0; i < 8; ++i) s[j][i] = s[j][i] * rstd * g[i];
        yr[c] = f32_to_chunk(s[j]);
    }
}

template <bool ADD>
int norm_launch(h1* x, h1* r, const h1* w, h1* y, int M, int K, float eps, hipStream_t st) {
    const int tall = M >= (K <= 1024 ? kManyRows : kTallRows) ? 100 : 0;
    switch (tall + (K >> 9)) {
#define TW4_NORM_ROWS(TALL, W, J, ROWS)                                                                                   \
    case TALL + W * J:                                                                                                    \
        rms_norm_kernel<ADD, W, J, ROWS><<<static_cast<unsigned>((M + ROWS - 1) / ROWS), 64 * W * ROWS, 0, st>>>(x, r, w, \
            y, M, K, eps);                                                                                                \
        break;
#define TW4_NORM_CASE(TALL, W, J) TW4_NORM_ROWS(TALL, W, J, 1)
        TW4_NORM_CASE(0, 1, 1) TW4_NORM_CASE(0, 2, 1) TW4_NORM_CASE(0, 3, 1) TW4_NORM_CASE(0, 4, 1)
        TW4_NORM_CASE(0, 5, 1) TW4_NORM_CASE(0, 6, 1) TW4_NORM_CASE(0, 7, 1) TW4_NORM_CASE(0, 8, 1)
        TW4_NORM_CASE(0, 5, 2) TW4_NORM_CASE(0, 6, 2) TW4_NORM_CASE(0, 7, 2) TW4_NORM_CASE(0, 8, 2)
        TW4_NORM_ROWS(100, 1, 1, 4) TW4_NORM_ROWS(100, 1, 2, 4) TW4_NORM_CASE(100, 1, 3) TW4_NORM_CASE(100, 2, 2)
        TW4_NORM_CASE(100, 1, 5) TW4_NORM_CASE(100, 3, 2) TW4_NORM_CASE(100, 1, 7) TW4_NORM_CASE(100, 4, 2)
        TW4_NORM_CASE(100, 2, 5) TW4_NORM_CASE(100, 4, 3) TW4_NORM_CASE(100, 7, 2) TW4_NORM_CASE(100, 4, 4)
#undef TW4_NORM_CASE
#undef TW4_NORM_ROWS
        default:
            tw4host::set_error("rms_norm: K = %d is not compiled (K / 512 in 1..8, 10, 12, 14, 16)", K);
            return TW4_EINVAL;
    }
    TW4_LAUNCH_CHECK("rms_norm: launch");
    return TW4_OK;
}

int norm_check(const void* x, const void* r, const void* w, const void* y, int M, int K, const char* who) {
    TW4_REQUIRE(x && r && w && y, TW4_EINVAL, "%s: null pointer", who);
    TW4_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(r) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0,
                TW4_EINVAL, "%s: rows must be 16-byte aligned", who);
    TW4_REQUIRE(M >= 0, TW4_EINVAL, "%s: M >= 0 (M = %d)", who, M);
    TW4_REQUIRE(K >= 512 && K % 512 == 0 && K <= 8192, TW4_EINVAL, "%s: K %% 512 == 0 and K <= 8192 (K = %d)", who,
                K);
    return TW4_OK;
}

}  // namespace tw4

using namespace tw4;

extern "C" int tw4_rms_norm(const uint16_t* x, const uint16_t* weight, uint16_t* y, int M, int K, float eps,
                            void* stream) {
    int rc = norm_check(x, x, weight, y, M, K, "rms_norm");
    if (rc || M == 0) return rc;
    auto xp = const_cast<h1*>(reinterpret_cast<const h1*>(x));  // read only (ADD = false)
    return norm_launch<false>(xp, xp, reinterpret_cast<const h1*>(weight), reinterpret_cast<h1*>(y), M, K, eps,
                              static_cast<hipStream_t>(stream));
}

extern "C" int tw4_add_rms_norm(uint16_t* x, uint16_t* residual, const uint16_t* weight, int M, int K, float eps,
                                void* stream) {
    int rc = norm_check(x, residual, weight, x, M, K, "add_rms_norm");
    if (rc || M == 0) return rc;
    auto xp = reinterpret_cast<h1*>(x);
    return norm_launch<true>(xp, reinterpret_cast<h1*>(residual), reinterpret_cast<const h1*>(weight), xp, M, K, eps,
                             static_cast<hipStream_t>(stream));
}
