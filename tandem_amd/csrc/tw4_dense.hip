// Dense fp16 GEMV for small batches (the lm_head of a W4A16 model and other fp16 projections):
// y[M, N] = x[M, K] @ w[N, K]^T, M <= 8, w row-major (nn.Linear layout), fp32 accumulation.
//
// Bound by streaming w once. A workgroup owns a contiguous block of rows; each wavefront takes
// RB rows at a time and reads each row as K / 512 fully coalesced 1 KB wavefront loads (lane l
// holds chunks l, l + 64, ... of 8 halves, non-temporal). The next RB rows are in flight (second
// register set, loop unrolled by two) while the current ones are reduced. x is staged in LDS once
// per workgroup; lane l reads the same x chunks for every row, so per row it costs M LDS reads of
// 16 bytes per 16 weight bytes (x chunks are read once per row block and shared by its RB rows).
// Each lane accumulates its chunks with v_dot2_f32_f16; a row's 64 partial sums are added with
// DPP (within rows of 16 lanes) and two permlane swaps, and lane 0 writes the RB x M results.
//
// For M = 5 .. 8 the v_dot2 form reads M x 16 bytes of x from LDS per 16 weight bytes, which makes
// it LDS-bound; the matrix-core form (rows_inflight = 16 or 32: one or two 128-k chunks per step in
// flight) takes 16-row tiles of w as the A operand of v_mfma_f32_16x16x32_f16 and x as B, so one
// 16-byte B fragment serves 16 rows.
#include "tw4_lds.h"

namespace tw4 {

// Sum over all 64 lanes, in every lane.
__device__ __forceinline__ float wave_sum(float v) {
    v += lane_xor1(v);
    v += lane_xor2(v);
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, false));  // row_ror:4
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, false));  // row_ror:8
    return sum_rows(v);
}

template <int RB, int J>
struct RowSet {
    u4 w[RB][J];
};

template <int RB, int J>
__device__ __forceinline__ void load_rows(RowSet<RB, J>& rs, const u4* w, int64_t kc, int row, int last_row, int lane) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const u4* p = w + static_cast<int64_t>(min(row + rb, last_row)) * kc + lane;  // past the end: a valid row
#pragma unroll
        for (int j = 0; j < J; ++j) rs.w[rb][j] = load_stream(p + 64 * j);
    }
}

// Rows [row, row + RB) against x (LDS, [MT][K / 8] chunks; rows past M repeat row M - 1): lane 0
// stores y for tokens < M and rows < row_end.
template <bool PF, int M, int RB, int J>
__device__ __forceinline__ void rows_step(const RowSet<RB, J>& cur, RowSet<RB, J>& nxt, const u4* w, int64_t kc,
                                          const u4* xs, h1* y, int N, int Mx, int row, int row_end, int last_row,
                                          int lane) {
    if constexpr (PF) load_rows<RB, J>(nxt, w, kc, row + RB, last_row, lane);
    __builtin_amdgcn_sched_barrier(0);  // keep the prefetch above the math
    float acc[RB][M];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[rb][m] = 0.0f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const u4 xv = xs[m * kc + 64 * j + lane];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                const u4 wv = cur.w[rb][j];
                float a = acc[rb][m];
                a = __builtin_amdgcn_fdot2(bitcast<h2>(wv.x), bitcast<h2>(xv.x), a, false);
                a = __builtin_amdgcn_fdot2(bitcast<h2>(wv.y), bitcast<h2>(xv.y), a, false);
                a = __builtin_amdgcn_fdot2(bitcast<h2>(wv.z), bitcast<h2>(xv.z), a, false);
                a = __builtin_amdgcn_fdot2(bitcast<h2>(wv.w), bitcast<h2>(xv.w), a, false);
                acc[rb][m] = a;
            }
        }
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float v = wave_sum(acc[rb][m]);
            if (lane == 0 && m < Mx && row + rb < row_end) y[static_cast<int64_t>(m) * N + row + rb] = static_cast<h1>(v);
        }
}

// J = K / 512 chunk loads per lane and row (K <= 4096 here); M tokens of x in LDS, 1 <= Mx <= M.
template <int M, int RB, int J>
__global__ void __launch_bounds__(256) dense_gemv_kernel(const h1* __restrict__ x, const u4* __restrict__ w,
                                                         h1* __restrict__ y, int Mx, int N, int rows_per_wave) {
    extern __shared__ u4 xs[];
    constexpr int kc = 64 * J;  // 16-byte chunks per row
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = (blockIdx.x * 4 + wave) * rows_per_wave;
    const int row_end = min(row0 + rows_per_wave, N);
    const int nblk = row_end > row0 ? (row_end - row0 + RB - 1) / RB : 0;

    RowSet<RB, J> a, b;
    if (nblk > 0) load_rows<RB, J>(a, w, kc, row0, N - 1, lane);
    // x -> LDS, all waves of the workgroup (M kc chunks)
    const u4* xg = reinterpret_cast<const u4*>(x);
    for (int c = threadIdx.x; c < M * kc; c += 256) {
        const int m = c / kc;  // kc is a power of two
        xs[c] = xg[static_cast<int64_t>(min(m, Mx - 1)) * kc + (c - m * kc)];
    }
    __syncthreads();

    int i = 0;
    for (; i + 2 < nblk; i += 2) {
        rows_step<true, M, RB, J>(a, b, w, kc, xs, y, N, Mx, row0 + RB * i, row_end, N - 1, lane);
        rows_step<true, M, RB, J>(b, a, w, kc, xs, y, N, Mx, row0 + RB * (i + 1), row_end, N - 1, lane);
    }
    if (i + 2 == nblk) {
        rows_step<true, M, RB, J>(a, b, w, kc, xs, y, N, Mx, row0 + RB * i, row_end, N - 1, lane);
        rows_step<false, M, RB, J>(b, a, w, kc, xs, y, N, Mx, row0 + RB * (i + 1), row_end, N - 1, lane);
    } else if (i + 1 == nblk) {
        rows_step<false, M, RB, J>(a, b, w, kc, xs, y, N, Mx, row0 + RB * i, row_end, N - 1, lane);
    }
}

// ------------------------------------------------------------------------- matrix cores, M <= 8
// A wavefront owns rows_per_wave rows (whole 16-row tiles) and walks them tile by tile, each over
// all of K in chunks of 128 k. Lane (kb, r) loads, for word s = 0..3 of a chunk, the 16 bytes of
// row r at k = 128 c + 8 (4 s + kb) .. + 7 (one instruction per s: 64 contiguous bytes per row), and
// feeds them as A row r; the B fragment of token r is x at the same k from LDS, so each MFMA sums 32
// distinct k of the chunk. D chunks form a step: the next step's D chunks (possibly the next tile's
// first) are in flight in a second register set while the current ones are multiplied, 4 D KB per
// wavefront. D holds rows 4 kb + i of token r in lane (kb, r).
// x: 8 token rows in LDS (rows past M repeat row M - 1; B columns r >= 8 read row 7 and feed D
// columns that are never stored), row stride K / 8 + 1 chunks so the 16 rows of a fragment read hit
// different banks. Staged once per workgroup, its loads issued before the first weight chunks.
constexpr int kMmaWaves = 8;  // wavefronts per workgroup of the matrix-core form (one x copy each)

template <int D>
struct ChunkSet {
    u4 w[D][4];
};

// Plain (cached) loads: an instruction reads 64 bytes of each of 16 rows, half of a 128-byte line whose
// other half the next word's load reads (with non-temporal loads the tile ran 2 % slower).
template <int D>
__device__ __forceinline__ void load_chunks16(ChunkSet<D>& cs, const u4* wrow, int c, int kb) {
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
        for (int s = 0; s < 4; ++s) cs.w[d][s] = wrow[16 * (c + d) + 4 * s + kb];
}

template <bool PF, int D>
__device__ __forceinline__ void mma16_step(const ChunkSet<D>& cur, ChunkSet<D>& nxt, const u4* nrow, int nc,
                                           const u4* xr, int c, int kb, f4& acc) {
    if constexpr (PF) load_chunks16<D>(nxt, nrow, nc, kb);
    __builtin_amdgcn_sched_barrier(0);  // keep the prefetch above the math
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
        for (int s = 0; s < 4; ++s)
            acc = mfma16x16x32(bitcast<h8>(cur.w[d][s]), bitcast<h8>(xr[16 * (c + d) + 4 * s + kb]), acc);
}

// J = K / 512 x chunks per thread for the staging (K <= 4096: at most 8); D = chunks per step, with
// 2 D <= 4 J (the K / 128 chunks of a row are a whole, even number of steps).
template <int J, int D>
__global__ void __launch_bounds__(kMmaWaves * 64) dense_mma_kernel(const h1* __restrict__ x, const u4* __restrict__ w,
                                                                   h1* __restrict__ y, int Mx, int N,
                                                                   int rows_per_wave) {
    extern __shared__ u4 xs[];
    constexpr int kc = 64 * J;  // 16-byte chunks per row of x and w
    constexpr int C = kc / 16;  // 128-k chunks per row
    static_assert(C % (2 * D) == 0, "a row is an even number of D-chunk steps");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, kb = lane >> 4;
    const int row0 = (blockIdx.x * kMmaWaves + wave) * rows_per_wave;
    const int tiles = (max(min(rows_per_wave, N - row0), 0) + 15) >> 4;  // the last one may be partial
    const int last_tile = max(tiles - 1, 0);
    auto wrow = [&](int t) {  // this lane's row of tile t (rows past N read row N - 1)
        return w + static_cast<int64_t>(min(row0 + 16 * t + r, N - 1)) * kc;
    };

    // x staging: thread i takes chunks i, i + 512, ... (J of them) of the 8 x kc token-row image
    const u4* xg = reinterpret_cast<const u4*>(x);
    u4 xv[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int f = threadIdx.x + kMmaWaves * 64 * j;  // < 8 kc
        const int m = f / kc;                            // kc is a power of two
        xv[j] = xg[static_cast<int64_t>(min(m, Mx - 1)) * kc + (f - m * kc)];
    }
    __builtin_amdgcn_sched_barrier(0);
    ChunkSet<D> a, b;
    load_chunks16<D>(a, wrow(0), 0, kb);  // tiles == 0: a valid row, never used
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int f = threadIdx.x + kMmaWaves * 64 * j;
        const int m = f / kc;
        xs[m * (kc + 1) + (f - m * kc)] = xv[j];
    }
    __syncthreads();

    const u4* xr = xs + min(r, 7) * (kc + 1);
    for (int t = 0; t < tiles; ++t) {
        const u4* cr = wrow(t);
        const u4* nr = wrow(min(t + 1, last_tile));  // the last tile prefetches its own first step: unused
        f4 acc = f4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int c = 0; c < C - 2 * D; c += 2 * D) {
            mma16_step<true, D>(a, b, cr, c + D, xr, c, kb, acc);
            mma16_step<true, D>(b, a, cr, c + 2 * D, xr, c + D, kb, acc);
        }
        mma16_step<true, D>(a, b, cr, C - D, xr, C - 2 * D, kb, acc);
        mma16_step<true, D>(b, a, nr, 0, xr, C - D, kb, acc);
        const int n = row0 + 16 * t + 4 * kb;
        if (r < Mx && n < N) {
            h1* yp = y + static_cast<int64_t>(r) * N + n;
            if (n + 3 < N && (N & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 7) == 0) {
                *reinterpret_cast<h4*>(yp) = h4{static_cast<h1>(acc.x), static_cast<h1>(acc.y),
                                                static_cast<h1>(acc.z), static_cast<h1>(acc.w)};
            } else {
                const float v[4] = {acc.x, acc.y, acc.z, acc.w};
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < N) yp[i] = static_cast<h1>(v[i]);
            }
        }
    }
}

// ------------------------------------------------------------------- matrix cores through LDS, M <= 32
// y = x w^T for a batch of up to 32 tokens, bound by streaming w once. Both operands go through LDS by direct-to-LDS
// loads in a ring of R stages of 64 k, so the loads of w are whole 128-byte lines (the form above reads 64 bytes of
// 16 rows 2 K bytes apart per instruction), no register holds data in flight, and x is read from LDS by the four
// wavefronts, 16 rows of w each.
//   A persistent workgroup owns a contiguous, even share of the 16-row tiles (a grid of one workgroup per 64 rows leaves
//   its last round nearly empty), and walks it in passes of 64 rows; the stages of all passes form one sequence, so the
//   loads of the next pass are in flight under the end of this one. Rows past the share repeat its last one (cached; never
//   stored).
//   A stage: 64 rows of w and 16 MT of x, 128 bytes per row, 8 rows per load instruction; 16-byte chunk c of row rho at
//   position c ^ ((rho >> 1) & 7), so the 16 rows of a fragment read touch every bank once.
//   Lane (q, r) feeds A row r and B column r chunk 4 j + q at substep j. D lane (q, r): rows 4 q + i of token r.
// What is left to the floor is x: 64 rows of w take 16 MT K 2 bytes of it from L2. Measured on the Qwen3-8B head
// (4096 x 151936, floor at 7.1 TB/s 175 us), hipBLASLt in the same run in brackets: M = 8 197 us (248; the form above 231),
// 24 212 (260), 32 221 (265). Timed and not kept: passes of 128 rows (two tiles per wavefront: half of x's traffic, but a
// ring of 4; M = 8 218 against 204, M = 24 226 against 214 in one run), a ring of 4 stages (209, 218), and 48 and 64 tokens
// (254 and 273: level with hipBLASLt).
template <int MT, int R>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
dense_skinny_kernel(const h1* __restrict__ x, const h1* __restrict__ w, h1* __restrict__ y, int M, int N, int K) {
    constexpr int ROWS = 64;                  // rows of w per pass
    constexpr int XL = 2 * MT;                // 1 KB loads of x per stage, 8 rows each
    constexpr int XI = (XL + 3) / 4, WI = 2;  // per wavefront (the last ones may repeat a load of x)
    constexpr int SLOT = (ROWS + 16 * MT) * 8;
    __shared__ u4 ring[R * SLOT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int tiles = (N + 15) >> 4;
    const int t0 = static_cast<int>(static_cast<int64_t>(blockIdx.x) * tiles / gridDim.x);
    const int t1 = static_cast<int>(static_cast<int64_t>(blockIdx.x + 1) * tiles / gridDim.x);
    const int row_end = min(16 * t1, N), passes = (t1 - t0 + 3) >> 2, ks = K >> 6;
    if (passes == 0) return;

    const u4 xr = lds_rsrc(x);
    u4 wr = lds_rsrc(w);
    const int rho = lane >> 3;  // row of this lane within a load
    uint32_t xoff[XI], woff[WI];
    const int xj = min(wave * XI, XL - XI);
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int row = 8 * (xj + i) + rho;
        xoff[i] = static_cast<uint32_t>(min(row, M - 1)) * K * 2u + 16u * ((lane & 7) ^ ((row >> 1) & 7));
    }
    auto pass_rows = [&](int p) {
#pragma unroll
        for (int i = 0; i < WI; ++i) {
            const int row = 8 * (wave * WI + i) + rho;
            woff[i] = static_cast<uint32_t>(min(16 * t0 + ROWS * p + row, row_end - 1)) * static_cast<uint32_t>(K) * 2u +
                      16u * ((lane & 7) ^ ((row >> 1) & 7));
        }
    };
    pass_rows(0);
    const uint32_t ring_addr = static_cast<uint32_t>(reinterpret_cast<size_t>((lds_void*)ring));
    const uint32_t wbase = ring_addr + 1024 * wave * WI, xbase = ring_addr + 16 * 8 * ROWS + 1024 * xj;

    int ip = 0, is = 0, islot = 0;  // the next stage to issue: pass, stage of the pass, ring slot
    auto issue = [&]() {
        const uint32_t s = 16 * SLOT * islot, soff = 128 * is;
        lds_dma16<0, true>(wr, woff[0], soff, wbase + s);
        lds_dma16<1024, true>(wr, woff[1], soff, wbase + s);
        lds_dma16<0>(xr, xoff[0], soff, xbase + s);
        islot = islot + 1 == R ? 0 : islot + 1;
        if (++is == ks) {
            is = 0, ++ip;
            if (ip < passes)
                pass_rows(ip);
            else
                wr.z = 0;  // past the end: empty loads keep the counts
        }
    };
#pragma unroll
    for (int i = 0; i < R - 1; ++i) issue();

    // fragment addresses in a slot (16-byte units): substep j at ^ 4 (chunk 4 j + q)
    const int sw = (r >> 1) & 7;
    const int wl = (16 * wave + r) * 8, xl = ROWS * 8 + r * 8;
    const int c0 = q ^ sw, c1 = (q + 4) ^ sw;
    int slot = 0;
    for (int p = 0; p < passes; ++p) {
        f4 acc[MT];
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[b] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int s = 0; s < ks; ++s) {
            wait_stage<(R - 2) * (XI + WI)>();  // this stage has landed (the stores of a pass's end only make it stricter)
            ring_barrier();                     // in every wavefront, and nobody reads the slot of the stage before any more
            issue();
            const u4* sl = ring + slot * SLOT;
            slot = slot + 1 == R ? 0 : slot + 1;
            const h8 a0 = bitcast<h8>(sl[wl + c0]), a1 = bitcast<h8>(sl[wl + c1]);
            h8 b0[MT], b1[MT];
#pragma unroll
            for (int b = 0; b < MT; ++b) b0[b] = bitcast<h8>(sl[xl + 128 * b + c0]), b1[b] = bitcast<h8>(sl[xl + 128 * b + c1]);
#pragma unroll
            for (int b = 0; b < MT; ++b) acc[b] = mfma16x16x32(a0, b0[b], acc[b]);
#pragma unroll
            for (int b = 0; b < MT; ++b) acc[b] = mfma16x16x32(a1, b1[b], acc[b]);
        }
        const bool wide = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & 7) == 0;
        const int n = 16 * t0 + ROWS * p + 16 * wave + 4 * q;
#pragma unroll
        for (int b = 0; b < MT; ++b) {
            const int m = 16 * b + r;
            if (m >= M || n >= row_end) continue;
            h1* yp = y + static_cast<int64_t>(m) * N + n;
            const f4 v = acc[b];
            if (wide) {  // n + 3 < row_end: both are multiples of 4
                *reinterpret_cast<h4*>(yp) = h4{static_cast<h1>(v.x), static_cast<h1>(v.y), static_cast<h1>(v.z), static_cast<h1>(v.w)};
            } else {
                const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (n + i < row_end) yp[i] = static_cast<h1>(e[i]);
            }
        }
    }
    wait_stage<0>();  // the empty loads past the end still write their slots
}

// Compiled (rows in flight RB, rows per wavefront) configurations.
#define TW4_DENSE_CONFIGS(X) X(1, 16) X(1, 32) X(2, 16) X(2, 32) X(2, 64) X(4, 32) X(4, 64)
// Matrix-core form (for tables that callers name it in: the M <= 32 kernel above is faster, 197 against 231 us on the Qwen3-8B
// head at M = 8; rows_inflight 16 D: 16-row tiles, D chunks of 128 k per step in flight): rows
// per wavefront, whole 16-row tiles.
// (4 chunks per step ran 5-30 % slower on the Qwen3 lm_heads: no configuration compiled.)
#define TW4_DENSE_MMA_CONFIGS(X) X(16, 16) X(16, 32) X(16, 64) X(16, 128) X(32, 16) X(32, 32)

template <int M, int RB, int J>
int dense_launch(const h1* x, const u4* w, h1* y, int Mx, int N, int rows_per_wave, hipStream_t st) {
    const int64_t waves = (static_cast<int64_t>(N) + rows_per_wave - 1) / rows_per_wave;
    const unsigned grid = static_cast<unsigned>((waves + 3) / 4);
    const size_t lds = static_cast<size_t>(M) * 64 * J * 16;  // <= 64 KB
    dense_gemv_kernel<M, RB, J><<<grid, 256, lds, st>>>(x, w, y, Mx, N, rows_per_wave);
    TW4_LAUNCH_CHECK("gemv_f16: launch");
    return TW4_OK;
}

template <int M, int RB>
int dense_by_k(const h1* x, const u4* w, h1* y, int Mx, int N, int K, int rows_per_wave, hipStream_t st) {
    switch (K >> 9) {
        case 1: return dense_launch<M, RB, 1>(x, w, y, Mx, N, rows_per_wave, st);
        case 2: return dense_launch<M, RB, 2>(x, w, y, Mx, N, rows_per_wave, st);
        case 4: return dense_launch<M, RB, 4>(x, w, y, Mx, N, rows_per_wave, st);
        case 8: return dense_launch<M, RB, 8>(x, w, y, Mx, N, rows_per_wave, st);
        default: break;
    }
    tw4host::set_error("gemv_f16: K = %d (K in 512, 1024, 2048, 4096)", K);
    return TW4_EINVAL;
}

template <int J, int D>
int dense_mma_launch(const h1* x, const u4* w, h1* y, int Mx, int N, int rows_per_wave, hipStream_t st) {
    const int64_t waves = (static_cast<int64_t>(N) + rows_per_wave - 1) / rows_per_wave;
    const unsigned grid = static_cast<unsigned>((waves + kMmaWaves - 1) / kMmaWaves);
    const size_t lds = static_cast<size_t>(8) * (64 * J + 1) * 16;  // <= 65.7 KB
    dense_mma_kernel<J, D><<<grid, kMmaWaves * 64, lds, st>>>(x, w, y, Mx, N, rows_per_wave);
    TW4_LAUNCH_CHECK("gemv_f16: launch");
    return TW4_OK;
}

template <int D>
int dense_mma(const h1* x, const u4* w, h1* y, int M, int N, int K, int rows_per_wave, hipStream_t st) {
    if (K / 128 < 2 * D) {
        tw4host::set_error("gemv_f16: rows in flight %d need K >= %d (K = %d)", 16 * D, 256 * D, K);
        return TW4_ECONFIG;
    }
    switch (K >> 9) {
        case 1: if constexpr (D <= 2) return dense_mma_launch<1, D>(x, w, y, M, N, rows_per_wave, st); break;
        case 2: return dense_mma_launch<2, D>(x, w, y, M, N, rows_per_wave, st);
        case 4: return dense_mma_launch<4, D>(x, w, y, M, N, rows_per_wave, st);
        case 8: return dense_mma_launch<8, D>(x, w, y, M, N, rows_per_wave, st);
        default: break;
    }
    tw4host::set_error("gemv_f16: K = %d (K in 512, 1024, 2048, 4096)", K);
    return TW4_EINVAL;
}

template <int MT, int R>
int skinny_launch(const h1* x, const h1* w, h1* y, int M, int N, int K, hipStream_t st) {
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return tw4host::hip_fail(e, "gemm_f16: device");
    const int tiles = (N + 15) >> 4;
    const int grid = tiles < 2 * cus ? tiles : 2 * cus;  // two workgroups fit a CU's LDS
    dense_skinny_kernel<MT, R><<<static_cast<unsigned>(grid), 256, 0, st>>>(x, w, y, M, N, K);
    TW4_LAUNCH_CHECK("gemm_f16: launch");
    return TW4_OK;
}

template <int RB>
int dense_by_m(const h1* x, const u4* w, h1* y, int M, int N, int K, int rows_per_wave, hipStream_t st) {
    if (M == 1) return dense_by_k<1, RB>(x, w, y, M, N, K, rows_per_wave, st);
    if (M == 2) return dense_by_k<2, RB>(x, w, y, M, N, K, rows_per_wave, st);
    if (M <= 4) return dense_by_k<4, RB>(x, w, y, M, N, K, rows_per_wave, st);
    return dense_by_k<8, RB>(x, w, y, M, N, K, rows_per_wave, st);  // token rows past M repeat row M - 1
}

}  // namespace tw4

using namespace tw4;

extern "C" int tw4_gemv_f16(const uint16_t* x, const uint16_t* w, uint16_t* y, int M, int N, int K, int rows_inflight,
                            int rows_per_wave, void* stream) {
    TW4_REQUIRE(x && w && y, TW4_EINVAL, "gemv_f16: null pointer");
    TW4_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0, TW4_EINVAL,
                "gemv_f16: x and w must be 16-byte aligned");
    TW4_REQUIRE(reinterpret_cast<uintptr_t>(y) % 2 == 0, TW4_EINVAL, "gemv_f16: y must be 2-byte aligned");
    TW4_REQUIRE(M >= 1 && M <= 8, TW4_EINVAL, "gemv_f16: 1 <= M <= 8 (M = %d)", M);
    TW4_REQUIRE(N >= 1, TW4_EINVAL, "gemv_f16: N >= 1 (N = %d)", N);
    TW4_REQUIRE(K == 512 || K == 1024 || K == 2048 || K == 4096, TW4_EINVAL,
                "gemv_f16: K in 512, 1024, 2048, 4096 (K = %d)", K);
    auto xp = reinterpret_cast<const h1*>(x);
    auto wp = reinterpret_cast<const u4*>(w);
    auto yp = reinterpret_cast<h1*>(y);
    auto st = static_cast<hipStream_t>(stream);
#define TW4_DENSE_CASE(RB, RPW) \
    if (rows_inflight == RB && rows_per_wave == RPW) return dense_by_m<RB>(xp, wp, yp, M, N, K, RPW, st);
    TW4_DENSE_CONFIGS(TW4_DENSE_CASE)
#undef TW4_DENSE_CASE
#define TW4_DENSE_MMA_CASE(RB, RPW) \
    if (rows_inflight == RB && rows_per_wave == RPW) return dense_mma<RB / 16>(xp, wp, yp, M, N, K, RPW, st);
    TW4_DENSE_MMA_CONFIGS(TW4_DENSE_MMA_CASE)
#undef TW4_DENSE_MMA_CASE
    tw4host::set_error("gemv_f16: unsupported rows in flight / rows per wavefront %d / %d", rows_inflight,
                       rows_per_wave);
    return TW4_ECONFIG;
}

extern "C" int tw4_gemv_f16_configs(int* out, int max_configs) {
    int n = 0;
#define TW4_LIST(RB, RPW)                 \
    if (out && n < max_configs) {         \
        out[2 * n] = RB;                  \
        out[2 * n + 1] = RPW;             \
    }                                     \
    ++n;
    TW4_DENSE_CONFIGS(TW4_LIST)
    TW4_DENSE_MMA_CONFIGS(TW4_LIST)
#undef TW4_LIST
    return n;
}

extern "C" int tw4_gemm_f16(const uint16_t* x, const uint16_t* w, uint16_t* y, int M, int N, int K, void* stream) {
    TW4_REQUIRE(x && w && y, TW4_EINVAL, "gemm_f16: null pointer");
    TW4_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0, TW4_EINVAL,
                "gemm_f16: x and w must be 16-byte aligned");
    TW4_REQUIRE(reinterpret_cast<uintptr_t>(y) % 2 == 0, TW4_EINVAL, "gemm_f16: y must be 2-byte aligned");
    TW4_REQUIRE(M >= 1 && M <= 32, TW4_EINVAL, "gemm_f16: 1 <= M <= 32 (M = %d)", M);
    TW4_REQUIRE(N >= 1, TW4_EINVAL, "gemm_f16: N >= 1 (N = %d)", N);
    TW4_REQUIRE(K >= 64 && K % 64 == 0, TW4_EINVAL, "gemm_f16: K %% 64 == 0 (K = %d)", K);
    TW4_REQUIRE(static_cast<int64_t>(N) * K < (1LL << 31) && static_cast<int64_t>(M) * K < (1LL << 31), TW4_EINVAL,
                "gemm_f16: N K < 2^31 (N %d, K %d)", N, K);  // the loads' byte offsets are 32-bit
    auto xp = reinterpret_cast<const h1*>(x);
    auto wp = reinterpret_cast<const h1*>(w);
    auto yp = reinterpret_cast<h1*>(y);
    auto st = static_cast<hipStream_t>(stream);
    return M <= 16 ? skinny_launch<1, 7>(xp, wp, yp, M, N, K, st) : skinny_launch<2, 6>(xp, wp, yp, M, N, K, st);
}
