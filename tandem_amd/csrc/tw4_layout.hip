// Load-time repack (AutoAWQ "gemm" tensors -> tile layout) and the dense dequantization
// (tile layout -> fp16 [N, K]).
//
// AutoAWQ packs output columns c = 0..7 of an int32 in nibble order [0, 2, 4, 6, 1, 3, 5, 7],
// so column c sits in nibble kAwqReverse[c] (python/tandem/layers/awq.py:38-46).
#include "tw4_common.h"

namespace tw4 {

__constant__ int kAwqReverse[8] = {0, 4, 1, 5, 2, 6, 3, 7};

// Repack: a workgroup takes one quant group (128 k) of 256 columns (16 row tiles, or 32 half tiles of an interleaved
// layer). It is bound by memory: every input and output byte moves once, in whole lines on both sides.
//   in:  16 bytes (4 words, 32 columns) per thread, a row's 128 bytes by eight threads, into LDS rows of 36 words (the
//        two 8-row blocks a wavefront reads below then sit in different halves of the banks).
//   out: a thread transposes the 8 x 8 nibbles of (8 k, 8 columns) in registers; the 8 words go through LDS into block
//        order (16-byte chunk c of tile t at c ^ t: the 16 tiles of one chunk in different banks), and every wavefront
//        writes whole 1 KB blocks (tile, group) with one 16-byte store per lane (interleaved: two half blocks of 128-byte
//        pieces). A partial last tile's rows past N are written as zeros.
//   params: thread t the column's scale and zero of the group.
// Against one thread per (8 k, 8 columns), whose eight 4-byte stores left 16 bytes between them (a line took 32 partial
// writes), after a fill of the whole output and with the parameters in a launch of their own: Qwen3-8B gate_up
// (4096 x 24576), all of it, 76 -> 24.3 us (4.35 TB/s of the int4 in and out).
constexpr int kRepackCols = 256;

__global__ void __launch_bounds__(256) repack_kernel(const uint32_t* __restrict__ qweight, const uint32_t* __restrict__ qzeros,
                                                     const h1* __restrict__ scales, uint32_t* __restrict__ packed,
                                                     h1* __restrict__ s_out, h1* __restrict__ z_out, int K, int N, int cbs,
                                                     int interleave, int wide_in, int wide_out) {
    constexpr int S = 36;
    __shared__ __attribute__((aligned(16))) uint32_t in[128 * S];
    __shared__ u4 out[16 * kBlockU4];
    const int tid = threadIdx.x, n8 = N >> 3, G = K >> 7;
    const int g = blockIdx.x / cbs, cb = blockIdx.x - g * cbs;
    const int c0 = 32 * cb + 4 * (tid & 7);  // this thread's 4 words of a row
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int k = 32 * i + (tid >> 3);
        const uint32_t* src = qweight + static_cast<int64_t>(128 * g + k) * n8 + c0;
        u4 v{};
        if (wide_in) {  // rows 16-byte aligned: n8 % 4 == 0, so a thread's words are all in or all out
            if (c0 < n8) v = load_stream(reinterpret_cast<const u4*>(src));
        } else {
            if (c0 < n8) v.x = src[0];
            if (c0 + 1 < n8) v.y = src[1];
            if (c0 + 2 < n8) v.z = src[2];
            if (c0 + 3 < n8) v.w = src[3];
        }
        *reinterpret_cast<u4*>(in + S * k + 4 * (tid & 7)) = v;
    }
    const int col = kRepackCols * cb + tid;  // the group parameters of one column
    if (col < N) {
        const uint32_t zw = qzeros[static_cast<int64_t>(g) * n8 + (col >> 3)];
        const int z = static_cast<int>((zw >> (4 * kAwqReverse[col & 7])) & 0xFu);
        const int64_t o = param_offset(interleave ? interleaved_dest_row(col, N) : col, g, N, G);
        s_out[o] = scales[static_cast<int64_t>(g) * N + col];
        z_out[o] = static_cast<h1>(static_cast<float>(z));
    }
    __syncthreads();
    uint32_t* ow = reinterpret_cast<uint32_t*>(out);
#pragma unroll
    for (int i = 0; i < 2; ++i) {  // (kq: 8 k, c8: 8 columns)
        const int c8 = tid & 31, kq = 8 * i + (tid >> 5), t = c8 >> 1;
        uint32_t src[8];
#pragma unroll
        for (int o = 0; o < 8; ++o) src[o] = in[S * (8 * kq + o) + c8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int shift = 4 * kAwqReverse[c];
            uint32_t word = 0;
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const uint32_t q = (src[o] >> shift) & 0xFu;
                word |= q << (4 * ((o >> 1) + 4 * (o & 1)));  // weight o = 2 q' + e in nibble q' + 4 e
            }
            const int chunk = (kq >> 2) * 16 + 8 * (c8 & 1) + c;  // 16 kb + row
            ow[t * kBlockWords + (chunk ^ t) * 4 + (kq & 3)] = word;
        }
    }
    __syncthreads();
    const int wave = tid >> 6, lane = tid & 63, tiles = (N + 15) >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int t = 4 * i + wave, tg = 16 * cb + t;
        if (tg >= tiles) continue;
        const u4 v = out[t * kBlockU4 + (lane ^ t)];
        int64_t dst = (static_cast<int64_t>(tg) * G + g) * kBlockU4 + lane;
        if (interleave) {  // rows 8 h .. 8 h + 7 of this LDS tile are a half of another tile
            const int d = interleaved_dest_row(16 * tg + (lane & 15), N);
            dst = (static_cast<int64_t>(d >> 4) * G + g) * kBlockU4 + (lane & 48) + (d & 15);
        }
        if (wide_out) {
            reinterpret_cast<u4*>(packed)[dst] = v;
        } else {
            packed[4 * dst] = v.x, packed[4 * dst + 1] = v.y, packed[4 * dst + 2] = v.z, packed[4 * dst + 3] = v.w;
        }
    }
}

// Dense weights: a workgroup takes 16 rows (one tile) x 512 k (four groups; fewer at the end of a row), a wavefront one
// group of 128 k: each lane dequantizes its 16 bytes (32 weights of one row) and parks them in LDS, and the workgroup
// writes the 16 rows' 1 KB pieces with whole lines per instruction (a wavefront store is one row's 1 KB). LDS rows are 65
// chunks of 16 bytes, so the 16 rows of a column of chunks sit in different banks.
// Bound by memory. Against four 16-byte stores per lane 64 bytes apart: Qwen3-8B down (12288 x 4096) 36.5 -> 22.3 us
// (5.9 TB/s), gate_up (4096 x 24576) 74 -> 41.
// STREAM: non-temporal stores, for a matrix that is kept or exceeds the 256 MB cache in front of HBM. Plain ones leave a smaller
// one there for the product that reads it next: dequantize + product of 5120 x 7168 at M = 4096 259 -> 234 us (244 with the
// strided stores), 17408 x 5120 at M = 100 183 -> 144; the dequantization alone takes up to 15 % longer (4096 x 6144 11.2 -> 12.9).
// 5120 x 34816 (356 MB) is faster non-temporal all the way: 1303 against 1320 at M = 4096.
template <bool STREAM>
__global__ void __launch_bounds__(256) dequant_kernel(const u4* __restrict__ packed, const h1* __restrict__ scales,
                                                      const h1* __restrict__ zeros, u4* __restrict__ out, int N, int K,
                                                      int pieces, int deinterleave) {
    __shared__ u4 tile[16 * 65];
    const int G = K >> 7;
    const int t = blockIdx.x / pieces, g0 = 4 * (blockIdx.x - t * pieces), wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 15, kb = lane >> 4, g = g0 + wave;
    const int rows = tile_rows(t, N);
    if (g < G) {
        const u4 v = load_stream(packed + (static_cast<int64_t>(t) * G + g) * kBlockU4 + lane);
        const int64_t sidx = static_cast<int64_t>(16) * t * G + static_cast<int64_t>(g) * rows + min(r, rows - 1);
        const GroupQ p = group_q(scales[sidx], zeros[sidx]);
        const uint32_t magic = magic_reg();
        u4* d = tile + 65 * r + 16 * wave + 4 * kb;
        d[0] = bitcast<u4>(dequant_word(v.x, p, magic));
        d[1] = bitcast<u4>(dequant_word(v.y, p, magic));
        d[2] = bitcast<u4>(dequant_word(v.z, p, magic));
        d[3] = bitcast<u4>(dequant_word(v.w, p, magic));
    }
    __syncthreads();
    const int chunks = min(G - g0, 4) * 16;  // 16-byte chunks of a row's piece
    if (lane < chunks) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int rr = 4 * wave + i, row = 16 * t + rr;
            if (rr >= rows) break;
            const int dst = deinterleave ? interleaved_source_row(row, N) : row;
            u4* o = out + static_cast<int64_t>(dst) * (K >> 3) + 16 * g0 + lane;
            if constexpr (STREAM)
                __builtin_nontemporal_store(tile[65 * rr + lane], o);
            else
                *o = tile[65 * rr + lane];
        }
    }
}

}  // namespace tw4

using namespace tw4;

extern "C" int tw4_repack_awq(const int32_t* qweight, const int32_t* qzeros, const uint16_t* scales,
                              int32_t* packed, uint16_t* scales_out, uint16_t* zeros_out, int K, int N,
                              int interleave, void* stream) {
    TW4_REQUIRE(K > 0 && K % 128 == 0, TW4_EINVAL, "repack_awq: K %% 128 == 0 (K = %d, group 128 only)", K);
    TW4_REQUIRE(N > 0 && N % 8 == 0, TW4_EINVAL, "repack_awq: N %% 8 == 0 (N = %d)", N);
    TW4_REQUIRE(!interleave || N % 16 == 0, TW4_EINVAL, "repack_awq: interleave needs N %% 16 == 0 (N = %d)", N);
    TW4_REQUIRE(qweight && qzeros && scales && packed && scales_out && zeros_out, TW4_EINVAL,
                "repack_awq: null pointer");
    auto st = static_cast<hipStream_t>(stream);
    const int cbs = (N + kRepackCols - 1) / kRepackCols;
    const int64_t blocks = static_cast<int64_t>(cbs) * (K >> 7);
    TW4_REQUIRE(blocks < (1LL << 31), TW4_EINVAL, "repack_awq: grid too large");
    // 16-byte loads and stores where the rows and the output allow them
    const int wide_in = (N >> 3) % 4 == 0 && reinterpret_cast<uintptr_t>(qweight) % 16 == 0;
    const int wide_out = reinterpret_cast<uintptr_t>(packed) % 16 == 0;
    repack_kernel<<<static_cast<unsigned>(blocks), 256, 0, st>>>(
        reinterpret_cast<const uint32_t*>(qweight), reinterpret_cast<const uint32_t*>(qzeros),
        reinterpret_cast<const h1*>(scales), reinterpret_cast<uint32_t*>(packed), reinterpret_cast<h1*>(scales_out),
        reinterpret_cast<h1*>(zeros_out), K, N, cbs, interleave, wide_in, wide_out);
    TW4_LAUNCH_CHECK("repack_awq: launch");
    return TW4_OK;
}

template <bool STREAM>
static int dequant_launch(const int32_t* packed, const uint16_t* scales, const uint16_t* zeros, uint16_t* out,
                           int N, int K, int deinterleave, void* stream) {
    TW4_REQUIRE(K > 0 && K % 128 == 0, TW4_EINVAL, "dequant: K %% 128 == 0 (K = %d)", K);
    TW4_REQUIRE(N > 0 && N % 8 == 0, TW4_EINVAL, "dequant: N %% 8 == 0 (N = %d)", N);
    TW4_REQUIRE(!deinterleave || N % 16 == 0, TW4_EINVAL, "dequant: deinterleave needs N %% 16 == 0 (N = %d)", N);
    TW4_REQUIRE(packed && scales && zeros && out, TW4_EINVAL, "dequant: null pointer");
    TW4_REQUIRE(reinterpret_cast<uintptr_t>(packed) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0,
                TW4_EINVAL, "dequant: packed and out must be 16-byte aligned");
    const int pieces = ((K >> 7) + 3) / 4;
    const int64_t blocks = static_cast<int64_t>((N + 15) >> 4) * pieces;
    TW4_REQUIRE(blocks < (1LL << 31), TW4_EINVAL, "dequant: grid too large");
    dequant_kernel<STREAM><<<static_cast<unsigned>(blocks), 256, 0, static_cast<hipStream_t>(stream)>>>(
        reinterpret_cast<const u4*>(packed), reinterpret_cast<const h1*>(scales), reinterpret_cast<const h1*>(zeros),
        reinterpret_cast<u4*>(out), N, K, pieces, deinterleave);
    TW4_LAUNCH_CHECK("dequant: launch");
    return TW4_OK;
}

extern "C" int tw4_dequant(const int32_t* packed, const uint16_t* scales, const uint16_t* zeros, uint16_t* out, int N, int K,
                           int deinterleave, void* stream) {
    return dequant_launch<true>(packed, scales, zeros, out, N, K, deinterleave, stream);
}

extern "C" int tw4_dequant_near(const int32_t* packed, const uint16_t* scales, const uint16_t* zeros, uint16_t* out, int N,
                                int K, int deinterleave, void* stream) {
    return dequant_launch<false>(packed, scales, zeros, out, N, K, deinterleave, stream);
}
