// Attention over a one-token context: the softmax over a single key is 1, so query head h of a token takes the value row
// of its KV head (grouped-query attention):
//
//   y[m, h D + d] = qkv[m, (heads + kv_heads) D + (h / (heads / kv_heads)) D + d]
//
// One 16-byte chunk per thread. At a decode batch it moves a few KB and is bound by its launch and one round trip to
// memory, past it by the output's bytes. The general strided copy it replaces takes 3.9-4.3 us there, most of it offset arithmetic
// over four dimensions; the Qwen3-8B decode step (36 copies) at M = 1 went from 1363 to 1274 us with it, Qwen3-1.7B
// at M = 5 from 887 to 845.
#include "tw4_common.h"

namespace tw4 {

__global__ void __launch_bounds__(256) attend_kernel(const u4* __restrict__ v, u4* __restrict__ y, int chunks, int row_chunks,
                                                     int src_chunks, int head_chunks, int group) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= chunks) return;
    const int m = i / row_chunks, c = i - m * row_chunks;  // chunk c of token m's output row
    const int h = c / head_chunks, kv = h / group;
    y[i] = v[static_cast<int64_t>(m) * src_chunks + kv * head_chunks + (c - h * head_chunks)];
}

}  // namespace tw4

using namespace tw4;

extern "C" int tw4_attend_one(const uint16_t* qkv, uint16_t* y, int M, int heads, int kv_heads, int head_dim, void* stream) {
    TW4_REQUIRE(qkv && y, TW4_EINVAL, "attend_one: null pointer");
    TW4_REQUIRE(reinterpret_cast<uintptr_t>(qkv) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0, TW4_EINVAL,
                "attend_one: qkv and y must be 16-byte aligned");
    TW4_REQUIRE(M >= 0, TW4_EINVAL, "attend_one: M >= 0 (M = %d)", M);
    TW4_REQUIRE(kv_heads >= 1 && heads >= 1 && heads % kv_heads == 0, TW4_EINVAL,
                "attend_one: heads a multiple of kv_heads (%d, %d)", heads, kv_heads);
    TW4_REQUIRE(head_dim >= 8 && head_dim % 8 == 0, TW4_EINVAL, "attend_one: head_dim %% 8 == 0 (%d)", head_dim);
    if (M == 0) return TW4_OK;
    const int hc = head_dim / 8;
    const int64_t row = static_cast<int64_t>(heads) * hc, src = row + 2LL * kv_heads * hc;
    TW4_REQUIRE(row * M < (1LL << 31) - 256 && src < (1LL << 31), TW4_EINVAL, "attend_one: too many values (M = %d)", M);
    const int chunks = static_cast<int>(row * M);
    attend_kernel<<<static_cast<unsigned>((chunks + 255) / 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
        reinterpret_cast<const u4*>(qkv) + (row + static_cast<int64_t>(kv_heads) * hc), reinterpret_cast<u4*>(y), chunks,
        static_cast<int>(row), static_cast<int>(src), hc, heads / kv_heads);
    TW4_LAUNCH_CHECK("attend_one: launch");
    return TW4_OK;
}
