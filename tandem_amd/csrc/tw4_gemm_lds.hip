// Fused-dequant GEMM for M > 16: y[M, N] = x[M, K] @ dequant(W)^T, with BOTH operand tiles staged through LDS by
// gfx950's direct-to-LDS loads (buffer_load ... lds), a ring of R slots.
//
// Workgroup tile BM x BN = (WM wavefronts x 16 MT tokens) x (WN wavefronts x 16 NT rows); wavefront (wm, wn) computes
// 16 MT tokens x 16 NT rows, over all of K or (WK = 2) two wavefronts over one of the two 32-k substeps of every stage
// each, added in LDS at the end. A stage is half a quant group (BK = 64 k): stage s covers k = 64 s .. 64 s + 63 of
// group s / 2.
//   x:       the BM x 64 fp16 tile, 128 B per token row, 8 rows per load instruction. LDS slot (row rho, position p)
//            holds 16-byte chunk p ^ ((rho >> 1) & 7) of the row. Two rows fill the 64 banks, even rows the lower 32,
//            odd rows the upper 32; the swizzle gives the 8 even (and the 8 odd) rows of a B-fragment read (16 rows, one
//            chunk) 8 different 16-byte positions, so its 16 lanes touch every bank once.
//   weights: the int4 tile as it sits in HBM: the k half of each (row tile, group) 1 KB block is 512 contiguous bytes
//            (words kb = 2 h, 2 h + 1 of [kb][r][s]), two row tiles per instruction. Every weight byte is read from
//            HBM once per workgroup; the WM wavefronts that share a row tile each read it from LDS as int4 (a quarter
//            of the fp16 bytes) and dequantize the words they need in registers.
//   params:  each wavefront's NT tiles' 16 scales and 16 zeros of the group (64 B per tile).
//   math:    v_mfma_f32_16x16x32_f16, A = dequantized weights fp16_rne((q - z) s) (16 rows x 32 k), B = x (32 k x 16
//            tokens). Substep j (0, 1) of a stage: lane (q, r) feeds A row r and B column r the k values of word
//            (kb = 2 h + (q >> 1), s = 2 (q & 1) + j), i.e. k = 64 s + 32 (q >> 1) + 16 (q & 1) + 8 j + 0..7, the same
//            permutation for both operands: a lane's two words of a stage are one 8-byte read.
//            D lane (q, r) = rows 4 q + i of token r, the layout finish_unit stores.
//   ring:    R slots. At stage i + 1's start the wavefront waits for its own loads of it (vmcnt), the workgroup meets,
//            and stage i's slot takes the loads of stage i + R, so R - 2 or more stages of loads are in flight.
//   split-K: work units (tile, split) take contiguous ranges of whole groups; the epilogue is the other GEMM's
//            finish_unit (deterministic last-arriver reduction, counters returned to zero).
//
// What bounds it. Long calls (M N K from about 2^36): the matrix cores with the dequantization beside them, at the clock the
// card's power allows: Qwen3-8B gate_up (4096 x 24576) at M = 4096 on 128 x 256 keeps them busy 67 % of the cycles, the VALU 51 %,
// at 1.6 GHz (52 % and 37 % at 1.9-2.1 GHz before the pipeline below); 17 % of a CU's cycles go to LDS bank
// conflicts. 1.24 PFLOP/s against 1.3-1.5 of hipBLASLt's fp16 product without the dequantization.
// A wavefront issues in order, about one instruction in 4 cycles, and an MFMA takes 16: the loop is software-pipelined in registers
// (the next fragments are read and the next weights dequantized between the current MFMAs, substep below), where a
// read - dequantize - multiply sequence per substep left the matrix core idle for the first two. Short calls: the wait
// for the first stages, the number of stages a CU runs in a row and how evenly the tiles divide over the CUs, hence the
// small tiles with WK = 2, two workgroups per CU and K splits. Before -> after, us, the same sizes (K x N, M), weights
// streamed from HBM: 4096 x 6144, 512: 48 -> 32; 4096 x 24576, 128 / 256 / 512: 43 / 78 / 105 -> 33 / 56 / 95;
// 12288 x 4096, 512: 66 -> 60; 4096 x 28672, 77: 48 -> 30; 5120 x 34816, 40 / 2048: 133 / 722 -> 37 / 600 (the last one
// dequantized + hipBLASLt before).
#include "tw4_lds.h"

namespace tw4 {

// Pair i (weights 2 i, 2 i + 1) of a word, dequantized: dequant_word in quarters.
__device__ __forceinline__ h2 dequant_pair(uint32_t w, int i, const GroupQ& p, uint32_t magic) {
    const h2 sixteenth = h2{static_cast<h1>(0.0625f), static_cast<h1>(0.0625f)};
    const uint32_t v = i < 2 ? w : w >> 8;
    if (i & 1) return (bitcast<h2>((v & 0x00F000F0u) | magic) * sixteenth + p.zhi) * p.s;
    return (bitcast<h2>((v & 0x000F000Fu) | magic) + p.zlo) * p.s;
}

#define TW4_STEP_FENCE __builtin_amdgcn_sched_barrier(0)

// acc += A B on v_mfma_f32_16x16x32_f16 with the accumulator held in accumulation registers for the whole loop: left
// to the compiler, the loop's accumulators move between the two register files at every iteration. FIRST: the first
// of a step, two wait states after the vector instructions that wrote A.
template <bool FIRST>
__device__ __forceinline__ void mfma_acc(f4& c, const h8& a, const h8& b) {
    if constexpr (FIRST)
        asm volatile("s_nop 1\n\tv_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    else
        asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// The accumulators after the loop's last MFMA: 32 wait states (16x16x32 needs 18 before a vector read of its result),
// after which they are ordinary values again.
template <int NT, int MT>
__device__ __forceinline__ void mfma_settle(f4 (&acc)[NT][MT]) {
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int b = 0; b < MT; ++b) asm volatile("" : "+a"(acc[t][b]));
}

template <int MT_, int NT_, int WM_, int WN_, int WK_, int R_>
struct LdsGemmCfg {
    static constexpr int MT = MT_, NT = NT_, WM = WM_, WN = WN_, WK = WK_, R = R_;
    static constexpr int BM = 16 * MT * WM;
    static constexpr int BN = 16 * NT * WN;
    static constexpr int WAVES = WM * WN * WK;
    static constexpr int THREADS = 64 * WAVES;
    static constexpr int X_U4 = BM * 8;               // x tile: BM rows x 8 chunks
    static constexpr int W_U4 = BN / 16 * 32;         // weights: BN / 16 half-blocks of 512 B
    static constexpr int P_INSTR = NT <= 4 ? 1 : 2;   // params loads per wavefront and group (256 B each)
    static constexpr int P_U4 = WAVES * 16 * P_INSTR; // per wavefront its tiles' 16 scales each, then their zeros
    static constexpr int SLOT_U4 = X_U4 + W_U4 + P_U4;
    static constexpr int X_LOADS = BM / 8;            // 1 KB loads of a stage: 8 token rows each
    static constexpr int W_LOADS = BN / 32;           // two half-blocks each
    static constexpr int X_INSTR = (X_LOADS + WAVES - 1) / WAVES;  // per wavefront (the last ones may repeat a load)
    static constexpr int W_INSTR = (W_LOADS + WAVES - 1) / WAVES;
    static constexpr int XW = X_INSTR + W_INSTR;
    static constexpr int LDS_BYTES = R * SLOT_U4 * 16;
    // wavefronts per SIMD the registers are kept for: two where the accumulators leave room for it and two
    // workgroups fit a CU's 160 KB of LDS (or the workgroup itself has eight wavefronts)
    static constexpr int MIN_WAVES_PER_SIMD = MT * NT <= 32 && (WAVES >= 8 || LDS_BYTES <= 80 * 1024 - 256) ? 2 : 1;
    // partial sums the last arriver of a K split loads per round (finish_unit): all of a wavefront's, unless they and the sums
    // they are added to fill every register, which left the compiler two loads in flight (128 x 256, 4096 x 4096 in 16
    // splits: 90 us; half of them per round 42)
    static constexpr int FRAGS = MT * NT == 64 || (MT * NT == 32 && MIN_WAVES_PER_SIMD == 2) ? MT * NT / 2 : MT * NT;
    static_assert(WK == 1 || (WK == 2 && WM * WN * MT * NT * 64 <= R * SLOT_U4), "the K halves' sums fit the ring");
    static_assert(R >= 3, "ring of at least 3 slots");
    static_assert(BM % 8 == 0 && BN % 32 == 0, "whole 1 KB loads");
    static_assert(NT >= 2 && NT <= 8, "params: one dword load covers 4 tiles' scales and zeros, or 8 tiles' of one");
    static_assert((R - 1) * (XW + P_INSTR) < 64, "s_waitcnt vmcnt immediate");
    static_assert(LDS_BYTES <= 160 * 1024 - 64, "one workgroup's LDS");
};

template <class C>
struct LdsGemmArgs {
    u4 x, w;                    // buffer resources; a stage's k offset is the loads' scalar offset
    uint32_t xoff[C::X_INSTR];  // this lane's byte offsets, fixed for the kernel (see lds_gemm_offsets)
    uint32_t woff[C::W_INSTR];
    const char* p[C::P_INSTR];  // this lane's scale / zero pair of group 0, and the bytes from a group to the next
    uint32_t pstep;
    uint32_t xw, ww, pw;        // this wavefront's first LDS byte of each part of a slot
};

// Per-lane addresses of the direct-to-LDS loads (everything but the stage's k position):
//   x load j (rows 8 j .. 8 j + 7 of the tile): lane l takes row rho = 8 j + l / 8 (rows past M read the last row;
//     never stored), 16-byte chunk (l & 7) ^ ((rho >> 1) & 7);
//   weight load j (row tiles 2 j, 2 j + 1 of the workgroup): lane l the 16 bytes l & 31 of the k half of tile
//     2 j + l / 32's block (tiles past the matrix read its last tile);
//   wavefront v issues loads v X_INSTR + i (W_INSTR alike); where those are more than the tile has (a count that does
//     not divide by the wavefronts), the last wavefronts start earlier and repeat loads of the one before them (the
//     same bytes to the same place);
//   params: lane l the values of rows 2 (l & 7), + 1 of one tile: NT <= 4, tile (l / 8) % 4, scales in lanes
//     0 .. 31 and zeros in 32 .. 63; else tile l / 8 of 8, scales and zeros by a load each. A last tile of 8 rows
//     (N % 16 == 8) has 16 bytes per group, whose lanes past row 7 read rows 6 and 7 (never stored).
template <class C>
__device__ __forceinline__ void lds_gemm_offsets(LdsGemmArgs<C>& a, const h1* scales, const h1* zeros,
                                                 int M, int N, int K, int G, int m0, int tile0, int tile_last, int wave,
                                                 int wn, int lane) {
#pragma unroll
    for (int i = 0; i < C::X_INSTR; ++i) {
        const int j = min(wave * C::X_INSTR, C::X_LOADS - C::X_INSTR) + i;
        const int rho = 8 * j + (lane >> 3), c = (lane & 7) ^ ((rho >> 1) & 7);
        const int row = min(m0 + rho, M - 1);
        a.xoff[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(K) * 2u + 16u * c;
    }
#pragma unroll
    for (int i = 0; i < C::W_INSTR; ++i) {
        const int j = min(wave * C::W_INSTR, C::W_LOADS - C::W_INSTR) + i;
        const int t = min(tile0 + 2 * j + (lane >> 5), tile_last);
        a.woff[i] = static_cast<uint32_t>(t) * static_cast<uint32_t>(G) * 1024u + 16u * (lane & 31);
    }
    const int t = min(tile0 + wn * C::NT + min((lane >> 3) & (C::P_INSTR == 1 ? 3 : 7), C::NT - 1), tile_last);
    const int rows = tile_rows(t, N);
    const int64_t off = static_cast<int64_t>(t) * 16 * G + min(2 * (lane & 7), rows - 2);
    a.pstep = 2u * rows;
    a.xw = 1024 * min(wave * C::X_INSTR, C::X_LOADS - C::X_INSTR);
    a.ww = 16 * C::X_U4 + 1024 * min(wave * C::W_INSTR, C::W_LOADS - C::W_INSTR);
    a.pw = 16 * (C::X_U4 + C::W_U4) + 256 * wave * C::P_INSTR;
    if constexpr (C::P_INSTR == 1) {
        a.p[0] = reinterpret_cast<const char*>((lane < 32 ? scales : zeros) + off);
    } else {
        a.p[0] = reinterpret_cast<const char*>(scales + off);
        a.p[1] = reinterpret_cast<const char*>(zeros + off);
    }
}

// Direct-to-LDS load I (of X_INSTR + W_INSTR, then P_INSTR at even stages) of stage `st` into the slot at LDS byte
// address `slot`. Every wavefront issues the same number per stage, so each can wait for a stage with one vmcnt.
// Stage st = (group g = st / 2, k half st & 1) moves the scalar offset only: x by 64 st halves, the weights by block g
// and half (512 st bytes), the scales and zeros by group g (pg; past the last group its own again).
template <int I, class C>
__device__ __forceinline__ void issue_load(uint32_t slot, const LdsGemmArgs<C>& a, const u4& xr, const u4& wr,
                                           int st, int pg) {
    if constexpr (I < C::X_INSTR)
        lds_dma16<1024 * I>(xr, a.xoff[I], 128u * st, slot + a.xw);
    else if constexpr (I < C::XW)
        lds_dma16<1024 * (I - C::X_INSTR)>(wr, a.woff[I - C::X_INSTR], 512u * st, slot + a.ww);
    else
        lds_dma4<256 * (I - C::XW)>(a.p[I - C::XW] + static_cast<uint64_t>(static_cast<uint32_t>(pg)) * a.pstep, slot + a.pw);
}

// The loads of LOADS per stage that step k of S issues (evenly spread), from load I on.
template <int I, int LOADS, int S, class C>
__device__ __forceinline__ void issue_loads_at(int k, uint32_t slot, const LdsGemmArgs<C>& a, const u4& xr,
                                               const u4& wr, int st, int pg) {
    if constexpr (I < LOADS) {
        if ((2 * I + 1) * S / (2 * LOADS) == k) issue_load<I>(slot, a, xr, wr, st, pg);
        issue_loads_at<I + 1, LOADS, S>(k, slot, a, xr, wr, st, pg);
    }
}

// Registers of the software pipeline: the B fragments of the current and the next 32-k substep, the current and next
// half group's weight words (WK = 1: one 8-byte pair per tile, both substeps; WK = 2: the wavefront's one), the
// group's dequantization constants.
template <class C>
struct LdsGemmRegs {
    h8 xb[2][C::MT];
    uint32_t wv[2][C::NT][3 - C::WK];
    GroupQ pq[C::NT];
    uint32_t ps[C::NT], pz[C::NT];
    h8 a;  // the dequantized A fragment of the next (substep, tile)
};

template <class C>
__device__ __forceinline__ void read_words(uint32_t (&w)[3 - C::WK], const char* p) {
    if constexpr (C::WK == 1) {
        const u2 v = *reinterpret_cast<const u2*>(p);
        w[0] = v.x, w[1] = v.y;
    } else {
        w[0] = *reinterpret_cast<const uint32_t*>(p);
    }
}

// One 32-k substep of a half group of parity PAR (0: k half 0), B fragments in set CUR and words J of set PAR: NT
// steps of MT MFMAs, beside which the next substep's B fragments are read from `nxt` (front-loaded over the first
// steps) and the next step's A fragment is dequantized. LAST, the wavefront's last substep of its half group: the
// words (and at PAR = 1 the scales and zeros) of the next half group are read too and LOADS loads of stage `st`
// issued into slot address `dma`. All of it sits between the MFMAs, at most a few instructions behind each, because
// a wavefront issues in order: side work in a block of its own leaves the matrix core idle after 16 cycles.
template <class C, int PAR, int CUR, int J, bool LAST, int LOADS>
__device__ __forceinline__ void substep(LdsGemmRegs<C>& v, f4 (&acc)[C::NT][C::MT], const u4* nxt, int xl, int wl, int pl,
                                        uint32_t dma, const LdsGemmArgs<C>& a, const u4& xr, const u4& wr, int st, int pg,
                                        uint32_t magic) {
    constexpr int MT = C::MT, NT = C::NT;
    constexpr int S = NT * MT;  // steps: one MFMA and the side work that issues while it runs
    const char* nb = reinterpret_cast<const char*>(nxt);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const h8 at = v.a;
        // the next step's tile: its word and constants
        const bool same = t + 1 < NT;
        const int tn = same ? t + 1 : 0;
        h2 d[4];
#pragma unroll
        for (int b = 0; b < MT; ++b) {
            const int k = t * MT + b;
            if (b == 0)
                mfma_acc<true>(acc[t][b], at, v.xb[CUR][b]);
            else
                mfma_acc<false>(acc[t][b], at, v.xb[CUR][b]);
            if (LAST && k < NT) read_words<C>(v.wv[1 - PAR][k], nb + wl + 512 * k);  // the next half group's words,
            if (LAST && PAR == 1 && k >= 1 && k <= NT) {                             // then its scales and zeros
                const uint16_t* ps = reinterpret_cast<const uint16_t*>(nb + pl);
                v.ps[k - 1] = ps[16 * (k - 1)], v.pz[k - 1] = ps[(NT <= 4 ? 64 : 128) + 16 * (k - 1)];
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)  // B fragment i in the first half of the steps
                if (i * S / (2 * MT) == k) v.xb[1 - CUR][i] = bitcast<h8>(*(reinterpret_cast<const u4*>(nb + xl) + 128 * i));
            // tile t's constants of the next group, once its words of this one are done with
            if (LAST && PAR == 1 && b == (MT > 4 ? MT / 2 : MT - 1) && same) v.pq[t] = group_q(as_h1(v.ps[t]), as_h1(v.pz[t]));
            if (LAST && PAR == 1 && b == 0 && !same) v.pq[NT - 1] = group_q(as_h1(v.ps[NT - 1]), as_h1(v.pz[NT - 1]));
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if ((2 * i + 1) * MT / 8 == b) {
                    const uint32_t word = same ? v.wv[PAR][tn][J] : LAST ? v.wv[1 - PAR][0][0] : v.wv[PAR][0][C::WK == 1 ? 1 : 0];
                    d[i] = dequant_pair(word, i, v.pq[tn], magic);
                }
            issue_loads_at<0, LOADS, S>(k, dma, a, xr, wr, st, pg);
            TW4_STEP_FENCE;
        }
        v.a = h8{d[0].x, d[0].y, d[1].x, d[1].y, d[2].x, d[2].y, d[3].x, d[3].y};
    }
}

// Half group i (parity PAR) from ring slot `slot`, which then moves to the next one. WK = 1: substep 0 reads the
// second substep's fragments from the slot. Then the wavefront waits for its own loads of stage i + 1 (the R - 2
// stages after it stay in flight) and for its LDS reads of stage i, and the workgroup meets: stage i + 1 is in LDS
// and nobody reads stage i any more, so its slot takes the loads of stage i + R beside the last substep's math,
// which reads stage i + 1. A stage past the end is issued with empty resources. WK = 2: each wavefront has one of
// the two substeps, read a whole half group ahead.
template <class C, int PAR>
__device__ __forceinline__ void half_step(LdsGemmRegs<C>& v, f4 (&acc)[C::NT][C::MT], const u4* ring, uint32_t ring_addr,
                                          int& slot, int i, int nst, int st0, int xl0, int xl1, int wl, int pl,
                                          const LdsGemmArgs<C>& a, int glast, uint32_t magic) {
    constexpr int R = C::R;
    const u4* cur = ring + slot * C::SLOT_U4;
    const uint32_t cur_addr = ring_addr + 16 * slot * C::SLOT_U4;
    slot = slot + 1 == R ? 0 : slot + 1;
    const u4* nxt = ring + slot * C::SLOT_U4;
    if constexpr (C::WK == 1) {
        const u4 none{};
        substep<C, PAR, 0, 0, false, 0>(v, acc, cur, xl1, wl, pl, 0, a, none, none, 0, 0, magic);
    }
    // loads of stages i + 2 .. i + R - 1: R - 2 stages, the first of this one's parity, params with the even ones
    constexpr int AHEAD = (R - 2) * C::XW + (R - 2 + (PAR == 0 ? 1 : 0)) / 2 * C::P_INSTR;
    constexpr int LOADS = C::XW + ((PAR + R) % 2 == 0 ? C::P_INSTR : 0);
    wait_stage<AHEAD>();
    ring_barrier();
    const int st = st0 + i + R;
    u4 xr = a.x, wr = a.w;
    xr.z = wr.z = __builtin_amdgcn_readfirstlane(i + R < nst ? 0xFFFFFFFFu : 0u);
    substep<C, PAR, C::WK == 1 ? 1 : PAR, C::WK == 1 ? 1 : 0, true, LOADS>(v, acc, nxt, xl0, wl, pl, cur_addr, a, xr, wr, st,
                                                                        min(st >> 1, glast), magic);
}

template <class C>
__global__ void __launch_bounds__(C::THREADS) __attribute__((amdgpu_waves_per_eu(C::MIN_WAVES_PER_SIMD)))
gemm_lds_kernel(const h1* __restrict__ x, const u4* __restrict__ w, const h1* __restrict__ scales,
                const h1* __restrict__ zeros, h1* __restrict__ y, float* __restrict__ ws, int* __restrict__ locks,
                int M, int N, int K, int mb, int nb, int splits, int act) {
    __shared__ u4 ring[C::R * C::SLOT_U4];
    __shared__ int last_flag;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int MT = C::MT, NT = C::NT, R = C::R;
    const int wn = wave % C::WN, wm = wave / C::WN % C::WM, wk = wave / (C::WN * C::WM);
    const int G = K >> 7, tiles_n = (N + 15) >> 4;

    // work unit -> (tile, split); tiles in bands of 8 token blocks, each XCD a contiguous range
    const int unit = xcd_remap(blockIdx.x, gridDim.x);
    const int tile = unit / splits, split = unit - tile * splits;
    const int band = tile / (8 * nb), band_rows = min(mb - band * 8, 8), rin = tile - band * 8 * nb;
    const int mblk = band * 8 + rin % band_rows, nblk = rin / band_rows;
    // whole quant groups per split; a split past the groups has none and contributes zeros
    const int g0 = static_cast<int>(static_cast<int64_t>(split) * G / splits);
    const int nst = 2 * (static_cast<int>(static_cast<int64_t>(split + 1) * G / splits) - g0);
    const int st0 = 2 * g0;

    const int m0 = mblk * C::BM, tile0 = nblk * (C::BN / 16);
    LdsGemmArgs<C> a;
    a.x = lds_rsrc(x);
    a.w = lds_rsrc(w);
    lds_gemm_offsets<C>(a, scales, zeros, M, N, K, G, m0, tile0, tiles_n - 1, wave, wn, lane);

    const uint32_t magic = magic_reg();
    f4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[t][b] = f4{0.0f, 0.0f, 0.0f, 0.0f};

    if (nst > 0) {
        // the ring's LDS byte address, taken once from the array itself (the direct-to-LDS loads take it in M0)
        const uint32_t ring_addr = static_cast<uint32_t>(reinterpret_cast<size_t>((lds_void*)ring));
        const int r = lane & 15, q = lane >> 4;
        // byte offsets inside a slot: this lane's 16-byte chunk of token row r at the wavefront's first substep (the
        // other one: ^ 16), its words of the wavefront's first tile, the row's scale of that tile
        const int c0 = 4 * (q >> 1) + 2 * (q & 1);
        const int xl0 = (wm * 16 * MT + r) * 128 + 16 * ((c0 + wk) ^ ((r >> 1) & 7)), xl1 = xl0 ^ 16;
        const int wl = 16 * C::X_U4 + wn * NT * 512 + ((q >> 1) * 16 + r) * 16 + 8 * (q & 1) + 4 * wk;
        const int pl = 16 * (C::X_U4 + C::W_U4) + 256 * wave * C::P_INSTR + 2 * r;
#pragma unroll
        for (int p = 0; p < R; ++p) {
            u4 xr = a.x, wr = a.w;
            xr.z = wr.z = __builtin_amdgcn_readfirstlane(p < nst ? 0xFFFFFFFFu : 0u);
            const uint32_t sa = ring_addr + 16 * p * C::SLOT_U4;
            if (p & 1)
                issue_loads_at<0, C::XW, 1>(0, sa, a, xr, wr, st0 + p, 0);
            else
                issue_loads_at<0, C::XW + C::P_INSTR, 1>(0, sa, a, xr, wr, st0 + p, min(g0 + (p >> 1), G - 1));
        }
        wait_stage<(R - 1) * C::XW + (R - 1) / 2 * C::P_INSTR>();  // stages 1 .. R - 1 may be in flight
        ring_barrier();
        LdsGemmRegs<C> v;
        {
            const char* s0 = reinterpret_cast<const char*>(ring);
            const uint16_t* ps = reinterpret_cast<const uint16_t*>(s0 + pl);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                read_words<C>(v.wv[0][t], s0 + wl + 512 * t);
                v.pq[t] = group_q(as_h1(ps[16 * t]), as_h1(ps[(NT <= 4 ? 64 : 128) + 16 * t]));
            }
#pragma unroll
            for (int b = 0; b < MT; ++b) v.xb[0][b] = bitcast<h8>(*(reinterpret_cast<const u4*>(s0 + xl0) + 128 * b));
            v.a = dequant_word(v.wv[0][0][0], v.pq[0], magic);
        }
        int slot = 0, i = 0;
        for (; i < nst; i += 2) {
            half_step<C, 0>(v, acc, ring, ring_addr, slot, i, nst, st0, xl0, xl1, wl, pl, a, G - 1, magic);
            half_step<C, 1>(v, acc, ring, ring_addr, slot, i + 1, nst, st0, xl0, xl1, wl, pl, a, G - 1, magic);
        }
        mfma_settle<NT, MT>(acc);
        wait_stage<0>();  // the empty loads past the end still write their slots
    }

    if constexpr (C::WK == 2) {  // the K halves' sums: the ring is free (every load has landed, every read is done)
        __syncthreads();
        f4* red = reinterpret_cast<f4*>(ring) + (wm * C::WN + wn) * NT * MT * 64 + lane;
        if (wk == 1) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int b = 0; b < MT; ++b) red[(t * MT + b) * 64] = acc[t][b];
        }
        __syncthreads();
        if (wk == 0) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int b = 0; b < MT; ++b) acc[t][b] += red[(t * MT + b) * 64];
        }
    }
    finish_unit<MT, NT, C::WM * C::WN, 64, C::FRAGS>(acc, wk == 0, wm * C::WN + wn, lane, tid, splits, tile, unit, ws, locks, last_flag, y, M, N,
                                 m0 + wm * 16 * MT, tile0 + wn * NT, tiles_n, act);
}

// Compiled configurations (MT, NT, WM, WN, WK, ring slots): tw4_gemm's stages-3 ones, and the others of tw4_gemm_tiled. Of the
// first list the rule takes (8, 4, 1, 4, 1, 3) only; the rest are there for ladders that callers name them in.
#define TW4_LDS_GEMM_CONFIGS(X) X(8, 4, 2, 4, 1, 3) X(16, 4, 1, 4, 1, 3) X(4, 4, 2, 4, 1, 3) X(8, 4, 2, 2, 1, 3) \
    X(8, 8, 1, 4, 1, 4) X(8, 4, 1, 4, 1, 3)
#define TW4_TILED_GEMM_CONFIGS(X) X(8, 6, 2, 2, 1, 3) X(8, 6, 1, 2, 2, 4) X(8, 4, 1, 2, 2, 4) X(8, 3, 1, 2, 2, 4) \
    X(8, 2, 1, 2, 2, 4) X(5, 4, 1, 2, 2, 4) X(5, 3, 1, 2, 2, 4) X(5, 2, 1, 2, 2, 4) X(4, 3, 1, 2, 2, 4) \
    X(4, 2, 1, 2, 2, 4) X(3, 3, 1, 2, 2, 4) X(3, 2, 1, 2, 2, 4) X(2, 3, 1, 2, 2, 4) X(2, 2, 1, 2, 2, 4)

template <class C>
int lds_gemm_launch(const h1* x, const u4* w, const h1* s, const h1* z, h1* y, float* ws, int* locks,
                    int64_t ws_floats, int64_t n_locks, int M, int N, int K, int splits, int cus, int act,
                    hipStream_t stream) {
    TW4_REQUIRE(reinterpret_cast<uintptr_t>(s) % 4 == 0 && reinterpret_cast<uintptr_t>(z) % 4 == 0, TW4_EINVAL,
                "gemm (both tiles in LDS): scales and zeros must be 4-byte aligned");
    const int G = K >> 7, stages = 2 * G;
    const int mb = (M + C::BM - 1) / C::BM, nb = (N + C::BN - 1) / C::BN;
    const int64_t tiles64 = static_cast<int64_t>(mb) * nb;
    TW4_REQUIRE(tiles64 < (1LL << 30), TW4_EINVAL, "gemm: too many tiles (%lld)", static_cast<long long>(tiles64));
    const int tiles = static_cast<int>(tiles64);
    int sp = splits;
    if (sp == 0) {  // enough units to fill the GPU once, within the default workspace (never the caller's)
        sp = 1;
        while (static_cast<int64_t>(tiles) * sp < cus && 2 * (sp + 1) <= stages &&
               static_cast<int64_t>(tiles) * (sp + 1) * C::BM * C::BN <= TW4_AUTO_SPLIT_FLOATS &&
               tiles <= TW4_AUTO_SPLIT_COUNTERS)
            ++sp;
    }
    TW4_REQUIRE(sp >= 1 && sp <= stages, TW4_EINVAL, "gemm: splits %d for %d stages", sp, stages);
    if (sp > 1) {
        TW4_REQUIRE(ws && locks, TW4_EINVAL, "gemm: split-K needs a workspace and counters");
        TW4_REQUIRE(static_cast<int64_t>(tiles) * sp * C::BM * C::BN <= ws_floats && tiles <= n_locks, TW4_ESPACE,
                    "gemm: split-K workspace too small for %d tiles x %d splits", tiles, sp);
    }
    const int64_t blocks = static_cast<int64_t>(tiles) * sp;
    TW4_REQUIRE(blocks < (1LL << 31), TW4_EINVAL, "gemm: grid too large");
    gemm_lds_kernel<C><<<static_cast<unsigned>(blocks), C::THREADS, 0, stream>>>(
        x, w, s, z, y, ws, locks, M, N, K, mb, nb, sp, act);
    TW4_LAUNCH_CHECK("gemm (both tiles in LDS): launch");
    return TW4_OK;
}

}  // namespace tw4

using namespace tw4;

// Called by tw4_gemm for stages == 3 (warps_k is then WM, the wavefronts along M).
int tw4_gemm_lds_dispatch(const uint16_t* x, const int32_t* packed, const uint16_t* scales, const uint16_t* zeros,
                          uint16_t* y, float* ws, int32_t* locks, int64_t ws_floats, int64_t n_locks, int M, int N,
                          int K, int mt, int nt, int warps_n, int warps_m, int splits, int cus, int act,
                          void* stream) {
    TW4_REQUIRE(N % 16 == 0, TW4_EINVAL, "gemm (stages 3): N %% 16 == 0 (N = %d)", N);
    TW4_REQUIRE(reinterpret_cast<uintptr_t>(scales) % 16 == 0 && reinterpret_cast<uintptr_t>(zeros) % 16 == 0, TW4_EINVAL,
                "gemm (stages 3): scales and zeros must be 16-byte aligned");
    auto xp = reinterpret_cast<const h1*>(x);
    auto wp = reinterpret_cast<const u4*>(packed);
    auto sp = reinterpret_cast<const h1*>(scales);
    auto zp = reinterpret_cast<const h1*>(zeros);
    auto yp = reinterpret_cast<h1*>(y);
    auto st = static_cast<hipStream_t>(stream);
#define TW4_LDS_CASE(MT, NT, WM, WN, WK, R)                                                                            \
    if (mt == MT && nt == NT && warps_m == WM && warps_n == WN)                                                        \
        return lds_gemm_launch<LdsGemmCfg<MT, NT, WM, WN, WK, R>>(xp, wp, sp, zp, yp, ws, locks, ws_floats, n_locks, M,\
                                                                  N, K, splits, cus, act, st);
    TW4_LDS_GEMM_CONFIGS(TW4_LDS_CASE)
#undef TW4_LDS_CASE
    tw4host::set_error("gemm: unsupported stages-3 config mt / nt / warps_n / warps_m %d / %d / %d / %d", mt, nt,
                       warps_n, warps_m);
    return TW4_ECONFIG;
}

// Called by tw4_gemm_tiled.
int tw4_gemm_tiled_dispatch(const uint16_t* x, const int32_t* packed, const uint16_t* scales, const uint16_t* zeros,
                            uint16_t* y, float* ws, int32_t* locks, int64_t ws_floats, int64_t n_locks, int M, int N,
                            int K, int mt, int nt, int warps_n, int warps_m, int warps_k, int ring, int splits, int cus,
                            int act, void* stream) {
    auto xp = reinterpret_cast<const h1*>(x);
    auto wp = reinterpret_cast<const u4*>(packed);
    auto sp = reinterpret_cast<const h1*>(scales);
    auto zp = reinterpret_cast<const h1*>(zeros);
    auto yp = reinterpret_cast<h1*>(y);
    auto st = static_cast<hipStream_t>(stream);
#define TW4_LDS_CASE(MT, NT, WM, WN, WK, R)                                                                            \
    if (mt == MT && nt == NT && warps_m == WM && warps_n == WN && warps_k == WK && ring == R)                          \
        return lds_gemm_launch<LdsGemmCfg<MT, NT, WM, WN, WK, R>>(xp, wp, sp, zp, yp, ws, locks, ws_floats, n_locks, M,\
                                                                  N, K, splits, cus, act, st);
    TW4_LDS_GEMM_CONFIGS(TW4_LDS_CASE)
    TW4_TILED_GEMM_CONFIGS(TW4_LDS_CASE)
#undef TW4_LDS_CASE
    tw4host::set_error("gemm_tiled: unsupported mt / nt / warps_n / warps_m / warps_k / ring %d / %d / %d / %d / %d / %d", mt,
                       nt, warps_n, warps_m, warps_k, ring);
    return TW4_ECONFIG;
}

int tw4_gemm_lds_configs(int* out, int max_configs, int start) {
    int n = 0;
#define TW4_LDS_LIST(MT, NT, WM, WN, WK, R)              \
    if (out && start + n < max_configs) {            \
        out[5 * (start + n)] = MT;                   \
        out[5 * (start + n) + 1] = NT;               \
        out[5 * (start + n) + 2] = WN;               \
        out[5 * (start + n) + 3] = WM;               \
        out[5 * (start + n) + 4] = 3;                \
    }                                                \
    ++n;
    TW4_LDS_GEMM_CONFIGS(TW4_LDS_LIST)
#undef TW4_LDS_LIST
    return n;
}

extern "C" int tw4_gemm_tiled_configs(int* out, int max_configs) {
    int n = 0;
#define TW4_LDS_LIST(MT, NT, WM, WN, WK, R)    \
    if (out && n < max_configs) {          \
        out[6 * n] = MT;                   \
        out[6 * n + 1] = NT;               \
        out[6 * n + 2] = WN;               \
        out[6 * n + 3] = WM;               \
        out[6 * n + 4] = WK;               \
        out[6 * n + 5] = R;                \
    }                                      \
    ++n;
    TW4_LDS_GEMM_CONFIGS(TW4_LDS_LIST)
    TW4_TILED_GEMM_CONFIGS(TW4_LDS_LIST)
#undef TW4_LDS_LIST
    return n;
}
