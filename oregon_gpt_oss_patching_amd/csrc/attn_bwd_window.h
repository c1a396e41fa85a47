// Single-pass backward for sliding-window layers (window <= 128): dQ, dK, dV and the dSinks
// terms from ONE read of Q, dO, O, K, V, five GEMMs per (query block, key block) pair.  Stands in for
// the reference's `_attn_bwd_precompute_D` + `_attn_bwd` (attention_kernel.py:102-217) on such
// layers; results are bit-reproducible (fixed summation orders; no word is added to by more than one lane).
//
// With a window of at most 128 a block u of 32 query rows sees the five 32-key blocks u-4 .. u, and a key block is seen by
// the query blocks u .. u+4.  A workgroup owns a chunk of consecutive query blocks [u0, u1) of one KV head (all r query heads
// of the group) and walks (query block, pair of heads), heads inner.  Twelve wavefronts, three per SIMD, in two groups: group 0 takes
// the even heads of the walk, group 1 the odd ones.  Each group has
//   * five "owners".  Owner p holds, as MFMA B operands in registers, the K and V rows of the one live key block kb with
//     kb % 5 == p and its group's dK / dV accumulators of that block.  Per step an owner does one 32 x 32 block
//     (window_block: S = Q K^T, dP = dO V^T, P, dS, dV^T += dO^T P, dK^T += Q^T dS) and leaves the bf16 dS block in LDS,
//     key-major.  When the walk moves on to query block u, key block u-5 is complete: its two owners have exchanged
//     one tensor each through LDS, group 0's adds and writes dK, group 1's dV, and both take over key block u.
//   * one "helper".  One step AHEAD of the owners it forms the row statistics -lse / scale and -rowsum(dO*O) of the
//     group's 32 rows (dO from the staged tile, O rows it reads itself) and leaves them in LDS; one step BEHIND them it turns
//     the dS blocks into dQ^T = K^T dS^T over all 160 live keys (K^T fragments resident in its registers) and writes the finished
//     dQ rows.  It also sums the dSinks terms exp(sink - lse) * (-delta) of its rows.
// All keys a query block can see are in the workgroup at the same time, so dQ is complete when the helper stores it.  A key
// block collects from five query blocks, so the last four key blocks of a chunk (and the four before it, which its first rows need for
// dQ) are completed by two neighbouring workgroups.  Two ways of closing that seam:
//   * boundary_partial set (gptoss_attn_bwd): each of the two workgroups leaves its fp32 share of
//     dK / dV of those blocks in the scratch, and attn_bwd_window_finish_kernel adds the two shares
//     in a fixed order, scales and rounds: 64 KB of partial sums per seam and side, and a
//     walk of exactly the chunk's own query blocks;
//   * boundary_partial NULL (gptoss_attn_bwd_static, which has no room for the partial sums): the
//     walk goes four query blocks past the chunk, for the sake of its last key blocks only, and
//     drops the dK / dV of the key blocks before the chunk (the neighbour produces them the
//     same way): recomputation instead of an exchange.
// Both are bit-reproducible.
//
// One barrier per step hands over the staged Q / dO tiles (asynchronous global->LDS copies, four stages), the row
// statistics of the next step and the dS blocks of the previous one (double buffered).  K / V rows of the next key block travel
// through an LDS transit buffer one query block ahead of their use.
//
// Why this split: the step is a chain of latencies (fragments out of LDS, 16 MFMAs, 16 exponentials, 16 MFMAs, the dS blocks over to the helpers), so the
// number of wavefronts that hide each other's decides.  Three per SIMD leave 168 registers: an owner's 64 accumulators, 32 of K / V, 32 of S / dP, and six
// fragments under way.  Whole backward, us, six owners with 64-row tiles and two helpers (two wavefronts per SIMD, one head per step) / so: 16384 tokens of 64
// heads on 8 KV heads 204 / 176, 2 x 3001 77 / 68, 4096 56.5 / 51.5.  What bounds it: all the copies, loads and stores without the owners' arithmetic take 134 us at 16384
// (660 MB, 4.9 TB/s), everything but the tiles' copies 128 us (1.8 us a step; matrix pipe 30 % busy, LDS 33 %), and a workgroup per compute unit lays
// the one over the other only in part.  The merge of the two groups' sums and the results' way out, once in
// five blocks per owner, were 14 us of it with one owner per block doing both tensors and are 11 with one tensor each (whole call, 16384 tokens 256 / 253, 2 x 3001 105.7 / 104.8).  A block's start and end
// cost about one step: 4096 tokens are four blocks of four steps per workgroup, 29 of 48 us.
#pragma once
#include <type_traits>

#include "attn_bwd.h"
#include "attn_common.h"

namespace gptoss {

struct WinCfg {
    static constexpr int NSLOT = 5, NOWN = 2 * NSLOT, NWAVES = NOWN + 2, NS = 4;
    static constexpr int kRows = 32;                                       // query rows, keys of a block
    static constexpr int kMaxWindow = 128;
    static constexpr int kBack = kMaxWindow / kRows;                       // key blocks in front of a query block's own that it sees
    static constexpr int kMaxGroup = 16;                                   // query heads per KV head
    // The weights are exp(scale * (S - lse / scale)), whose quotient has to stay finite.  Smaller scales take this one's weights: a sum of
    // up to 128 exponentials and a sink has an lse below 2^11 (or no room beside its sink), and S is nothing beside it up to 2^100.
    static constexpr float kMinScale = 0x1p-116f;
    static constexpr int kBlockBytes = kRows * kRowBytes;                  // 4 KB: a block's rows of one tensor
    static constexpr int kMergeBytes = 2 * 2 * 16 * 64 * 4;                // an owner's dK and dV accumulators
    static constexpr int kStageOff = 0;                                    // [NS][group][Q, dO][4 KB]; behind the walk four merge buffers
    static constexpr int kMergeOff = kStageOff + NS * 2 * 2 * kBlockBytes; // of the block that is complete: group 1's dK, group 0's dV
    static constexpr int kStatOff = kMergeOff + kMergeBytes;               // [2][group][-lse / scale, -delta][32] floats
    static constexpr int kDsOff = kStatOff + 2 * 2 * 2 * kRows * 4;        // [2][slot][32 keys][group][32 rows] bf16
    static constexpr int kDsBytes = NSLOT * kBlockBytes;
    static constexpr int kTransitOff = kDsOff + 2 * kDsBytes;              // [2][K, V][4 KB] of the next key block
    static constexpr int kOutOff = kTransitOff + 2 * 2 * kBlockBytes;      // [group][32 x kLS] bf16 output stages of the helpers
    static constexpr int kSinkOff = kOutOff + 2 * kRows * kLS * 2;         // [group][kMaxGroup / 2][64 lanes] floats
    static constexpr int kLogitOff = kSinkOff + kMaxGroup * 64 * 4;        // [group][kMaxGroup / 2] floats
    static constexpr int kLdsBytes = kLogitOff + kMaxGroup * 4;
    static_assert(NSLOT * kMergeBytes == kStatOff - kStageOff, "behind the walk every slot has a merge buffer");
    static_assert(kDsOff % 128 == 0 && kTransitOff % 128 == 0, "swizzled tiles start on 128-byte boundaries");
    static_assert(kRows * kLS * 2 <= kMergeBytes / 2, "an owner's output stage is its merge buffer");
    static_assert(kLdsBytes <= 160 * 1024, "one workgroup per CU");
};

// (query block, pair of heads) of a position of the walk
struct WinPos {
    int u, hp;
    __device__ __forceinline__ void step(int pairs) { if (++hp == pairs) { hp = 0; ++u; } }
};

// dS exchange through LDS.  A slot's blocks are key-major: a key row is 128 bytes (32 query rows of group 0, then of group 1, in bf16), chunk-swizzled by
// swz(key).  A lane of an owner (key, half = lane / 32) holds, per 16-row step u, the B fragment dsf: elements 0..3 are rows 16u + 4*half + 0..3, elements 4..7
// rows 16u + 8 + 4*half + 0..3, i.e. two 8-byte pieces in the logical chunks 2*u and 2*u + 1 (+ 4 for group 1) of its key row, at byte 8*half of the
// chunk.  With the row's swizzle folded into the base address the chunk selection is one XOR with an immediate.
__device__ __forceinline__ uint32_t ds_store_addr(uint32_t blocks, int key, int half) { return blocks + key * kRowBytes + (swz(key) << 4) + 8 * half; }
__device__ __forceinline__ void ds_store(uint32_t base, int u, const bf16x8 dsf) {
    typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
    bf16x4 p0, p1;
#pragma unroll
    for (int e = 0; e < 4; ++e) { p0[e] = dsf[e]; p1[e] = dsf[4 + e]; }
    *reinterpret_cast<lds_bf16x4 *>((uintptr_t)(base ^ ((2 * u) << 4))) = p0;
    *reinterpret_cast<lds_bf16x4 *>((uintptr_t)(base ^ ((2 * u + 1) << 4))) = p1;
}
__device__ __forceinline__ void ds_store_zero(uint32_t base) {
    bf16x8 z;
#pragma unroll
    for (int e = 0; e < 8; ++e) z[e] = (bf16)0.0f;
    ds_store(base, 0, z);
    ds_store(base, 1, z);
}

// Which (row, key) pairs of a block are visible: per accumulator register the lanes (keys) that see its row.  Row r sees the key iff 0 <= dbase + r <
// weff and r < row_lim, dbase = (first query position) - (this lane's key), or a huge negative number for a dead key.  With r = rc + 4*half (rc a compile-time
// constant per accumulator register) that is (unsigned)(dbh + rc) < width.  The same for all heads: formed once per query block, in scalar registers.
struct WinMask { uint64_t lanes[16]; };
__device__ __forceinline__ void window_mask(WinMask &m, int dbase, unsigned weff, int row_lim, int half) {
    const int dbh = dbase + 4 * half;
    const unsigned width = (unsigned)max(0, min((int)weff, dbh + max(row_lim, -8) - 4 * half));
#pragma unroll
    for (int i = 0; i < 16; ++i) m.lanes[i] = __builtin_amdgcn_ballot_w64((unsigned)(dbh + crow(i, 0)) < width);
}

// One block of 32 query rows against an owner's 32 keys.  at: lane offsets of the staged Q tile (dO 4 KB behind it);
// stat_lane: address of this lane's first -lse / scale (rows 4*half..), -delta 32 floats further on.
// The bf16 dS values go to LDS, key-major: the lane's key row at ds_out (which holds the row's swizzle, see ds_store_addr).
__device__ __forceinline__ void window_block(uint32_t stat_lane, const TileLaneOffsets &at, const bf16x8 (&kf)[4], const bf16x8 (&vf)[4],
                                             f32x16 (&dk)[2], f32x16 (&dv)[2], float c, const WinMask &mask, uint32_t ds_out) {
    f32x16 s, dp;
    // the accumulators start at -lse / scale and at -delta of their rows, so the MFMAs deliver S - lse / scale and dP - delta
#pragma unroll
    for (int a4 = 0; a4 < 4; ++a4) {
        const f32x4 nl = lds_load128f(stat_lane, 8 * a4 * 4), nd = lds_load128f(stat_lane, (WinCfg::kRows + 8 * a4) * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { s[4 * a4 + e] = nl[e]; dp[4 * a4 + e] = nd[e]; }
    }
    // Fragments are requested ahead of the MFMAs that take them: a step or two of the S / dP contraction, then the transposed ones of the first 16 rows
    // while the exponentials run (the fences keep the compiler from moving a read next to its use, where a wavefront waits for each).
    bf16x8 fq[4], fg[4], tg[2], tq[2];
    auto natural = [&](int ks) __attribute__((always_inline)) { fq[ks] = ofrag_nat(0u, at, 0, ks); fg[ks] = ofrag_nat(0u, at, 1, ks); };
    auto transposed = [&](int u, int dblk) __attribute__((always_inline)) { tg[dblk] = ofrag_tr(0u, at, 1, u, dblk); tq[dblk] = ofrag_tr(0u, at, 0, u, dblk); };
    auto contract = [&](int ks) __attribute__((always_inline)) {
        s = mfma_bf16(fq[ks], kf[ks], s);
        dp = mfma_bf16(fg[ks], vf[ks], dp);
    };
    natural(0);
    natural(1);
    __builtin_amdgcn_sched_barrier(0);
    contract(0);
    natural(2);
    __builtin_amdgcn_sched_barrier(0);
    contract(1);
    natural(3);
    __builtin_amdgcn_sched_barrier(0);
    contract(2);
    transposed(0, 0);
    __builtin_amdgcn_sched_barrier(0);
    contract(3);
    transposed(0, 1);
    __builtin_amdgcn_sched_barrier(0);
    auto weights = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 8 * u; i < 8 * u + 8; ++i) {
            const float pe = __builtin_amdgcn_inverse_ballot_w64(mask.lanes[i]) ? fast_exp2(s[i] * c) : 0.0f;
            s[i] = pe;
            dp[i] = pe * dp[i];
        }
    };
    auto sums = [&](int u) __attribute__((always_inline)) {
        const bf16x8 pf = cfrag(s, u), dsf = cfrag(dp, u);
        ds_store(ds_out, u, dsf);
#pragma unroll
        for (int dblk = 0; dblk < 2; ++dblk) {
            dv[dblk] = mfma_bf16(tg[dblk], pf, dv[dblk]);
            dk[dblk] = mfma_bf16(tq[dblk], dsf, dk[dblk]);
        }
    };
    weights(0);
    sums(0);
    transposed(1, 0);
    transposed(1, 1);
    __builtin_amdgcn_sched_barrier(0);
    weights(1);
    sums(1);
}

// store_rows32 with the row addresses as scalar base + 32-bit lane offset (row strides are at most 2^24 elements): one lane register
// instead of a 64-bit address per row.
__device__ __forceinline__ void window_store_rows(bf16 *stage, const f32x16 (&acc)[2], float mul, bf16 *grow0, int stride, int nvalid, int lane) {
    const int l32 = lane & 31, half = lane >> 5;
#pragma unroll
    for (int dblk = 0; dblk < 2; ++dblk)
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) {
            bf16x4 pk;
#pragma unroll
            for (int e = 0; e < 4; ++e) pk[e] = (bf16)(acc[dblk][4 * a4 + e] * mul);
            *reinterpret_cast<bf16x4 *>(stage + l32 * kLS + 32 * dblk + 8 * a4 + 4 * half) = pk;
        }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int c = lane & 7, rr = lane >> 3;
    const uint32_t off = (uint32_t)(rr * stride + c * 8) * 2u;
    char *at = reinterpret_cast<char *>(grow0);
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {
        if (rr + 8 * pass < nvalid) *reinterpret_cast<u32x4 *>(at + off) = *reinterpret_cast<const u32x4 *>(stage + (rr + 8 * pass) * kLS + c * 8);
        at += (int64_t)stride * 16;
    }
    __builtin_amdgcn_wave_barrier();
}

__global__ __launch_bounds__(WinCfg::NWAVES * 64, 1) void attn_bwd_window_kernel(const KArgs a) {
    using C = WinCfg;
    constexpr int NS = C::NS, kRows = C::kRows;
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    float *const sstat = reinterpret_cast<float *>(lds + C::kStatOff);

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform: keeps everything derived from it in scalar registers
    const int l32 = lane & 31, half = lane >> 5;
    // the lane index for rare code, formed there: derived from `lane` its addresses would be held, or spilled, throughout the walk
    auto fresh_lane = []() __attribute__((always_inline)) {
        int n = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        asm volatile("" : "+v"(n));
        return n;
    };
    const bool owner = w < C::NOWN;
    const int grp = owner ? (w >= C::NSLOT) : w - C::NOWN;    // group: even or odd heads of the walk

    int bid = blockIdx.x;
    const int g = bid % a.G; bid /= a.G;
    const int b = bid % a.B; bid /= a.B;
    const int chunk = bid;
    const int n_chunks = gridDim.x / (a.G * a.B);
    const int n_blocks = (a.Sq + kRows - 1) / kRows;
    const int u0 = chunk * a.chunk_blocks;                 // first query block (and first own key block)
    const int u1 = min(u0 + a.chunk_blocks, n_blocks);     // end of the chunk
    const bool seam_sums = a.boundary_partial != nullptr;  // see the file comment
    const int u_end = seam_sums ? u1 : min(u1 + C::kBack, n_blocks);
    const int pairs = (a.r + 1) / 2;                       // steps per query block
    const int n_it = (u_end - u0) * pairs;

    const int kv_len = a.seqlens ? min(a.Skv, a.seqlens[b]) : a.Skv;
    const int q_len = a.seqlens ? a.seqlens[b] : 0x7fffffff;

    const int u_rows = min(u_end, (min(a.Sq, q_len) + kRows - 1) / kRows);     // query blocks with rows that exist

    const TileLaneOffsets lo = make_tile_offsets(lane);
    const uint32_t stage_base = lds_addr(lds + C::kStageOff), stat_base = lds_addr(sstat), ds_base = lds_addr(lds + C::kDsOff);
    const uint32_t transit_base = lds_addr(lds + C::kTransitOff);
    const bf16 *kbase = a.k + (int64_t)b * a.ks.b + (int64_t)g * a.ks.h;
    const bf16 *vbase = a.v + (int64_t)b * a.vs.b + (int64_t)g * a.vs.h;

    // key block that slot p holds while the walk is at query block u: the one of u-4 .. u that is congruent to p modulo 5
    auto block_of_slot = [](int p, int u) { return u - ((u - p) % C::NSLOT + C::NSLOT) % C::NSLOT; };

    // ---- copies of the walk's Q / dO tiles: wavefronts 5 to 8 (owners of group 1), one (group, tensor) each,
    // four 16-byte-per-lane instructions per step; K / V of the next key block: wavefront 9 ----
    constexpr int kWaveTile0 = C::NSLOT, kWaveTransit = C::NSLOT + 4;
    const bool copies = w >= kWaveTile0 && w < kWaveTile0 + 4;
    const int cp_grp = ((w - kWaveTile0) >> 1) & 1, cp_do = (w - kWaveTile0) & 1;
    const int64_t cp_hs = (cp_do ? a.dos.h : a.qs.h) * 2;      // bytes
    const int cp_s = (int)(cp_do ? a.dos.s : a.qs.s);
    const int cp_heads = (a.r - cp_grp + 1) / 2;               // (a step without a head for group 1 re-reads its last one)
    const char *cp_tile = reinterpret_cast<const char *>((cp_do ? a.d_o : a.q) + (int64_t)b * (cp_do ? a.dos.b : a.qs.b)) + (g * a.r + cp_grp) * cp_hs +
                          (int64_t)(u0 * kRows) * cp_s * 2;
    WinPos p_cp{u0, 0};
    // lane offset of rows 0..7 of a block; eight rows further on 16-byte chunk c is chunk c ^ 2, sixteen rows further on c again
    const uint32_t cp_off = (uint32_t)((lane >> 3) * cp_s + (((lane & 7) ^ swz(lane >> 3)) * 8)) * 2u;
    auto issue = [&](int it) __attribute__((always_inline)) {
        const uint32_t dst = stage_base + (((it % NS) * 2 + cp_grp) * 2 + cp_do) * C::kBlockBytes;
        const int over = a.Sq - p_cp.u * kRows;
        if (over >= kRows) {
            const uint32_t off2 = cp_off + 32u - (uint32_t)((fresh_lane() & 2) << 5);
            const int64_t eight = (int64_t)cp_s * 16;
            lds_dma16(dst, cp_tile, cp_off);
            lds_dma16_plus<8 * kRowBytes>(dst, cp_tile + eight, off2);
            lds_dma16_plus<16 * kRowBytes>(dst, cp_tile + 2 * eight, cp_off);
            lds_dma16_plus<24 * kRowBytes>(dst, cp_tile + 3 * eight, off2);
        } else {                                               // rows past the end of the tensor re-read the last one
            const int ln = fresh_lane();
#pragma unroll 1
            for (int k = 0; k < 4; ++k) {
                const int rr = 8 * k + (ln >> 3);
                lds_dma16(dst + k * 8 * kRowBytes, cp_tile, (uint32_t)(min(rr, over - 1) * cp_s + (((ln & 7) ^ swz(rr)) * 8)) * 2u);
            }
        }
        ++p_cp.hp;
        cp_tile += p_cp.hp < cp_heads ? 2 * cp_hs : p_cp.hp < pairs ? 0 : (int64_t)cp_s * (2 * kRows) - 2 * (cp_heads - 1) * cp_hs;
        if (p_cp.hp == pairs) { p_cp.hp = 0; ++p_cp.u; }
    };
    auto issue_transit = [&](int kb) __attribute__((always_inline)) {
        const uint32_t dst = transit_base + (kb & 1) * (2 * C::kBlockBytes);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int ln = fresh_lane(), rr = 8 * k + (ln >> 3);
            const int64_t row = min(kb * kRows + rr, a.Skv - 1);
            const int cc = (ln & 7) ^ swz(rr);
            lds_dma16(dst + k * 8 * kRowBytes, kbase + (int64_t)(kb * kRows) * a.ks.s, (uint32_t)((row - kb * kRows) * a.ks.s + cc * 8) * 2u);
            lds_dma16(dst + C::kBlockBytes + k * 8 * kRowBytes, vbase + (int64_t)(kb * kRows) * a.vs.s, (uint32_t)((row - kb * kRows) * a.vs.s + cc * 8) * 2u);
        }
    };

    // ---- prologue: the five key blocks live at the first query block, and the first three steps' tiles -----------
    // Their K rows go through LDS (slot p of the first dS buffer) so that the helpers can pick
    // them up as transposed fragments; rows outside the tensor repeat a valid row (finite values
    // that only ever meet dS = 0).
    for (int i = w; i < 4 * C::NSLOT; i += C::NWAVES) {
        const int p = i >> 2, r8 = i & 3;
        const int rr = 8 * r8 + (lane >> 3);
        const int cc = (lane & 7) ^ swz(rr);
        const int row = min(max(block_of_slot(p, u0) * kRows + rr, 0), a.Skv - 1);
        __builtin_amdgcn_global_load_lds((glb_void_t *)(kbase + (int64_t)row * a.ks.s + cc * 8),
                                         (lds_void_t *)(lds + C::kDsOff + p * C::kBlockBytes + r8 * 8 * kRowBytes), 16, 0, 0);
    }
    if (copies) {
        for (int it = 0; it < min(n_it, NS - 1); ++it) issue(it);
    }

    if (!owner) {
        // the two helpers are the only wavefronts of their kind; whenever one of them can issue it goes
        // before the owners it shares its SIMD with
        __builtin_amdgcn_s_setprio(1);
        // =================================== helper wavefronts ===================================
        const int srow = lane >> 1, hr = lane & 1;                 // statistics: two lanes per row, 32 columns each
        bf16 *const out_stage = reinterpret_cast<bf16 *>(lds + C::kOutOff) + grp * kRows * kLS;
        // dSinks terms are summed per lane (own LDS slot per head, no cross-lane traffic in the loop)
        float *const sink_sums = reinterpret_cast<float *>(lds + C::kSinkOff) + grp * (C::kMaxGroup / 2) * 64;
        float *const sink2 = reinterpret_cast<float *>(lds + C::kLogitOff) + grp * (C::kMaxGroup / 2);   // sink logits * log2(e)
        for (int h = 0; h < pairs; ++h) {
            sink_sums[h * 64 + lane] = 0.0f;
            if (lane == 0) sink2[h] = sink_logit(a, g * a.r + min(2 * h + grp, a.r - 1)) * kLog2e;
        }

        // The group's rows of the walk, one step after the other, as byte addresses: O and lse two steps ahead, dQ one behind.
        const int grp_heads = (a.r - grp + 1) / 2;             // (a step without a head for group 1 re-reads its last one)
        auto advance = [&](const char *&at, WinPos &pos, int64_t head, int64_t row) __attribute__((always_inline)) {
            ++pos.hp;
            at += pos.hp < grp_heads ? 2 * head : pos.hp < pairs ? 0 : kRows * row - 2 * (grp_heads - 1) * head;
            if (pos.hp == pairs) { pos.hp = 0; ++pos.u; }
        };
        const int64_t head0 = g * a.r + grp, row_0 = (int64_t)u0 * kRows;
        const char *o_at = reinterpret_cast<const char *>(a.o + (int64_t)b * a.os.b + head0 * a.os.h + row_0 * a.os.s);
        const char *lse_at = reinterpret_cast<const char *>(a.lse + ((int64_t)b * a.H + head0) * a.Sq + row_0);
        const char *dq_at = reinterpret_cast<const char *>(a.dq + (int64_t)b * a.dqs.b + head0 * a.dqs.h + row_0 * a.dqs.s);
        const float inv_scale = 1.0f / fmaxf(a.scale, C::kMinScale);
        // O half rows + lse of this lane's row of a walk position (rows past the end of the tensor re-read the last one)
        u32x4 pre_o[4];
        float pre_lse = 0.0f;
        auto prefetch = [&](WinPos &pos) __attribute__((always_inline)) {
            const int row = min(srow, a.Sq - 1 - pos.u * kRows);
            const uint32_t off = (uint32_t)(row * (int)a.os.s + 32 * hr) * 2u;
#pragma unroll
            for (int j = 0; j < 4; ++j) pre_o[j] = *reinterpret_cast<const u32x4 *>(o_at + off + 16 * j);
            pre_lse = *reinterpret_cast<const float *>(lse_at + (uint32_t)row * 4u);
            WinPos p = pos;
            advance(o_at, p, a.os.h * 2, a.os.s * 2);
            advance(lse_at, pos, (int64_t)a.Sq * 4, 4);
        };
        // row statistics of the prefetched rows, dO from stage it % NS; dSinks terms of own rows
        const uint32_t do_lane = stage_base + (grp * 2 + 1) * C::kBlockBytes + srow * kRowBytes + (((4 * hr) ^ swz(srow)) << 4);
        auto statistics = [&](const WinPos &pos, int it) __attribute__((always_inline)) {
            typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
            const uint32_t at = do_lane + (it % NS) * (4 * C::kBlockBytes);
            u32x4 dov[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) dov[j] = lds_load128(at ^ (j << 4), 0);
            __builtin_amdgcn_sched_barrier(0);                 // (all four reads under way together)
            float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    union { uint32_t u; bf16x2 v; } x, y;
                    x.u = pre_o[j][e];
                    y.u = dov[j][e];
                    part[e] = __builtin_amdgcn_fdot2_f32_bf16(x.v, y.v, part[e], false);
                }
            float nd = -((part[0] + part[1]) + (part[2] + part[3]));
            nd += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(nd), 0xB1, 0xF, 0xF, true));     // + the other half row's (lane ^ 1)
            float *const st = sstat + (((it & 1) * 2 + grp) * 2) * kRows + srow;
            if (hr == 0) {
                st[0] = -pre_lse * inv_scale;
                st[kRows] = nd;
            }
            const int h = 2 * pos.hp + grp;
            if (a.dsinks && pos.u < u1 && h < a.r) {            // rows of the chunk itself, each counted once
                const float term = (hr == 0 && pos.u * kRows + srow < a.Sq) ? fast_exp2(sink2[pos.hp] - pre_lse * kLog2e) * nd : 0.0f;
                // (a lane's own word: the order of the additions is that of the walk)
                __builtin_amdgcn_ds_faddf((__attribute__((address_space(3))) float *)(sink_sums + pos.hp * 64 + lane), term, 0, 0, false);
            }
        };
        // dQ rows of the group's tile at `pos` from the dS blocks at LDS address ds_tile
        const uint32_t ds_lane[2] = {grp ? lo.tr[1][0] : lo.tr[0][0], grp ? lo.tr[1][1] : lo.tr[0][1]};
        bf16x8 kfr[C::NSLOT][2][2];
        auto helper_dq = [&](uint32_t ds_tile, const WinPos &pos) __attribute__((always_inline)) {
            constexpr int kSteps = 2 * C::NSLOT, kAhead = 4;
            f32x16 acc[2];
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[db][i] = 0.0f;
            if (pos.u < u_rows) {                              // (K rows of padding may hold anything)
                bf16x8 f[kSteps];
                auto request = [&](int k) __attribute__((always_inline)) {
                    const int imm = (k >> 1) * C::kBlockBytes + 16 * (k & 1) * kRowBytes;
                    union { struct { s16x4 a, b; } s; bf16x8 v; } x;
                    x.s.a = lds_load_tr64(ds_tile + ds_lane[0], imm);
                    x.s.b = lds_load_tr64(ds_tile + ds_lane[1], imm);
                    f[k] = x.v;
                };
#pragma unroll
                for (int k = 0; k < kAhead; ++k) request(k);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < kSteps; ++k) {
#pragma unroll
                    for (int db = 0; db < 2; ++db) acc[db] = mfma_bf16(kfr[k >> 1][k & 1][db], f[k], acc[db]);
                    if (k + kAhead < kSteps) request(k + kAhead);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            window_store_rows(out_stage, acc, a.scale, reinterpret_cast<bf16 *>(const_cast<char *>(dq_at)), (int)a.dqs.s, a.Sq - pos.u * kRows, lane);
        };
        auto wants_dq = [&](const WinPos &pos) { return pos.u < u1 && 2 * pos.hp + grp < a.r; };
        auto reload = [&](auto slot_tag, uint32_t from) __attribute__((always_inline)) {
            constexpr int P = decltype(slot_tag)::value;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int db = 0; db < 2; ++db) kfr[P][kk][db] = ofrag_tr(from, lo, 0, kk, db);
        };

        WinPos p_stat{u0, 0}, p_pre{u0, 0}, p_prev{u0, 0};
        prefetch(p_pre);
        wait_vmcnt<0>();
        __syncthreads();                                       // the K blocks and the first tiles are in LDS
        // K^T fragments (A operands: lane = column, slots = keys) of the five live key blocks
#pragma unroll
        for (int p = 0; p < C::NSLOT; ++p)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int db = 0; db < 2; ++db) kfr[p][kk][db] = ofrag_tr(ds_base + p * C::kBlockBytes, lo, 0, kk, db);
        statistics(p_stat, 0);                                 // statistics of the first step
        p_stat.step(pairs);
        if (n_it > 1) prefetch(p_pre);

        WinPos cur{u0, 0};
        for (int it = 0; it < n_it; ++it) {
            __syncthreads();
            if (it + 1 < n_it) {
                statistics(p_stat, it + 1);
                p_stat.step(pairs);
            }
            if (it + 2 < n_it) prefetch(p_pre);                // (a step's time to arrive)
            if (it > 0 && wants_dq(p_prev)) helper_dq(ds_base + ((it - 1) & 1) * C::kDsBytes, p_prev);
            if (cur.hp == 0 && cur.u > u0 && cur.u < u1) {
                // key block cur.u has arrived in the transit buffer; it replaces block cur.u - 5
                const uint32_t from = transit_base + (cur.u & 1) * (2 * C::kBlockBytes);
                const int slot = cur.u % C::NSLOT;
                if (slot == 0) reload(std::integral_constant<int, 0>{}, from);
                if (slot == 1) reload(std::integral_constant<int, 1>{}, from);
                if (slot == 2) reload(std::integral_constant<int, 2>{}, from);
                if (slot == 3) reload(std::integral_constant<int, 3>{}, from);
                if (slot == 4) reload(std::integral_constant<int, 4>{}, from);
            }
            if (pairs == 1) __syncthreads();                   // (see the owners)
            if (it > 0) advance(dq_at, p_prev, a.dqs.h * 2, a.dqs.s * 2);
            cur.step(pairs);
        }
        __syncthreads();                                       // the last dS blocks are complete
        if (wants_dq(p_prev)) helper_dq(ds_base + ((n_it - 1) & 1) * C::kDsBytes, p_prev);
        __syncthreads();                                       // (group 1's owners have left their sums)
        if (a.dsinks) {
            for (int h = grp; h < a.r; h += 2) {
                float v = sink_sums[(h >> 1) * 64 + fresh_lane()];
#pragma unroll
                for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
                if (fresh_lane() == 0) a.dsink_partial[((int64_t)b * n_chunks + chunk) * a.H + g * a.r + h] = v;
            }
        }
        return;
    }

    // ===================================== owner wavefronts =====================================
    const int slot = grp ? w - C::NSLOT : w;
    int kb = block_of_slot(slot, u0), my_kb = kb;              // key block held (negative: none)
    bf16x8 kf[4], vf[4];
    f32x16 dk[2], dv[2];
    {
        const int j = my_kb * kRows + l32;
        const bool ok = my_kb >= 0 && j < a.Skv;
        const bf16 *krow = kbase + (int64_t)(ok ? j : 0) * a.ks.s;
        const bf16 *vrow = vbase + (int64_t)(ok ? j : 0) * a.vs.s;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            u32x4 zk = {0u, 0u, 0u, 0u}, zv = {0u, 0u, 0u, 0u};
            if (ok) {
                zk = *reinterpret_cast<const u32x4 *>(krow + 16 * ks + 8 * half);
                zv = *reinterpret_cast<const u32x4 *>(vrow + 16 * ks + 8 * half);
            }
            kf[ks] = as_bf16x8(zk);
            vf[ks] = as_bf16x8(zv);
        }
    }
    // Unscaled sums of one tensor as accumulator quads of 64 lanes: on their way to the owner of the same slot in the other group, and the
    // shares of seam blocks.
    // (A group's tensor is chosen value by value: chosen by branches, the accumulators end up in memory.)
    constexpr int kHalf = C::kMergeBytes / 2;
    auto quad = [&](bool of_dv, int dblk, int a4) __attribute__((always_inline)) {
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = of_dv ? dv[dblk][4 * a4 + e] : dk[dblk][4 * a4 + e];
        return x;
    };
    // into a slot's merge buffer: group 1's dK, group 0's dV
    auto exchange = [&](char *buf) __attribute__((always_inline)) {
        f32x4 *q = reinterpret_cast<f32x4 *>(buf + (grp ? 0 : kHalf)) + fresh_lane();
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j * 64] = quad(grp == 0, j >> 2, j & 3);
    };
    // fp32 share of a seam block: [b][g][seam][block 0..3][workgroup before / after the seam], dK then dV, accumulator quads of 64 lanes as above
    auto seam_share = [&](int seam, int block, int side) {
        return a.boundary_partial + (((((int64_t)b * a.G + g) * (n_chunks - 1) + seam) * C::kBack + block) * 2 + side) * (2 * kRows * kD);
    };
    // One tensor of the key block held (group 0: dK, group 1: dV), the other group's sums in `buf` added: written out if it is complete,
    // left as this workgroup's share if it sits on a seam, dropped if it belongs to the neighbour (recomputation mode).  `buf` then stages
    // the rows.
    auto flush = [&](char *buf) __attribute__((always_inline)) {
        if (my_kb < 0 || (!seam_sums && (my_kb < u0 || my_kb >= u1))) return;
        const int ln = fresh_lane();
        char *const half_buf = buf + (grp ? kHalf : 0);
        const f32x4 *q = reinterpret_cast<const f32x4 *>(half_buf) + ln;
        f32x16 sum[2];
#pragma unroll
        for (int dblk = 0; dblk < 2; ++dblk) {
            f32x4 x[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = q[(4 * dblk + j) * 64];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const f32x4 own = quad(grp == 1, dblk, j);
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[dblk][4 * j + e] = own[e] + x[j][e];
            }
            asm volatile("" ::: "memory");                     // (four reads at a time: all eight would spill what the walk holds)
        }
        float *share = nullptr;
        if (seam_sums && my_kb < u0) share = seam_share(chunk - 1, my_kb - (u0 - C::kBack), 1);
        else if (seam_sums && my_kb >= u1 - C::kBack && u1 < n_blocks) share = seam_share(chunk, my_kb - (u1 - C::kBack), 0);
        if (share) {
            f32x4 *to = reinterpret_cast<f32x4 *>(share + grp * (kRows * kD)) + ln;
#pragma unroll
            for (int j = 0; j < 8; ++j) to[j * 64] = f32x4{sum[j >> 2][4 * (j & 3)], sum[j >> 2][4 * (j & 3) + 1], sum[j >> 2][4 * (j & 3) + 2], sum[j >> 2][4 * (j & 3) + 3]};
            return;
        }
        const int r0 = my_kb * kRows;
        const Strides &st = grp ? a.dvs : a.dks;
        window_store_rows(reinterpret_cast<bf16 *>(half_buf), sum, grp ? 1.0f : a.scale, (grp ? a.dv : a.dk) + (int64_t)b * st.b + (int64_t)g * st.h + (int64_t)r0 * st.s, (int)st.s,
                          a.Skv - r0, ln);
    };

    const float c = a.scale_log2;
    const uint32_t ds_out0 = ds_store_addr(ds_base + slot * C::kBlockBytes, l32, half) ^ (grp << 6);
    wait_vmcnt<0>();
    __syncthreads();                                           // prologue barrier (the helpers read the K blocks now)

    // the fragment offsets with the address of the stage at hand folded in: one add each per step, and every
    // read of the step's Q and dO tiles is (register) + (immediate)
    uint32_t at_stage = stage_base + grp * (2 * C::kBlockBytes);
    TileLaneOffsets at = tile_offsets_at(lo, at_stage);
    int it = 0, u = u0, hp = 0;                                // the step, and its place in the walk
    auto begin = [&]() __attribute__((always_inline)) {
        // this step's tiles and the next one's (whose dO the helpers read now) have arrived
        if (copies) { if (it + 2 >= n_it) wait_vmcnt<0>(); else wait_vmcnt<4>(); }
        else if (w == kWaveTransit && hp == 0) wait_vmcnt<0>();       // the transit copy of the key block that starts now
        __syncthreads();
        const uint32_t to = stage_base + ((it % NS) * 2 + grp) * (2 * C::kBlockBytes);
        tile_offsets_move(at, to - at_stage);
        at_stage = to;
    };
    auto copy_ahead = [&]() __attribute__((always_inline)) {
        // (one step per query block: the other group may still be reading the sums that this one left)
        if (pairs == 1) __syncthreads();
        if (w == kWaveTransit && hp == 0 && u + 1 < u1) issue_transit(u + 1);
        if (copies && it + NS - 1 < n_it) issue(it + NS - 1);
    };
    auto ds_out = [&]() { return ds_out0 + (it & 1) * C::kDsBytes; };
    auto next = [&]() __attribute__((always_inline)) {
        ++it;
        if (++hp == pairs) { hp = 0; ++u; }
    };
    // A key block stays with its owner for the five query blocks that may see it: the ones that do, then those that only keep the rhythm.
    // Each is a plain loop (with the kinds of blocks as branches of one loop the compiler copies the 64 accumulator registers every step).
    const int behind = (a.window + kRows - 2) / kRows;         // query blocks behind its own that see a key block
    for (;;) {
        begin();
        if (u > u0) {
            flush(lds + C::kMergeOff);                         // the block held so far
            kb += C::NSLOT;
            my_kb = u < u1 ? u : -1;
            const uint32_t from = transit_base + (u & 1) * (2 * C::kBlockBytes) - at_stage;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                kf[ks] = ofrag_nat(from, at, 0, ks);
                vf[ks] = ofrag_nat(from, at, 1, ks);
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) { dk[0][i] = dk[1][i] = 0.0f; dv[0][i] = dv[1][i] = 0.0f; }
        const int wj0 = my_kb * kRows;                         // first key of the wavefront
        const int u_seen = my_kb >= 0 && wj0 < kv_len ? min(my_kb + behind + 1, u_rows) : u;
        const int u_last = min(kb + C::NSLOT, u_end);
        bool begun = true;
        if (u < u_seen) {
            WinMask mask;
            for (;;) {
                copy_ahead();
                if (hp == 0 || (grp == 1 && (a.r & 1))) {
                    const int ln = fresh_lane(), i0 = u * kRows, j = wj0 + (ln & 31);
                    const int dbase = j < kv_len ? i0 - j : -0x40000000;
                    // (a step without a head for group 1: nothing of it counts)
                    window_mask(mask, dbase, 2 * hp + grp < a.r ? (unsigned)a.window : 0u, min(min(a.Sq, q_len) - i0, kRows), ln >> 5);
                }
                window_block(stat_base + (((it & 1) * 2 + grp) * 2 * kRows + half * 4) * 4, at, kf, vf, dk, dv, c, mask, ds_out());
                next();
                if (u == u_seen) break;
                begin();
            }
            begun = false;
        }
        while (u < u_last) {
            if (!begun) begin();
            begun = false;
            copy_ahead();
            ds_store_zero(ds_out());
            next();
        }
        if (u == u_end) break;
        exchange(lds + C::kMergeOff);
    }
    __syncthreads();                                           // hands the last dS blocks over; nobody reads a stage any more
    char *const last = lds + C::kStageOff + slot * C::kMergeBytes;
    exchange(last);
    __syncthreads();
    flush(last);
}

// ---------------------------------------------------------------------------------
// What is left after the window kernel, in one small launch.  Blocks [0, seam_blocks): dK / dV of
// the seam blocks = round(scale * (share of the workgroup before the seam + share of the one after)),
// one thread per 16-byte output chunk.  Blocks from seam_blocks on: one block per query head adds
// that head's dSinks partial sums (per batch row and chunk) in a fixed tree order.
__global__ __launch_bounds__(256) void attn_bwd_window_finish_kernel(const KArgs a, int n_chunks, int seam_blocks) {
    if ((int)blockIdx.x >= seam_blocks) {
        __shared__ float red[256];
        const int h = blockIdx.x - seam_blocks;
        const int n = a.B * n_chunks;
        float acc = 0.0f;
        for (int i = threadIdx.x; i < n; i += 256) acc += a.dsink_partial[(int64_t)i * a.H + h];
        red[threadIdx.x] = acc;
        __syncthreads();
        for (int off = 128; off > 0; off >>= 1) {
            if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
            __syncthreads();
        }
        if (threadIdx.x == 0) store_dsink(a, h, red[0]);
        return;
    }
    // chunk index over (b, g, seam, block, tensor, key, 8 columns)
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int c8 = (int)(idx & 7) * 8;
    const int key = (int)((idx >> 3) & 31);
    const int which = (int)((idx >> 8) & 1);                      // 0 = dK, 1 = dV
    const int block = (int)((idx >> 9) & 3);
    const int64_t rest = idx >> 11;                               // (b * G + g) * (n_chunks - 1) + seam
    if (rest >= (int64_t)a.B * a.G * (n_chunks - 1)) return;
    const int seam = (int)(rest % (n_chunks - 1));
    const int bg = (int)(rest / (n_chunks - 1));
    const int g = bg % a.G, b = bg / a.G;
    const int row = ((seam + 1) * a.chunk_blocks - WinCfg::kBack + block) * WinCfg::kRows + key;
    if (row >= a.Skv) return;
    // eight columns of a key: the quads of both halves of its lane pair (accumulator order, see quad and seam_share)
    const float *before = a.boundary_partial + ((rest * WinCfg::kBack + block) * 2) * (2 * WinCfg::kRows * kD) + ((which * 8 + c8 / 8) * 64 + key) * 4;
    const float *after = before + 2 * WinCfg::kRows * kD;
    const float mul = which == 0 ? a.scale : 1.0f;
    bf16x8 out;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const f32x4 x = *reinterpret_cast<const f32x4 *>(before + 128 * j), y = *reinterpret_cast<const f32x4 *>(after + 128 * j);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[4 * j + e] = (bf16)((x[e] + y[e]) * mul);
    }
    const Strides &st = which == 0 ? a.dks : a.dvs;
    bf16 *dst = (which == 0 ? a.dk : a.dv) + (int64_t)b * st.b + (int64_t)g * st.h + (int64_t)row * st.s + c8;
    union { bf16x8 v; u32x4 u; } cv;
    cv.v = out;
    *reinterpret_cast<u32x4 *>(dst) = cv.u;
}

}  // namespace gptoss
