// Forward kernel for full-causal rows (bf16, no window, query heads per KV head a multiple of 4): the formulas of
// attn_fwd_kernel<4, 2> (attn_fwd.h; the reference's `_attn_fwd`, attention_kernel.py:11-100) with the
// interior key tiles software-pipelined by hand.  Against that kernel only the order of the row sums of a
// row's first tile differs: lse agrees to a few units of its last place, O to one bf16 rounding.
//
// Why.  Two wavefronts share a SIMD.  attn_fwd_kernel's wavefront issues its MFMAs in clumps of eight with a
// softmax step (about 120 vector instructions, no MFMA) between them; while one wavefront sits in such a
// vector stretch the matrix pipe has only the other one to feed it, and when both do, it idles.  An
// instruction stream in which every MFMA is followed by its share of the vector work keeps both pipes
// supplied whatever the phase of the neighbour: measured with synthetic streams of the forward's
// instruction mix at two wavefronts per SIMD, 53.6 cycles per MFMA against 58.8 for the clumped order.
//
// How.  A tile is four units u = (32-key block kb, 32-row block qb).  Slot u issues, as eight micro-slots
// of {one MFMA, two elements of softmax, at most two LDS reads} closed by sched_barrier(0):
//   * the four S MFMAs of unit u + 1 (the next tile's first unit in the tile's last slot),
//   * the four O += P V MFMAs of unit u - 1,
//   * exp2 / row sum / bf16 packing of unit u's sixteen logits per lane.
// K fragments (natural) and V fragments (transposed) each feed both row blocks and are reloaded in place
// right after their last use, one slot before their first.  The next tile must have landed before the
// third slot of a tile (which loads its first K fragments), so the iteration's barrier sits there; with four
// LDS stages the copy requested at that barrier is two tiles ahead, as in attn_fwd_kernel.
// The softmax reference of a row (see fwd_tile_lean) is the sink logit or the largest logit of the row's first
// tile, taken by a pass over that tile that forms the logits and nothing else; the tile then goes through the
// loop like the others.  The diagonal tile (masked) goes through attn_fwd.h's fwd_tile_lean; rows of a single
// key tile, and the rare second pass of a workgroup whose frozen reference turned out too low, go through one
// loop of exact steps (fwd_tile).
#pragma once
#include <type_traits>

#include "attn_fwd.h"

namespace gptoss {

struct FwdPipe {
    static constexpr int NS = 4;                                  // LDS stages
    static constexpr int kStageBytes = 2 * kStageTileBytes;       // K tile, V tile
};

// The plain instantiation is for self-attention of whole tiles (Sq == Skv a multiple of 64, nothing else): key tiles
// 0 .. qt - 1 are interior, tile qt is the diagonal.  GENERAL takes any lengths, a query offset, right-padded batch rows and
// packed documents (64 keys at least).  A workgroup's key tiles are then [t_lo, t_hi): first the tile in front of t_a, where a
// packed row's document starts inside a tile (an exact masked step, which also gives the softmax reference); the interior
// tiles [t_a, t_b) through the pipeline; the tiles from t_b on (the diagonal, which an offset spreads over two tiles, and
// the end of the keys) with masked steps.  Where a document ends inside the workgroup's rows, only the rows of
// the first one see the tiles in front of the diagonal: the others run along unmasked (like rows that do not exist, past
// the tensor or the padding: their values are garbage but finite or at worst NaN, and stay in their own lanes) and start
// afresh at the diagonal tile.  Workgroups without any row that exists write O = 0 and lse = sink and do nothing else.
// Measured against attn_fwd_kernel, which took these cases before (64 query heads on 8 KV heads): 1024 queries behind 7168
// keys 181 -> 135 us a call; 2 x 3001 tokens 164 -> 160 us, 1 x 1000 33.6 -> 25.2, 2 x 383 16.1 -> 14.8; seven documents in 8192 tokens
// 185 -> 180 (without letting the other documents' rows run along, every tile of such a workgroup being an exact
// step: 230).
// Few queries on a long cache, or few heads, leave most of the chip idle (100 queries on 4096 keys: 32 workgroups).  With kv_splits > 1 a query block's
// key tiles are cut into that many consecutive shares, one workgroup each, which leave their unnormalised rows with (reference,
// sum) in the scratch; attn_fwd_combine_kernel adds them in share order.  Each share freezes a reference of its own (100 queries on 4096 keys
// of 64 heads: 62 -> 30 us, the sum included; 4000 tokens of 8 heads 60 -> 41).
template <bool GENERAL, bool DOCS = false>       // DOCS: packed documents (needs GENERAL)
__global__ __launch_bounds__(256, 2) void attn_fwd_pipe_kernel(const KArgs a) {
    constexpr int NS = FwdPipe::NS;
    constexpr int SB = FwdPipe::kStageBytes;
    __shared__ __attribute__((aligned(16))) char smem[NS][2][kStageTileBytes];

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);      // wave-uniform: the head and everything derived from it stay in scalar registers
    const int l32 = lane & 31, half = lane >> 5;
    // What follows the pipelined loop (the diagonal tile, the rare second pass, the epilogue) recomputes the lane
    // index and what hangs on it, so that none of it has to live through the loop in a register file that is full there.
    auto fresh_lane = []() __attribute__((always_inline)) { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); };

    // workgroup -> (kv head, chunk of 4 heads, batch, query tile), as attn_fwd_kernel; longest key loops first
    const int n_hc = a.r / 4;
    int bid = blockIdx.x;
    const int g = bid % a.G; bid /= a.G;
    const int hc = bid % n_hc; bid /= n_hc;
    int split = 0;                                 // few query blocks: a share of the key tiles each (see attn_fwd_combine_kernel)
    if constexpr (GENERAL && !DOCS) { split = bid % a.kv_splits; bid /= a.kv_splits; }
    const int bi = bid % a.B; bid /= a.B;
    const int b = rotated_batch_row(bi, bid, a.B);
    const int q_offset = GENERAL ? query_offset(a) : 0;
    const int qt = (GENERAL ? (a.Sq + kTile - 1) / kTile : a.Sq / kTile) - 1 - bid;
    const int head = g * a.r + hc * 4 + w;
    const int qw0 = qt * kTile;                    // the four wavefronts hold the same 64 rows of four heads
    int t_lo = 0, t_a = 0, t_b = qt, t_hi = qt + 1;                       // see above
    int kv_len = a.Skv, q_len = 0x7fffffff;                               // keys / query positions from here on do not exist
    const int32_t *dsrow = nullptr;
    if constexpr (GENERAL) {
        if (a.seqlens) { q_len = a.seqlens[b]; kv_len = max(0, min(a.Skv, q_len)); }
        const int pos0 = q_offset + qw0, pos1 = min(q_offset + min(a.Sq, qw0 + kTile) - 1, q_len - 1);
        int ds0 = 0;
        bool later = false;
        if constexpr (DOCS) {
            dsrow = a.doc_start + (int64_t)b * a.Sq;
            ds0 = max(dsrow[qw0], 0);
            // (starts that are not the first row of their document, so that a later document reaches in front of these rows,
            // leave no interior tile)
            const int ds = dsrow[min(qw0 + lane, a.Sq - 1)];
            later = ds > ds0 && ds < qw0;
        }
        const int hi = pos1 >= pos0 ? min(kv_len, pos1 + 1) : 0;
        t_lo = DOCS ? __builtin_amdgcn_readfirstlane(ds0 / kTile) : 0;
        t_hi = __builtin_amdgcn_readfirstlane(max(t_lo, (hi + kTile - 1) / kTile));
        if constexpr (DOCS) t_a = __builtin_amdgcn_ballot_w64(later) != 0ull ? t_hi : __builtin_amdgcn_readfirstlane((ds0 + kTile - 1) / kTile);
        t_b = __builtin_amdgcn_readfirstlane(min(pos0 + 1, kv_len) / kTile);
        if constexpr (!DOCS) {
            if (a.kv_splits > 1) {
                const int n = t_hi;
                t_lo = t_a = (int)((int64_t)n * split / a.kv_splits);
                t_hi = (int)((int64_t)n * (split + 1) / a.kv_splits);
                t_b = min(max(t_b, t_lo), t_hi);
            }
        }
    }
    const int n_it = t_hi - t_lo;

    const bf16 *kbase = a.k + (int64_t)b * a.ks.b + (int64_t)g * a.ks.h;
    const bf16 *vbase = a.v + (int64_t)b * a.vs.b + (int64_t)g * a.vs.h;

    bf16x8 qf[2][4];
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
        const int row = GENERAL ? min(qw0 + 32 * qb + l32, a.Sq - 1) : qw0 + 32 * qb + l32;
        const bf16 *qrow = a.q + (int64_t)b * a.qs.b + (int64_t)head * a.qs.h + (int64_t)row * a.qs.s;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) qf[qb][ks] = as_bf16x8(*reinterpret_cast<const u32x4 *>(qrow + 16 * ks + 8 * half));
    }

    const float c = a.scale_log2;
    const float sink2 = sink_logit(a, head) * kLog2e;
    const float m_first = fast_max(sink2, kNoLogit);
    float m[2], l[2];
    f32x16 o[2][2];

    const TileLaneOffsets lo = make_tile_offsets(lane);
    const uint32_t smem_base = lds_addr(&smem[0][0][0]);
    const AsyncLaneOffsets klane = make_async_offsets(a.ks.s, lane, w), vlane = make_async_offsets(a.vs.s, lane, w);
    const uint32_t copy_base = smem_base + w * (16 * kRowBytes);   // this wavefront copies rows 16 w .. 16 w + 15
    // Requests are branch-free (a branch inside the fenced loop body lets the compiler sink vector work of
    // earlier micro-slots past it): every arrive() is followed by exactly one request, and once the row's
    // tiles are exhausted a request copies the last tile again, into the stage that is free by then, so that
    // "at most one request outstanding" keeps meaning "the tile before it has landed".
    const bf16 *ktile = kbase, *vtile = vbase;
    // (a tile that sticks out of the tensor is not requested here: see fetch_end)
    const int t_req = GENERAL ? min(t_lo, a.Skv / kTile - 1) : 0, n_req = GENERAL ? max(1, min(t_hi, a.Skv / kTile) - t_req) : n_it;
    int iss_stage = 0, iss_left = n_req;
    auto issue = [&]() __attribute__((always_inline)) {       // the next tile in order, into the next stage in rotation
        // (through the inline-assembly copy: the compiler's own bookkeeping would make every LDS read that
        // follows a copy wait for all outstanding copies, i.e. for the tile just requested)
        const uint32_t dst = copy_base + iss_stage * SB;
        lds_dma16_plus<0>(dst, ktile, klane.off[0]);
        lds_dma16_plus<8 * kRowBytes>(dst, ktile, klane.off[1]);
        lds_dma16_plus<kStageTileBytes>(dst, vtile, vlane.off[0]);
        lds_dma16_plus<kStageTileBytes + 8 * kRowBytes>(dst, vtile, vlane.off[1]);
        const bool more = iss_left > 1;
        ktile += more ? kTile * a.ks.s : 0;
        vtile += more ? kTile * a.vs.s : 0;
        iss_left -= 1;
        iss_stage = (iss_stage + 1) & (NS - 1);
    };
    constexpr int kLoadsPerIt = 4;
    auto reset = [&]() __attribute__((always_inline)) {
        ktile = kbase + (GENERAL ? (int64_t)t_req * kTile * a.ks.s : 0);
        vtile = vbase + (GENERAL ? (int64_t)t_req * kTile * a.vs.s : 0);
        iss_stage = 0;
        iss_left = n_req;
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            m[qb] = m_first;
            l[qb] = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) { o[qb][0][i] = 0.0f; o[qb][1][i] = 0.0f; }
        }
        issue();
        issue();
    };
    // tile k has landed in every wavefront (the k-th call); the stage of tile k - 2 is free and takes tile k + 2
    auto arrive = [&]() __attribute__((always_inline)) {
        wait_vmcnt<kLoadsPerIt>();
        __syncthreads();
        issue();
    };
    // Tile k of the walk if it sticks out of the tensor, into its stage, rows past the end re-reading the last one; everybody
    // waits for it.  It can only be the walk's last tile, of the few workgroups that see the last keys at all, and keeping
    // its lane offsets out of the loop is worth the wait.
    auto fetch_end = [&](int k) __attribute__((always_inline)) {
        if (!GENERAL || (t_lo + k + 1) * kTile <= a.Skv) return;
        const int n0 = (t_lo + k) * kTile, last = a.Skv - 1 - n0, ln = fresh_lane();
        wait_vmcnt<0>();
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = 16 * w + 8 * j + (ln >> 3), ch = ((ln & 7) ^ swz(r)) * 16, rr = min(r, last);
            const uint32_t dst = copy_base + (k & (NS - 1)) * SB + j * 8 * kRowBytes;
            lds_dma16(dst, kbase + (int64_t)n0 * a.ks.s, (uint32_t)(rr * (int)a.ks.s) * 2u + ch);
            lds_dma16(dst + kStageTileBytes, vbase + (int64_t)n0 * a.vs.s, (uint32_t)(rr * (int)a.vs.s) * 2u + ch);
        }
        wait_vmcnt<0>();
        __syncthreads();
    };
    // A row description for the masked tile functions, from scratch (see fresh_lane): lane's position (hugely negative for a
    // row that does not exist) and how far back it sees.
    auto describe_rows = [&](int l32_, int (&pq)[2], unsigned (&wl)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            const int row = qw0 + 32 * qb + l32_, p = q_offset + row;
            pq[qb] = row < a.Sq && p < q_len ? p : -0x40000000;
            wl[qb] = 0x3fffffffu;
            if (DOCS) wl[qb] = (unsigned)(p - dsrow[min(row, a.Sq - 1)] + 1);
        }
    };
    // Workgroups without an interior tile (rows of a single key tile) go straight to the exact pass below.
    const bool pipelined = n_it > 0 && t_a < t_b && t_b > t_lo;
    const int k_a = t_a - t_lo;            // tiles of the walk in front of the first interior one
    if (!pipelined) {
        // (also the state a workgroup without rows ends with: nothing requested, nothing attended)
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            m[qb] = m_first;
            l[qb] = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) { o[qb][0][i] = 0.0f; o[qb][1][i] = 0.0f; }
        }
    } else {
        reset();
        if (DOCS && k_a > 0) {
            int pq[2], dbase[2];
            unsigned wl[2];
            describe_rows(l32, pq, wl);
            for (int k = 0; k < k_a; ++k) {
                arrive();
                const int n0 = (t_lo + k) * kTile;
                const uint32_t ksm = smem_base + (k & (NS - 1)) * SB;
#pragma unroll
                for (int qb = 0; qb < 2; ++qb) dbase[qb] = pq[qb] - n0;
                fwd_tile<true, 2>(ksm, ksm + kStageTileBytes, lo, qf, o, m, l, c, lane, dbase, wl, 0x3fffffffu, kv_len - n0, q_offset + qw0 - n0);
            }
        }
        arrive();
        // The softmax reference of a row: the sink logit or the largest logit of the row's first tile
        // (ref :53, :79-81 after one tile), from a pass over that tile that forms the logits and nothing else
        // (16 MFMAs per row block, against 32 for each of its tiles).  The tile then goes through the pipelined
        // loop like every other interior tile.
        if (!DOCS || k_a == 0) {
            f32x16 s[2][2];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) {
                    const bf16x8 akf = ofrag_nat(smem_base, lo, kb, ks);
#pragma unroll
                    for (int qb = 0; qb < 2; ++qb) {
                        f32x16 z;
#pragma unroll
                        for (int i = 0; i < 16; ++i) z[i] = 0.0f;
                        s[kb][qb] = mfma_bf16(akf, qf[qb][ks], ks == 0 ? z : s[kb][qb]);
                    }
                }
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) {
                float mx0 = s[0][qb][0], mx1 = s[1][qb][0];
#pragma unroll
                for (int i = 1; i < 16; ++i) { mx0 = fast_max(mx0, s[0][qb][i]); mx1 = fast_max(mx1, s[1][qb][i]); }
                m[qb] = fast_max(m[qb], xhalf_max(fast_max(mx0, mx1)) * c);
            }
        }
    }
    float nm[2] = {-m[0], -m[1]};

    if (pipelined) {
#define GPTOSS_FP_FENCE() __builtin_amdgcn_sched_barrier(0)
        // (an MFMA's result is not needed before the next slot, and instruction selection would place it there,
        // across the fences, which only bind the scheduler that runs afterwards: an empty volatile statement
        // that takes the result as an operand keeps the MFMA inside its micro-slot)
#define GPTOSS_FP_PIN(x) asm volatile("" : "+v"(x))
        // ---- pipeline state ----
        f32x16 sa, sb;                      // logits of the unit in the softmax / of the unit being multiplied
        bf16x8 pa[2], pb[2];                // [u16] P of the unit in the softmax / of the unit before it
        bf16x8 ak[4];                       // [ks] K fragments of the key block whose S is being formed
        bf16x8 av[2][2];                    // [u16][dblk] V fragments of the key block being multiplied into O
        uint32_t kadr[4], vadr[2][2];       // per-lane LDS addresses: K of the stage the next K fragments come from, V of this tile's
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) kadr[ks] = smem_base + (DOCS ? (k_a & (NS - 1)) * SB : 0) + lo.nat[ks];    // tile 0 of the walk is in stage 0
#pragma unroll
        for (int dblk = 0; dblk < 2; ++dblk)
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2) vadr[dblk][t2] = smem_base + (DOCS ? (k_a & (NS - 1)) * SB : 0) + kStageTileBytes + lo.tr[dblk][t2];
        // fill: S of unit 0 of the first tile; the first slot's O MFMAs multiply zeros (exact: O keeps its bits)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) ak[ks] = as_bf16x8(lds_load128(kadr[ks], 0));
#pragma unroll
        for (int u16 = 0; u16 < 2; ++u16) {
#pragma unroll
            for (int e = 0; e < 8; ++e) { pb[u16][e] = (bf16)0.0f; av[u16][0][e] = (bf16)0.0f; av[u16][1][e] = (bf16)0.0f; }
        }
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            f32x16 z;
#pragma unroll
            for (int i = 0; i < 16; ++i) z[i] = 0.0f;
            sa = mfma_bf16(ak[ks], qf[0][ks], ks == 0 ? z : sa);
        }
        GPTOSS_FP_FENCE();

        // slot U of a tile: softmax of unit U (logits s_cur -> P pf_cur), S of unit U + 1 (-> s_next), O += P V of unit U - 1 (pf_prev)
        auto slot = [&](auto u_, f32x16 &s_cur, f32x16 &s_next, bf16x8 (&pf_prev)[2], bf16x8 (&pf_cur)[2]) __attribute__((always_inline)) {
            constexpr int U = decltype(u_)::value;
            constexpr int qb = U & 1, qo = qb ^ 1;            // the units before and after U are of the other row block
            constexpr bool RELOAD = (U & 1) == 0;             // they are the last users of the fragments in registers
            float rs0 = 0.0f, rs1 = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int i = j >> 1;
                if ((j & 1) == 0) {
                    f32x16 z;
#pragma unroll
                    for (int e = 0; e < 16; ++e) z[e] = 0.0f;
                    s_next = mfma_bf16(ak[i], qf[qo][i], i == 0 ? z : s_next);
                    GPTOSS_FP_PIN(s_next);
                    // U == 0: key block 1 of this tile; U == 2: key block 0 of the next one (kadr is there already)
                    if (RELOAD) ak[i] = as_bf16x8(lds_load128(kadr[i], U == 0 ? 32 * kRowBytes : 0));
                } else {
                    const int u16 = i >> 1, dblk = i & 1;
                    o[qo][dblk] = mfma_bf16(av[u16][dblk], pf_prev[u16], o[qo][dblk]);
                    GPTOSS_FP_PIN(o[qo][dblk]);
                    if (RELOAD) {                             // the V fragments of unit U's own key block
                        const int imm = (32 * (U >> 1) + 16 * u16) * kRowBytes;
                        union { struct { s16x4 a, b; } s; bf16x8 v; } x;
                        x.s.a = lds_load_tr64(vadr[dblk][0], imm);
                        x.s.b = lds_load_tr64(vadr[dblk][1], imm);
                        av[u16][dblk] = x.v;
                    }
                }
                const float e0 = fast_exp2(fmaf(s_cur[2 * j], c, nm[qb])), e1 = fast_exp2(fmaf(s_cur[2 * j + 1], c, nm[qb]));
                rs0 += e0;
                rs1 += e1;
                pf_cur[j >> 2][(2 * j) & 7] = (bf16)e0;
                pf_cur[j >> 2][((2 * j) & 7) + 1] = (bf16)e1;
                GPTOSS_FP_FENCE();
            }
            l[qb] += rs0 + rs1;
        };
        using I0 = std::integral_constant<int, 0>; using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>; using I3 = std::integral_constant<int, 3>;

        // (whatever loads the compiler itself has in flight here, reloads of spilled registers included, are
        // known to have arrived after this wait, so it puts no vmcnt wait of its own into the loop, where it
        // would also wait for the copies in flight)
        // (the Q fragments, which the first tile's exact step pushes out to scratch, are asked for here so that
        // their reloads come before the wait rather than after it)
#pragma unroll
        for (int qb = 0; qb < 2; ++qb)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) asm volatile("" ::"v"(qf[qb][ks]));
        wait_vmcnt<0>();
        const int k_end = GENERAL ? t_b - t_lo : n_it - 1;
        for (int t = DOCS ? k_a : 0; t < k_end; ++t) {
            GPTOSS_FP_FENCE();
            slot(I0{}, sa, sb, pb, pa);
            slot(I1{}, sb, sa, pa, pb);
            // the next tile has landed; its first K fragments are loaded in the slot that follows, its V fragments
            // from the next pass of this loop on
            arrive();
            const uint32_t step = ((t + 1) & (NS - 1)) ? (uint32_t)SB : (uint32_t)(SB - NS * SB);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) kadr[ks] += step;
            GPTOSS_FP_FENCE();
            slot(I2{}, sa, sb, pb, pa);
            slot(I3{}, sb, sa, pa, pb);
#pragma unroll
            for (int dblk = 0; dblk < 2; ++dblk)
#pragma unroll
                for (int t2 = 0; t2 < 2; ++t2) vadr[dblk][t2] += step;
        }
        // drain: O += P V of the last pipelined tile's last unit (sa holds S of the diagonal tile's first unit,
        // which the masked tile function below forms again with the mask)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int u16 = i >> 1, dblk = i & 1;
            o[1][dblk] = mfma_bf16(av[u16][dblk], pb[u16], o[1][dblk]);
        }
        GPTOSS_FP_FENCE();
#undef GPTOSS_FP_FENCE
#undef GPTOSS_FP_PIN
    }
    const int lane_b = fresh_lane(), l32_b = lane_b & 31, half_b = lane_b >> 5;
    const TileLaneOffsets lo_b = make_tile_offsets(lane_b);
    int pq_b[2];
    unsigned wl_b[2];
    describe_rows(l32_b, pq_b, wl_b);
    auto masked_args_b = [&](int n0, int (&dbase)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) dbase[qb] = pq_b[qb] - n0;
    };
    // rows that do not exist: nothing attended, whatever the interior tiles made of them
    auto clear_rows = [&](int qb, bool dead_row) __attribute__((always_inline)) {
        m[qb] = dead_row ? m_first : m[qb];
        l[qb] = dead_row ? 0.0f : l[qb];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            o[qb][0][i] = dead_row ? 0.0f : o[qb][0][i];
            o[qb][1][i] = dead_row ? 0.0f : o[qb][1][i];
        }
    };
    // A sum beyond 2^96 (or not finite): some logit stood 95 or more above its row's frozen reference; the
    // workgroup repeats its key loop with the exact online-softmax step on every tile (see attn_fwd_kernel; the
    // masked form of the step for every tile: this pass is rare and the kernel stays small).
    auto frozen_too_low = [&]() __attribute__((always_inline)) {
        bool unsafe = false;
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) unsafe = unsafe || !(l[qb] < 0x1p96f);
        return __syncthreads_or(unsafe);
    };
    auto exact_tile = [&](int it) __attribute__((always_inline)) {
        const uint32_t ksm = smem_base + (it & (NS - 1)) * SB;
        int dbase[2];
        const int n0 = (t_lo + it) * kTile;
        masked_args_b(n0, dbase);
        fwd_tile<true, 2>(ksm, ksm + kStageTileBytes, lo_b, qf, o, m, l, c, lane_b, dbase, wl_b, 0x3fffffffu, kv_len - n0, q_offset + qw0 - n0);
    };
    auto lean_tile = [&](int it) __attribute__((always_inline)) {
        const uint32_t ksm = smem_base + (it & (NS - 1)) * SB;
        int dbase[2];
        const int n0 = (t_lo + it) * kTile;
        masked_args_b(n0, dbase);
        fwd_tile_lean<true, 2>(ksm, ksm + kStageTileBytes, lo_b, qf, o, nm, l, c, lane_b, dbase, wl_b, 0x3fffffffu, kv_len - n0, GENERAL ? q_offset + qw0 - n0 : 0);
    };
    if constexpr (!DOCS) {
        if (pipelined) {
            // (the first of these tiles has landed: the pipeline's last pass waited for it)
            if constexpr (GENERAL) {
#pragma unroll 1
                for (int it = t_b - t_lo; it < n_it; ++it) {
                    if (it > t_b - t_lo) arrive();
                    fetch_end(it);
                    lean_tile(it);
                }
#pragma unroll
                for (int qb = 0; qb < 2; ++qb) clear_rows(qb, pq_b[qb] < 0);
            } else {
                lean_tile(qt);
            }
        }
        // (rows of a single tile take this pass as their only one)
        const bool second_pass = pipelined && frozen_too_low();
        if (second_pass || (!pipelined && n_it > 0)) {
            if (second_pass) {
                wait_vmcnt<0>();      // the repeated copies of the last requests
                __syncthreads();
            }
            reset();
            for (int it = 0; it < n_it; ++it) {
                arrive();
                fetch_end(it);
                exact_tile(it);
            }
            if (GENERAL)
#pragma unroll
                for (int qb = 0; qb < 2; ++qb) clear_rows(qb, pq_b[qb] < 0);
        }
    } else {
        // With an interior tile in front, a row that cannot see tile t_a sees nothing in front of the diagonal tile: it starts
        // afresh here, and needs a reference of its own, so the workgroup's last tiles take the exact step.  Otherwise the
        // reference stays frozen.
        bool fresh = false;
        if (pipelined) {
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) {
                const bool late = pq_b[qb] - (int)wl_b[qb] + 1 > t_a * kTile;
                fresh = fresh || late;
                clear_rows(qb, pq_b[qb] < 0 || late);
            }
        }
        bool lean = pipelined && __builtin_amdgcn_ballot_w64(fresh) == 0ull;
        int k_exact = pipelined ? t_b - t_lo : 0;
        bool landed = pipelined;      // the pipeline's last pass waited for the tile that comes next
        bool repeat = pipelined;      // the reference was frozen: the sums have to be looked at
        if (!pipelined && n_it > 0) reset();
#pragma unroll 1
        for (;;) {
#pragma unroll 1
            for (int it = k_exact; it < n_it; ++it) {
                if (!landed) arrive();
                landed = false;
                fetch_end(it);
                if (lean) lean_tile(it); else exact_tile(it);
            }
            if (!repeat) break;
            repeat = false;
            lean = false;
#pragma unroll
            for (int qb = 0; qb < 2; ++qb) clear_rows(qb, pq_b[qb] < 0);
            if (!frozen_too_low()) break;
            wait_vmcnt<0>();          // the repeated copies of the last requests
            __syncthreads();
            reset();
            k_exact = 0;
            landed = false;
        }
        // (rows that do not exist and met only masked tiles end as they began: nothing attended)
    }

    // epilogue: z = l + exp(sink - m); O = acc / z; M = m + log z   (ref :93-98)
    wait_vmcnt<0>();              // the repeated copies of the last requests
    __syncthreads();
    bf16 *stage = reinterpret_cast<bf16 *>(&smem[0][0][0]) + w * 32 * kLS;
#pragma unroll
    for (int qb = 0; qb < 2; ++qb) {
        const float l_tot = l[qb] + __shfl_xor(l[qb], 32);
        if constexpr (GENERAL && !DOCS) {
            if (a.kv_splits > 1) {
                // this share's unnormalised rows and their (reference, sum); lane = row, four consecutive columns per store
                const int row = qw0 + 32 * qb + l32_b;
                if (row < a.Sq) {
                    const int64_t rows = (int64_t)a.B * a.H * a.Sq, rid = ((int64_t)b * a.H + head) * a.Sq + row;
                    float *part = a.fwd_partial + ((int64_t)split * rows + rid) * kD;
#pragma unroll
                    for (int dblk = 0; dblk < 2; ++dblk)
#pragma unroll
                        for (int a4 = 0; a4 < 4; ++a4)
                            *reinterpret_cast<f32x4 *>(part + 32 * dblk + 8 * a4 + 4 * half_b) =
                                f32x4{o[qb][dblk][4 * a4], o[qb][dblk][4 * a4 + 1], o[qb][dblk][4 * a4 + 2], o[qb][dblk][4 * a4 + 3]};
                    if (half_b == 0) {
                        float *ml = a.fwd_partial + (int64_t)a.kv_splits * rows * kD + 2 * ((int64_t)split * rows + rid);
                        ml[0] = m[qb];
                        ml[1] = l_tot;
                    }
                }
                continue;
            }
        }
        const float z = l_tot + fast_exp2(sink2 - m[qb]);
        const float inv = 1.0f / z;
        const int r0 = qw0 + 32 * qb;
        bf16 *orow0 = a.o + (int64_t)b * a.os.b + (int64_t)head * a.os.h + (int64_t)r0 * a.os.s;
        store_rows32(stage, o[qb], inv, orow0, a.os.s, a.Sq - r0, lane_b);
        __builtin_amdgcn_wave_barrier();
        if (half_b == 0 && (!GENERAL || r0 + l32_b < a.Sq)) a.lse[((int64_t)b * a.H + head) * a.Sq + r0 + l32_b] = (m[qb] + fast_log2(z)) * kLn2;
    }
}

// The shares of a row's keys, added in their order: eight lanes per row, eight columns each.
__global__ __launch_bounds__(256) void attn_fwd_combine_kernel(const KArgs a) {
    const int64_t rows = (int64_t)a.B * a.H * a.Sq, rid = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 3);
    if (rid >= rows) return;
    const int c8 = (threadIdx.x & 7) * 8;
    const int s_ = (int)(rid % a.Sq);
    const int bh = (int)(rid / a.Sq), h = bh % a.H, b = bh / a.H;
    const float sink2 = sink_logit(a, h) * kLog2e;
    const float *ml = a.fwd_partial + (int64_t)a.kv_splits * rows * kD + 2 * rid;
    float mm = fast_max(sink2, kNoLogit);
    for (int i = 0; i < a.kv_splits; ++i) mm = fast_max(mm, ml[2 * rows * i]);
    float z = fast_exp2(sink2 - mm), acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
    for (int i = 0; i < a.kv_splits; ++i) {
        const float f = fast_exp2(ml[2 * rows * i] - mm);
        z = fmaf(f, ml[2 * rows * i + 1], z);
        const float *p = a.fwd_partial + ((int64_t)i * rows + rid) * kD + c8;
        const f32x4 x = *reinterpret_cast<const f32x4 *>(p), y = *reinterpret_cast<const f32x4 *>(p + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { acc[e] = fmaf(f, x[e], acc[e]); acc[4 + e] = fmaf(f, y[e], acc[4 + e]); }
    }
    const float inv = 1.0f / z;
    union { bf16x8 v; u32x4 u; } out;
#pragma unroll
    for (int e = 0; e < 8; ++e) out.v[e] = (bf16)(acc[e] * inv);
    *reinterpret_cast<u32x4 *>(a.o + (int64_t)b * a.os.b + (int64_t)h * a.os.h + (int64_t)s_ * a.os.s + c8) = out.u;
    if (c8 == 0) a.lse[rid] = (mm + fast_log2(z)) * kLn2;
}

}  // namespace gptoss
