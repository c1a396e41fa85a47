// Forward for a handful of new queries on a long key / value cache (bf16; decoding, q_offset = the cache's length): the
// results of attn_fwd_kernel (the reference's `_attn_fwd` with `start_q`, attention_kernel.py:11-100).
//
// What bounds it: reading K and V once from HBM.  attn_fwd_kernel gives 64 rows x 4 heads of ONE query to a workgroup, so
// a decoding step is 2 G B workgroups, each walking the whole cache tile by tile, and every K / V row is staged twice.
//
// Work split.  The Sq * r (query, head of the group) pairs of a KV head are the columns of one S^T block (two for up to 64
// pairs), so K and V are read once.  The keys are cut over `kv_splits` workgroups of four wavefronts, or walked by one of eight (NW) where
// they are so few that the second launch costs more; inside a workgroup
// the wavefronts take 32-key tiles in turn, each through LDS stages of its own (no barrier in the loop, NS tiles in
// flight per wavefront), and merge their (m, l, O) at the end.  With one split the workgroup writes O and lse;
// otherwise it leaves fp32 partials in the scratch and attn_decode_combine_kernel adds them in an order that depends on
// their number only.
//
// Measured (64 query heads on 8 KV heads, one query, MI355X): B = 16 on 8192 keys 246 us with attn_fwd_kernel, 42 + 4 us
// here (268 MB: 6.3 TB/s, a plain 4 GiB copy moves 4.7); B = 1 on 2049 keys 57 us,
// 5.4 + 4.2 us here (launch latencies); on 1024 keys a call takes 12.4 us in slices and 11.1 in one launch.
#pragma once
#include "attn_common.h"

namespace gptoss {

struct Decode {
    static constexpr int kKeys = 32;                               // keys per tile
    static constexpr int kTileBytes = 2 * kKeys * kRowBytes;       // K rows, then V rows
    static constexpr int NS = 2;                                   // LDS stages per wavefront
    static constexpr int kCopies = 8;                              // copy instructions per tile
    static constexpr int kMaxPairs = 64;                           // (query, head) pairs per KV head
};
// scratch per (batch, KV head, split): the unnormalised output rows, then (m, l) per row (a multiple of 16 bytes)
__host__ __device__ inline int64_t decode_partial_floats(int pairs) { return ((int64_t)pairs * (kD + 2) + 3) & ~(int64_t)3; }

// Bytes of LDS of a workgroup of NW wavefronts: their stages, later their results.
template <int NQB, int NW>
constexpr int decode_lds_bytes() {
    constexpr int merge = NW * 32 * NQB * (kD + 2) * 4, stages = NW * Decode::NS * Decode::kTileBytes;
    return stages > merge ? stages : merge;
}

template <int NQB, int NW>
__global__ __launch_bounds__(64 * NW, 2) void attn_decode_kernel(const KArgs a) {
    using C = Decode;
    extern __shared__ __attribute__((aligned(1024))) char smem[];

    const int q_offset = query_offset(a);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    int bid = blockIdx.x;
    const int g = bid % a.G; bid /= a.G;
    const int split = bid % a.kv_splits;
    const int b = bid / a.kv_splits;
    const int pairs = a.Sq * a.r;

    const int kv_len = a.seqlens ? min(a.Skv, a.seqlens[b]) : a.Skv;
    const int q_len = a.seqlens ? a.seqlens[b] : 0x7fffffff;
    const int weff = a.window ? a.window : 0x3fffffff;
    const int pos0 = q_offset, pos1 = q_offset + a.Sq - 1;         // first and last query position
    const int hi = pos0 < q_len ? max(0, min(kv_len, min(pos1, q_len - 1) + 1)) : 0;
    const int t_first = max(0, pos0 - weff + 1) / C::kKeys;
    const int n_all = max(0, (hi + C::kKeys - 1) / C::kKeys - t_first);
    const int t_lo = t_first + (int)((int64_t)n_all * split / a.kv_splits);
    const int n_wg = t_first + (int)((int64_t)n_all * (split + 1) / a.kv_splits) - t_lo;
    const int n_it = n_wg > w ? (n_wg - w + NW - 1) / NW : 0;      // this wavefront's tiles: t_lo + w + NW j

    // columns: pair 32 qb + l32 = (query row, head of the group)
    bf16x8 qf[NQB][4];
    int pq[NQB];            // the column's query position, hugely negative where there is none
    float sink2[NQB], m[NQB], l[NQB];
    f32x16 o[NQB][2];
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {
        const int pair = 32 * qb + l32;
        const bool ok = pair < pairs;
        const int row = ok ? pair / a.r : 0, head = g * a.r + (ok ? pair % a.r : 0);
        const bf16 *qrow = a.q + (int64_t)b * a.qs.b + (int64_t)head * a.qs.h + (int64_t)row * a.qs.s;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) qf[qb][ks] = as_bf16x8(*reinterpret_cast<const u32x4 *>(qrow + 16 * ks + 8 * half));
        pq[qb] = ok && q_offset + row < q_len ? q_offset + row : -0x40000000;
        sink2[qb] = sink_logit(a, head) * kLog2e;
        m[qb] = fast_max(sink2[qb], kNoLogit);
        l[qb] = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) { o[qb][0][i] = 0.0f; o[qb][1][i] = 0.0f; }
    }
    const float c = a.scale_log2;

    // ---- the wavefront's own staging: rows past the tensor's end re-read the last one (masked below) ----
    const uint32_t stage0 = lds_addr(smem) + w * (C::NS * C::kTileBytes);
    const bf16 *kbase = a.k + (int64_t)b * a.ks.b + (int64_t)g * a.ks.h, *vbase = a.v + (int64_t)b * a.vs.b + (int64_t)g * a.vs.h;
    auto issue = [&](int j) __attribute__((always_inline)) {
        const int n0 = (t_lo + w + NW * j) * C::kKeys;
        const uint32_t dst = stage0 + (j % C::NS) * C::kTileBytes;
        const bf16 *kt = kbase + (int64_t)n0 * a.ks.s, *vt = vbase + (int64_t)n0 * a.vs.s;
        const int last = a.Skv - 1 - n0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int r = 8 * k + (lane >> 3), ch = ((lane & 7) ^ swz(r)) * 16, rr = min(r, last);
            lds_dma16(dst + k * 8 * kRowBytes, kt, (uint32_t)(rr * (int)a.ks.s) * 2u + ch);
            lds_dma16(dst + (C::kKeys + k * 8) * kRowBytes, vt, (uint32_t)(rr * (int)a.vs.s) * 2u + ch);
        }
    };
    const TileLaneOffsets lo = make_tile_offsets(lane);
#pragma unroll
    for (int j = 0; j < C::NS - 1; ++j)
        if (j < n_it) issue(j);
    for (int j = 0; j < n_it; ++j) {
        if (j + C::NS - 1 < n_it) {
            // (every LDS read of the stage's last tile has been consumed: nothing of it is outstanding)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            issue(j + C::NS - 1);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(C::kCopies * (C::NS - 1)) : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        const int n0 = (t_lo + w + NW * j) * C::kKeys;
        const uint32_t ksm = stage0 + (j % C::NS) * C::kTileBytes, vsm = ksm + C::kKeys * kRowBytes;
        const bool interior = n0 + C::kKeys - 1 <= pos0 && n0 > pos1 - weff && n0 + C::kKeys <= kv_len && pos1 < q_len;
        f32x16 s[NQB];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const bf16x8 ak = ofrag_nat(ksm, lo, 0, ks);
#pragma unroll
            for (int qb = 0; qb < NQB; ++qb) {
                f32x16 z;
#pragma unroll
                for (int i = 0; i < 16; ++i) z[i] = 0.0f;
                s[qb] = mfma_bf16(ak, qf[qb][ks], ks == 0 ? z : s[qb]);
            }
        }
#pragma unroll
        for (int qb = 0; qb < NQB; ++qb) {
            if (!interior) {
                const KeyMask km = make_key_mask(pq[qb] - n0, (unsigned)weff, kv_len - n0, half);
#pragma unroll
                for (int i = 0; i < 16; ++i) s[qb][i] = key_visible(km, 8 * (i >> 2) + (i & 3)) ? s[qb][i] : -INFINITY;
            }
            float mx0 = s[qb][0], mx1 = s[qb][1];
#pragma unroll
            for (int i = 2; i < 16; i += 2) { mx0 = fast_max(mx0, s[qb][i]); mx1 = fast_max(mx1, s[qb][i + 1]); }
            const float m_new = fast_max(m[qb], xhalf_max(fast_max(mx0, mx1)) * c);
            if (__builtin_amdgcn_ballot_w64(m_new != m[qb]) != 0ull) {
                const float alpha = fast_exp2(m[qb] - m_new);
                l[qb] *= alpha;
#pragma unroll
                for (int i = 0; i < 16; ++i) { o[qb][0][i] *= alpha; o[qb][1][i] *= alpha; }
                m[qb] = m_new;
            }
            float rs0 = 0.0f, rs1 = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                const float e0 = fast_exp2(fmaf(s[qb][i], c, -m[qb])), e1 = fast_exp2(fmaf(s[qb][i + 1], c, -m[qb]));
                s[qb][i] = e0;
                s[qb][i + 1] = e1;
                rs0 += e0;
                rs1 += e1;
            }
            l[qb] += rs0 + rs1;
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int dblk = 0; dblk < 2; ++dblk) {
                const bf16x8 av = ofrag_tr(vsm, lo, 0, u, dblk);
#pragma unroll
                for (int qb = 0; qb < NQB; ++qb) o[qb][dblk] = mfma_bf16(av, cfrag(s[qb], u), o[qb][dblk]);
            }
    }

    // ---- merge the wavefronts: rows [wavefront][pair][64 + (m, l)] in LDS ----
    __syncthreads();
    constexpr int kRow = kD + 2, kWave = 32 * NQB * kRow;
    float *red = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int qb = 0; qb < NQB; ++qb) {
        const float l_tot = xhalf_sum(l[qb]);
        float *row = red + w * kWave + (32 * qb + l32) * kRow;
#pragma unroll
        for (int dblk = 0; dblk < 2; ++dblk)
#pragma unroll
            for (int i = 0; i < 16; ++i) row[32 * dblk + crow(i, half)] = o[qb][dblk][i];
        if (half == 0) { row[kD] = m[qb]; row[kD + 1] = l_tot; }
    }
    __syncthreads();
    // eight lanes per row, eight columns each
    const int c8 = (tid & 7) * 8;
    for (int pair = tid >> 3; pair < pairs; pair += 8 * NW) {
        float mw[NW], lw = 0.0f, acc[8], mm;
#pragma unroll
        for (int k = 0; k < NW; ++k) mw[k] = red[k * kWave + pair * kRow + kD];
        mm = mw[0];
#pragma unroll
        for (int k = 1; k < NW; ++k) mm = fast_max(mm, mw[k]);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            const float f = fast_exp2(mw[k] - mm);
            const float *row = red + k * kWave + pair * kRow;
            lw += f * row[kD + 1];
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] += f * row[c8 + e];
        }
        if (a.kv_splits > 1) {
            float *part = a.fwd_partial + (((int64_t)b * a.G + g) * a.kv_splits + split) * decode_partial_floats(pairs);
            float *row = part + pair * kD + c8;
            *reinterpret_cast<f32x4 *>(row) = f32x4{acc[0], acc[1], acc[2], acc[3]};
            *reinterpret_cast<f32x4 *>(row + 4) = f32x4{acc[4], acc[5], acc[6], acc[7]};
            if (c8 == 0) { part[pairs * kD + 2 * pair] = mm; part[pairs * kD + 2 * pair + 1] = lw; }
        } else {
            const int row = pair / a.r, head = g * a.r + pair % a.r;
            const float z = lw + fast_exp2(sink_logit(a, head) * kLog2e - mm), inv = 1.0f / z;
            union { bf16x8 v; u32x4 u; } out;
#pragma unroll
            for (int e = 0; e < 8; ++e) out.v[e] = (bf16)(acc[e] * inv);
            *reinterpret_cast<u32x4 *>(a.o + (int64_t)b * a.os.b + (int64_t)head * a.os.h + (int64_t)row * a.os.s + c8) = out.u;
            if (c8 == 0) a.lse[((int64_t)b * a.H + head) * a.Sq + row] = (mm + fast_log2(z)) * kLn2;
        }
    }
}

// The splits' partials of one (batch, KV head, pair) row, one wavefront per row: lane = (group of splits, 8 columns).  The
// order of the additions depends on the number of splits only.
__global__ __launch_bounds__(256) void attn_decode_combine_kernel(const KArgs a) {
    const int pairs = a.Sq * a.r, lane = threadIdx.x & 63;
    const int64_t idx = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (idx >= (int64_t)a.B * a.G * pairs) return;
    const int c8 = (lane & 7) * 8, sg = lane >> 3;
    const int pair = (int)(idx % pairs);
    const int bg = (int)(idx / pairs), g = bg % a.G, b = bg / a.G;
    const int row = pair / a.r, head = g * a.r + pair % a.r;
    const int64_t step = decode_partial_floats(pairs);
    const float *part = a.fwd_partial + (int64_t)bg * a.kv_splits * step;
    const float sink2 = sink_logit(a, head) * kLog2e;
    float mm = fast_max(sink2, kNoLogit), z = 0.0f, acc[8];         // mm: the largest reference among this lane's splits so far
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.0f;
    for (int s = sg; s < a.kv_splits; s += 8) {
        const float *p = part + s * step;
        const float ms = p[pairs * kD + 2 * pair], ls = p[pairs * kD + 2 * pair + 1];
        const f32x4 x = *reinterpret_cast<const f32x4 *>(p + pair * kD + c8), y = *reinterpret_cast<const f32x4 *>(p + pair * kD + c8 + 4);
        const float mn = fast_max(mm, ms), fo = fast_exp2(mm - mn), f = fast_exp2(ms - mn);
        z = z * fo + f * ls;
#pragma unroll
        for (int e = 0; e < 4; ++e) { acc[e] = acc[e] * fo + f * x[e]; acc[4 + e] = acc[4 + e] * fo + f * y[e]; }
        mm = mn;
    }
    float mt = mm;
    mt = fast_max(mt, __shfl_xor(mt, 8));
    mt = fast_max(mt, __shfl_xor(mt, 16));
    mt = fast_max(mt, __shfl_xor(mt, 32));
    const float f = fast_exp2(mm - mt);
    z *= f;
    z += __shfl_xor(z, 8); z += __shfl_xor(z, 16); z += __shfl_xor(z, 32);
    z += fast_exp2(sink2 - mt);
    const float inv = 1.0f / z;
    union { bf16x8 v; u32x4 u; } out;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float x = acc[e] * f;
        x += __shfl_xor(x, 8); x += __shfl_xor(x, 16); x += __shfl_xor(x, 32);
        out.v[e] = (bf16)(x * inv);
    }
    if (sg == 0) {
        *reinterpret_cast<u32x4 *>(a.o + (int64_t)b * a.os.b + (int64_t)head * a.os.h + (int64_t)row * a.os.s + c8) = out.u;
        if (c8 == 0) a.lse[((int64_t)b * a.H + head) * a.Sq + row] = (mt + fast_log2(z)) * kLn2;
    }
}

}  // namespace gptoss
