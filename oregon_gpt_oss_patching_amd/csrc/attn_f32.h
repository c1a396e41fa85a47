// float32 kernels (dtype GPTOSS_ATTN_FP32): the same forward / backward as the bf16 kernels
// for callers that keep the model in float32 (the reference runs such tensors natively,
// attention_kernel.py:11-217 are dtype-generic).  Larger problems take the kernels of attn_f32_split.h, which come here for the numbers they
// do not hold; the rest starts here.  Every product runs on the fp32 matrix instruction
// v_mfma_f32_32x32x2_f32 with fp32 operands and fp32 accumulation.
//
// What bounds them: that instruction takes 64 cycles for 4096 FLOP (157 TFLOP/s on the chip), sixteen times the bf16
// instruction's price, so LDS traffic, L2 traffic and vector work are small beside it, and what matters is that every SIMD
// always has a wavefront with its operands at hand.  A wavefront stages its tiles (32 rows of two tensors, 16 KB) in LDS of
// its own, without a barrier in the loop; each tensor's half is requested again as soon as its last product has read it, so a
// request has the time of at least one product to arrive.  A workgroup is four wavefronts, two workgroups share a
// compute unit, and wavefronts that work on the same rows (KS of them in the forward and dQ, all four in dK/dV) take
// the tiles these rows meet in turn and add their partial results at the end: a row block of S = 1024 is then 8 or 16
// steps long instead of 32, and the chip fills from a few hundred rows on.
//
// Measured (64 query heads on 8 KV heads, S = 1024, full causal; before, with operands straight from global memory, one
// wavefront per row block and none sharing it): forward 200 -> 101 us (85 TFLOP/s), dQ with the row statistics 306 -> 134
// us, dK/dV 2227 -> 176 us (its 256 key blocks were 256 wavefronts).  The matrix pipes are busy 59 % (forward), 65 % (dQ) and 67 %
// (dK/dV) of the cycles there, 73 to 81 % at S = 4096 (2.2 GHz).
//
// Weights come from exp2f, not from the bare exponential instruction (fast_exp2), which flushes what is below 2^-126: a key far down
// the softmax still counts where the others' values are small or zero.  S = 1024, with the bare instruction and so: forward 97 and
// 101 us, dQ 131 and 134, dK/dV 180 and 176, a whole call 410 and 414.
//
// Register layouts of v_mfma_f32_32x32x2_f32 (lane = 0..63, half = lane/32, l32 = lane%32):
//   A (32 x 2): lane holds A[l32][half]      B (2 x 32): lane holds B[half][l32]
//   C (32 x 32): register i holds C[crow(i, half)][l32]   (as for the bf16 instruction)
// A contraction over head_dim takes 32 such steps; step ks uses d = 32*half + ks, so a lane
// reads 32 CONSECUTIVE floats of its row.  A contraction over the 32 rows held in C registers
// takes 16 steps: step (a4, e) multiplies C register 4*a4 + e, whose row is 8*a4 + 4*half + e,
// by the matching row of the other operand -- C registers are fed back as the B operand
// without any data movement.
#pragma once
#include "attn_bwd.h"
#include "attn_common.h"

namespace gptoss {

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, const f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

struct F32Ptrs {
    const float *q, *k, *v, *d_o, *o_in;
    float *o, *dq, *dk, *dv;
};
__device__ __forceinline__ F32Ptrs f32_ptrs(const KArgs &a) {
    F32Ptrs p;
    p.q = reinterpret_cast<const float *>(a.q);
    p.k = reinterpret_cast<const float *>(a.k);
    p.v = reinterpret_cast<const float *>(a.v);
    p.d_o = reinterpret_cast<const float *>(a.d_o);
    p.o_in = reinterpret_cast<const float *>(a.o);
    p.o = reinterpret_cast<float *>(a.o);
    p.dq = reinterpret_cast<float *>(a.dq);
    p.dk = reinterpret_cast<float *>(a.dk);
    p.dv = reinterpret_cast<float *>(a.dv);
    return p;
}

// 32 consecutive floats starting at p (16-byte aligned) into r[0..31]; zero when !valid.
__device__ __forceinline__ void load_row32(float (&r)[32], const float *p, bool valid) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
        if (valid) z = *reinterpret_cast<const f32x4 *>(p + 4 * j);
#pragma unroll
        for (int e = 0; e < 4; ++e) r[4 * j + e] = z[e];
    }
}

// ---- LDS tiles of 32 rows x 64 floats ---------------------------------------------------------------------
// Rows are 256 bytes (all banks once), so the sixteen 16-byte chunks of a row are XOR-swizzled with the row number:
// physical chunk p of row r holds logical chunk p ^ (r & 15).  Sixteen rows reading one logical chunk (natural 128-bit
// fragment reads) then hit sixteen different bank groups.
struct F32Tile {
    static constexpr int kRows = 32, kRowBytes = 256, kBytes = kRows * kRowBytes, kCopies = 8;
};
// requests the tile whose first row is `tile` (kCopies instructions of this wavefront); rows past `last` re-read that one
__device__ __forceinline__ void f32_copy_tile(uint32_t lds_tile, const float *tile, int stride, int last, int lane) {
#pragma unroll
    for (int i = 0; i < F32Tile::kCopies; ++i) {
        const int r = 4 * i + (lane >> 4), ch = (lane & 15) ^ (r & 15);
        lds_dma16(lds_tile + i * 1024, tile, (uint32_t)(min(r, last) * stride) * 4u + ch * 16);
    }
}
// at most n of this wavefront's copies outstanding, and no LDS access moved across
#define GPTOSS_F32_WAIT(n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory")
// every LDS read issued so far has its data: the tile it came from may be overwritten
#define GPTOSS_F32_READS_DONE() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")
struct F32Offsets {
    uint32_t nat;      // natural fragment: row l32, logical chunk 8 * half; chunk j of it is at nat ^ (j << 4)
    uint32_t tr[4];    // [e]: element (row 4 * half + e, column l32); (row + 8 a4, column + 32 dblk) by immediates
};
__device__ __forceinline__ F32Offsets make_f32_offsets(int lane) {
    F32Offsets o;
    const int l32 = lane & 31, half = lane >> 5;
    o.nat = l32 * F32Tile::kRowBytes + (((8 * half) ^ (l32 & 15)) << 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) o.tr[e] = (4 * half + e) * F32Tile::kRowBytes + (((l32 >> 2) ^ (4 * half + e)) << 4) + (l32 & 3) * 4;
    return o;
}
__device__ __forceinline__ f32x4 f32_nat(uint32_t tile, const F32Offsets &o, int j) { return lds_load128f(tile + (o.nat ^ (j << 4)), 0); }
// (bit 3 of the chunk index is 0 in tr[e]: XOR with 8 adds 128 bytes)
__device__ __forceinline__ float f32_tr(uint32_t tile, const F32Offsets &o, int a4, int e, int dblk) {
    typedef __attribute__((address_space(3))) float lds_f32;
    return *reinterpret_cast<const lds_f32 *>((uintptr_t)(tile + o.tr[e] + 8 * a4 * F32Tile::kRowBytes + ((dblk ^ (a4 & 1)) << 7)));
}
// The operands of the next few MFMAs are read from LDS while the current ones run (an MFMA takes 64 cycles; read, wait,
// multiply one by one, which is what the compiler makes of the plain loops, doubles a tile's time).
#define GPTOSS_F32_FENCE() __builtin_amdgcn_sched_barrier(0)
// s += X Y^T over head_dim: X's rows from the tile (result rows), y[] the lane's row of Y (result columns)
__device__ __forceinline__ void f32_rows_product(f32x16 &s, uint32_t tile, const F32Offsets &o, const float (&y)[32]) {
    f32x4 x = f32_nat(tile, o, 0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        f32x4 next = x;
        if (j < 7) next = f32_nat(tile, o, j + 1);
        GPTOSS_F32_FENCE();
#pragma unroll
        for (int e = 0; e < 4; ++e) s = mfma_f32(x[e], y[4 * j + e], s);
        GPTOSS_F32_FENCE();
        x = next;
    }
}
// acc^T[d][col] += tile^T[d][row] p[row][col] over the tile's 32 rows (p in C registers)
__device__ __forceinline__ void f32_cols_product(f32x16 (&acc)[2], uint32_t tile, const F32Offsets &o, const f32x16 &p) {
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = f32_tr(tile, o, 0, e >> 1, e & 1);
#pragma unroll
    for (int a4 = 0; a4 < 4; ++a4) {
        float next[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) next[e] = a4 < 3 ? f32_tr(tile, o, a4 + 1, e >> 1, e & 1) : 0.0f;
        GPTOSS_F32_FENCE();
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e & 1] = mfma_f32(x[e], p[4 * a4 + (e >> 1)], acc[e & 1]);
        GPTOSS_F32_FENCE();
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = next[e];
    }
}

// Where a wavefront of the forward / dQ kernels stands: 32 query rows of one head (a unit; 4 / KS units per workgroup) and
// every KS-th of the 32-key tiles they see.
struct F32Unit { int head, b, q0; bool live; };
template <int KS, int NW = 4>
struct F32QueryWork {
    int g, b, head, q0, q_len, kv_len, weff, pos0, pos1, ds1, t_lo, n, t0, n_it, w, lane;
    const float *kbase, *vbase;
    uint32_t ksm, vsm;         // this wavefront's K and V tile in LDS
    // unit i of the workgroup: KV head fastest (its K / V stay in one XCD's L2), then the heads of the group, longest key loops first
    static __device__ __forceinline__ F32Unit unit(const KArgs &a, int i) {
        F32Unit u;
        constexpr bool kSome = NW == 8;        // attn_f32_split.h: some of the batch rows and KV heads
        const int G = kSome ? a.split_ng : a.G, B = kSome ? a.split_nb : a.B;
        const int g = (int)(blockIdx.x % G) + (kSome ? a.split_g0 : 0);
        int n = (int)(blockIdx.x / G) * (NW / KS) + i;
        u.head = g * a.r + n % a.r; n /= a.r;
        const int bi = n % B, z = n / B, n_q = (a.Sq + 31) / 32;
        u.b = rotated_batch_row(bi, z, B) + (kSome ? a.split_b0 : 0);
        u.live = z < n_q;
        u.q0 = 32 * max(n_q - 1 - z, 0);
        return u;
    }
    __device__ __forceinline__ F32QueryWork(const KArgs &a, const F32Ptrs &t, int q_offset, char *lds) {
        lane = threadIdx.x & 63;
        w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        ksm = lds_addr(lds) + w * (2 * F32Tile::kBytes);
        vsm = ksm + F32Tile::kBytes;
        const F32Unit u = unit(a, w / KS);
        b = u.b; head = u.head; q0 = u.q0; g = head / a.r;
        kv_len = a.seqlens ? min(a.Skv, a.seqlens[b]) : a.Skv;
        q_len = a.seqlens ? a.seqlens[b] : 0x7fffffff;
        weff = a.window ? a.window : 0x3fffffff;
        pos0 = q_offset + q0;
        pos1 = min(q_offset + min(a.Sq, q0 + 32) - 1, q_len - 1);
        const int32_t *dsrow = a.doc_start ? a.doc_start + (int64_t)b * a.Sq : nullptr;
        const int ds0 = dsrow ? dsrow[min(q0, a.Sq - 1)] : 0;
        ds1 = dsrow ? dsrow[min(q0 + 31, a.Sq - 1)] : 0;
        const int hi = pos1 >= pos0 && u.live ? max(0, min(kv_len, pos1 + 1)) : 0;
        t_lo = max(max(0, pos0 - weff + 1), ds0) / F32Tile::kRows;
        n = max(0, (hi + F32Tile::kRows - 1) / F32Tile::kRows - t_lo);
        t0 = t_lo + w % KS;
        n_it = (n - w % KS + KS - 1) / KS;               // tiles t0 + KS it  (0 if n <= w % KS)
        kbase = t.k + (int64_t)b * a.ks.b + (int64_t)g * a.ks.h;
        vbase = t.v + (int64_t)b * a.vs.b + (int64_t)g * a.vs.h;
    }
    __device__ __forceinline__ int first_key(int it) const { return (t0 + KS * it) * F32Tile::kRows; }
    __device__ __forceinline__ void request_k(const KArgs &a, int it) const {
        const int n0 = first_key(it);
        f32_copy_tile(ksm, kbase + (int64_t)n0 * a.ks.s, (int)a.ks.s, a.Skv - 1 - n0, lane);
    }
    __device__ __forceinline__ void request_v(const KArgs &a, int it) const {
        const int n0 = first_key(it);
        f32_copy_tile(vsm, vbase + (int64_t)n0 * a.vs.s, (int)a.vs.s, a.Skv - 1 - n0, lane);
    }
    __device__ __forceinline__ bool interior(const KArgs &a, int n0) const {
        return n0 + 31 <= pos0 && n0 > pos1 - weff && n0 + 32 <= kv_len && pos0 + 31 <= pos1 && n0 >= ds1;
    }
    // the lane's query position (hugely negative: no such row) and its own window (packed rows: back to its document's start)
    __device__ __forceinline__ void row_info(const KArgs &a, int q_offset, int row, int &pos, unsigned &win) const {
        const int p = q_offset + row;
        pos = row < a.Sq && p < q_len ? p : -0x40000000;
        win = (unsigned)weff;
        if (a.doc_start && row < a.Sq) win = (unsigned)min(weff, p - a.doc_start[(int64_t)b * a.Sq + row] + 1);
    }
};

// Partial results of the four wavefronts through LDS: a wavefront leaves its transposed 64 x 32 accumulators as 32 rows of 64
// floats, chunks swizzled like a tile's ...
__device__ __forceinline__ void f32_leave_partial(char *mine, const f32x16 (&acc)[2], int lane) {
    const int l32 = lane & 31, half = lane >> 5;
#pragma unroll
    for (int dblk = 0; dblk < 2; ++dblk)
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4)
            *reinterpret_cast<f32x4 *>(mine + l32 * F32Tile::kRowBytes + (((8 * dblk + 2 * a4 + half) ^ (l32 & 15)) << 4)) =
                f32x4{acc[dblk][4 * a4], acc[dblk][4 * a4 + 1], acc[dblk][4 * a4 + 2], acc[dblk][4 * a4 + 3]};
}
// ... and a thread picks up its 16-byte chunk `ch` of row r of wavefront k's
__device__ __forceinline__ f32x4 f32_partial(const char *smem, int wave_bytes, int k, int r, int ch) {
    return *reinterpret_cast<const f32x4 *>(smem + k * wave_bytes + r * F32Tile::kRowBytes + ((ch ^ (r & 15)) << 4));
}

// ---- forward ------------------------------------------------------------------------
// (the merge of the wavefronts' shares: m, l and O of each in its own registers)
template <int KS, int NW>
__device__ __forceinline__ void f32_fwd_merge(const KArgs &a, const F32Ptrs &t, char *smem, int w, int lane, float m, float l, const f32x16 (&o)[2]) {
    using W = F32QueryWork<KS, NW>;
    const int l32 = lane & 31, half = lane >> 5;
    // merge: the row's reference is the largest of the KS wavefronts', z and O are scaled to it
    float *const ml = reinterpret_cast<float *>(smem + NW * F32Tile::kBytes);       // [wavefront][m, l][row]
    const float l_tot = xhalf_sum(l);
    __syncthreads();
    f32_leave_partial(smem + w * F32Tile::kBytes, o, lane);
    if (half == 0) { ml[(2 * w) * 32 + l32] = m; ml[(2 * w + 1) * 32 + l32] = l_tot; }
    __syncthreads();
#pragma unroll
    for (int pass = 0; pass < 8 / KS; ++pass) {                     // a pass takes NW / 8 units
        const int i = 4 * NW * pass / 32, r = (threadIdx.x >> 4) + 4 * NW * pass % 32, ch = threadIdx.x & 15;
        const F32Unit u = W::unit(a, i);
        const float sink = sink_logit(a, u.head) * kLog2e;
        float mm = fast_max(sink, kNoLogit);
#pragma unroll
        for (int k = 0; k < KS; ++k) mm = fast_max(mm, ml[2 * (KS * i + k) * 32 + r]);
        float z = exp2f(sink - mm);
        f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const float f = exp2f(ml[2 * (KS * i + k) * 32 + r] - mm);
            z += f * ml[(2 * (KS * i + k) + 1) * 32 + r];
            const f32x4 y = f32_partial(smem, F32Tile::kBytes, KS * i + k, r, ch);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = fmaf(f, y[e], x[e]);
        }
        const float inv = 1.0f / z;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] *= inv;
        if (u.live && u.q0 + r < a.Sq) {
            *reinterpret_cast<f32x4 *>(t.o + (int64_t)u.b * a.os.b + (int64_t)u.head * a.os.h + (int64_t)(u.q0 + r) * a.os.s + 4 * ch) = x;
            if (ch == 0) a.lse[((int64_t)u.b * a.H + u.head) * a.Sq + u.q0 + r] = (mm + log2f(z)) * kLn2;
        }
    }
}
// The forward of a workgroup of NW wavefronts (16 KB of LDS each).
template <int KS, int NW>
__device__ __forceinline__ void f32_fwd_rows(const KArgs &a, char *smem) {
    const int q_offset = query_offset(a);
    const F32Ptrs t = f32_ptrs(a);
    using W = F32QueryWork<KS, NW>;
    const W wk(a, t, q_offset, smem);
    const int lane = wk.lane, l32 = lane & 31, half = lane >> 5, row = wk.q0 + l32;
    int pos;
    unsigned win;
    wk.row_info(a, q_offset, row, pos, win);
    if (wk.n_it > 0) { wk.request_k(a, 0); wk.request_v(a, 0); }
    float qr[32];    // Q[row][32*half + ks]
    load_row32(qr, t.q + (int64_t)wk.b * a.qs.b + (int64_t)wk.head * a.qs.h + (int64_t)min(row, a.Sq - 1) * a.qs.s + 32 * half, row < a.Sq);
    const F32Offsets lo = make_f32_offsets(lane);
    const float c = a.scale_log2;
    const float sink2 = sink_logit(a, wk.head) * kLog2e;
    float m = fast_max(sink2, kNoLogit), l = 0.0f;
    f32x16 o[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) { o[0][i] = 0.0f; o[1][i] = 0.0f; }

    wait_vmcnt<0>();       // the compiler's own loads have arrived: it puts no vmcnt wait (which would also drain the copies) into the loop
    for (int it = 0; it < wk.n_it; ++it) {
        const int n0 = wk.first_key(it);
        const bool more = it + 1 < wk.n_it;
        GPTOSS_F32_WAIT(F32Tile::kCopies);         // K is here; V may be on its way
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.0f;
        f32_rows_product(s, wk.ksm, lo, qr);       // S^T: rows = keys, lane = query row
        GPTOSS_F32_READS_DONE();
        if (more) wk.request_k(a, it + 1);
        if (!wk.interior(a, n0)) {
            const KeyMask km = make_key_mask(pos - n0, win, wk.kv_len - n0, half);
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = key_visible(km, 8 * (i >> 2) + (i & 3)) ? s[i] : -INFINITY;
        }
        float mx0 = s[0], mx1 = s[1];
#pragma unroll
        for (int i = 2; i < 16; i += 2) { mx0 = fast_max(mx0, s[i]); mx1 = fast_max(mx1, s[i + 1]); }
        const float m_new = fast_max(m, xhalf_max(fast_max(mx0, mx1)) * c);
        if (__builtin_amdgcn_ballot_w64(m_new != m) != 0ull) {
            const float alpha = exp2f(m - m_new);
            m = m_new;
            l *= alpha;
#pragma unroll
            for (int i = 0; i < 16; ++i) { o[0][i] *= alpha; o[1][i] *= alpha; }
        }
        float rs0 = 0.0f, rs1 = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            s[i] = exp2f(fmaf(s[i], c, -m));
            s[i + 1] = exp2f(fmaf(s[i + 1], c, -m));
            rs0 += s[i];
            rs1 += s[i + 1];
        }
        l += rs0 + rs1;
        if (more) GPTOSS_F32_WAIT(F32Tile::kCopies); else GPTOSS_F32_WAIT(0);
        f32_cols_product(o, wk.vsm, lo, s);        // O^T[d][row] += V^T[d][key] P^T[key][row]
        GPTOSS_F32_READS_DONE();
        if (more) wk.request_v(a, it + 1);
    }

    f32_fwd_merge<KS, NW>(a, t, smem, wk.w, lane, m, l, o);
}
template <int KS>
__global__ __launch_bounds__(256, 2) void attn_f32_fwd_kernel(const KArgs a) {
    __shared__ __attribute__((aligned(1024))) char smem[8 * F32Tile::kBytes];
    f32_fwd_rows<KS, 4>(a, smem);
}

// ---- backward step 1: -delta and lse*log2(e) into the scratch (same layout as the bf16 path) ----
template <typename Int>
__device__ __forceinline__ void f32_delta_rows(const KArgs &a, Int total) {
    const F32Ptrs t = f32_ptrs(a);
    const int c = threadIdx.x & 15;                                   // 16 lanes x 16 bytes = one 256-byte row
    const Int rid = (Int)blockIdx.x * 16 + (threadIdx.x >> 4);
    float acc = 0.0f, lse = 0.0f;
    if (rid < total) {
        const Int bh = rid / (Int)a.Sq, s = rid - bh * (Int)a.Sq, b = bh / (Int)a.H, h = bh - b * (Int)a.H;
        const f32x4 ov = *reinterpret_cast<const f32x4 *>(t.o + (int64_t)b * a.os.b + (int64_t)h * a.os.h + (int64_t)s * a.os.s + 4 * c);
        const f32x4 gv = *reinterpret_cast<const f32x4 *>(t.d_o + (int64_t)b * a.dos.b + (int64_t)h * a.dos.h + (int64_t)s * a.dos.s + 4 * c);
        lse = a.lse[rid];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = fmaf(ov[e], gv[e], acc);
    }
    acc += __shfl_xor(acc, 1);
    acc += __shfl_xor(acc, 2);
    acc += __shfl_xor(acc, 4);
    acc += __shfl_xor(acc, 8);
    if (c == 0 && rid < total) {
        a.delta[rid] = -acc;
        a.delta[total + rid] = lse * kLog2e;
    }
}
__global__ __launch_bounds__(256) void attn_f32_delta_kernel(const KArgs a) {
    const int64_t total = (int64_t)a.B * a.H * a.Sq;
    if (total < ((int64_t)1 << 30)) f32_delta_rows(a, (uint32_t)total); else f32_delta_rows(a, total);
}

// ---- backward step 2: dK, dV ------------------------------------------------------------
// Problems with few key blocks are cut into slices of the query tiles besides (fp32 partials in the scratch, as in the
// bf16 path).
struct F32Dkdv {
    static constexpr int kStatBytes = 2 * 32 * 4;                      // 32 x -delta, 32 x lse * log2(e)
    static constexpr int kStatOff = 8 * F32Tile::kBytes;
    static constexpr int kLdsBytes = kStatOff + 4 * kStatBytes;
};
// The 32-row query tiles [t_lo, t_hi) whose rows can see any key of [j0, j0 + keys): positions [j0, last key + window), within the
// documents of the keys.
struct F32TileSpan { int t_lo, t_hi, row_lim; };
__device__ __forceinline__ F32TileSpan f32_tiles_of_keys(const KArgs &a, int q_offset, int b, int j0, int keys, int lane) {
    const int kv_len = a.seqlens ? min(a.Skv, a.seqlens[b]) : a.Skv;
    const int q_len = a.seqlens ? a.seqlens[b] : 0x7fffffff;
    const int j1 = min(j0 + keys, kv_len) - 1;
    const int32_t *dsrow = a.doc_start ? a.doc_start + (int64_t)b * a.Sq : nullptr;
    const int weff = a.window ? a.window : 0x3fffffff;
    F32TileSpan x;
    x.row_lim = (int)min((int64_t)a.Sq, max((int64_t)0, (int64_t)q_len - q_offset));
    const int row_lo = max(0, j0 - q_offset);
    int row_hi = j1 >= j0 ? (int)min((int64_t)x.row_lim, max((int64_t)0, (int64_t)j1 + weff - q_offset)) : 0;
    if (dsrow && row_hi > row_lo) row_hi = min(row_hi, document_end(dsrow, a.Sq, j1, lane));
    x.t_lo = row_lo / 32;
    x.t_hi = max(x.t_lo, (row_hi + 31) / 32);
    return x;
}
// Step `it` of a walk over (query tile, head): the heads of the group tile by tile, all of them with rows that see the keys.
struct F32TileWalk {
    int t0, n_it;
    __device__ __forceinline__ int tile(int it, int r) const { return t0 + it / r; }
    __device__ __forceinline__ int readable_tile(int it, int r) const { return tile(it, r); }
    __device__ __forceinline__ int head(int it, int r) const { return it % r; }
    __device__ __forceinline__ bool sees(int) const { return true; }
};
// The same by pairs of tiles (both of a head, the heads of the group, the pair after these) from step `first` on, for one of several key blocks:
// tiles outside [t_from, t_to) have no row that sees its keys and are passed over, one past the last is read as that one.  (A type of its own: with both walks
// in one, attn_f32_dkdv_kernel divided by a run-time number more often per request and step; forward + backward of 1000 rows of 8 heads on one KV head 148.9 us
// instead of 148.0, of 64 on 8 with a window of 128 144.5 instead of 143.0.)
struct F32PairWalk {
    int t0, t_end, first, n_it, t_from, t_to;
    __device__ __forceinline__ int tile(int it, int r) const { return t0 + 2 * ((first + it / 2) / r) + it % 2; }
    __device__ __forceinline__ int readable_tile(int it, int r) const { return min(tile(it, r), t_end - 1); }
    __device__ __forceinline__ int head(int it, int r) const { return (first + it / 2) % r; }
    __device__ __forceinline__ bool sees(int tile) const { return tile >= t_from && tile < t_to; }
};
// dK, dV of 32 keys from j0 over a walk (its steps dealt to the NW wavefronts in turn); out: fp32 partial sums, rows of 64 floats, or
// NULL for the scaled results
template <int NW, typename Walk>
__device__ __forceinline__ void f32_dkdv_keys(const KArgs &a, char *smem, int g, int b, int j0, const Walk walk, float *out_k, float *out_v) {
    using C = F32Dkdv;
    const int q_offset = query_offset(a);
    const F32Ptrs t = f32_ptrs(a);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, half = lane >> 5;
    const int kv_len = a.seqlens ? min(a.Skv, a.seqlens[b]) : a.Skv;
    const int q_len = a.seqlens ? a.seqlens[b] : 0x7fffffff;
    const int key = j0 + l32;
    const int64_t total = (int64_t)a.B * a.H * a.Sq;
    const int32_t *dsrow = a.doc_start ? a.doc_start + (int64_t)b * a.Sq : nullptr;

    float kr[32], vr[32];    // K / V[key][32*half + ks]  (B operands of S and dP)
    load_row32(kr, t.k + (int64_t)b * a.ks.b + (int64_t)g * a.ks.h + (int64_t)min(key, a.Skv - 1) * a.ks.s + 32 * half, key < a.Skv);
    load_row32(vr, t.v + (int64_t)b * a.vs.b + (int64_t)g * a.vs.h + (int64_t)min(key, a.Skv - 1) * a.vs.s + 32 * half, key < a.Skv);
    f32x16 dk[2], dv[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) { dk[0][i] = dk[1][i] = 0.0f; dv[0][i] = dv[1][i] = 0.0f; }

    const int weff = a.window ? a.window : 0x3fffffff;
    const int row_lim = (int)min((int64_t)a.Sq, max((int64_t)0, (int64_t)q_len - q_offset));
    const int n_it = walk.n_it;

    const uint32_t qsm = lds_addr(smem) + w * (2 * F32Tile::kBytes), gsm = qsm + F32Tile::kBytes;
    const uint32_t ssm = lds_addr(smem) + NW * 2 * F32Tile::kBytes + w * C::kStatBytes;
    const F32Offsets lo = make_f32_offsets(lane);
    const float c = a.scale_log2;
    // requests for step `it`: the Q tile; the dO tile and the row statistics
    auto request_q = [&](int it) __attribute__((always_inline)) {
        const int q0 = 32 * walk.readable_tile(it, a.r), head = g * a.r + walk.head(it, a.r);
        f32_copy_tile(qsm, t.q + (int64_t)b * a.qs.b + (int64_t)head * a.qs.h + (int64_t)q0 * a.qs.s, (int)a.qs.s, a.Sq - 1 - q0, lane);
    };
    auto request_g = [&](int it) __attribute__((always_inline)) {
        const int q0 = 32 * walk.readable_tile(it, a.r), head = g * a.r + walk.head(it, a.r);
        f32_copy_tile(gsm, t.d_o + (int64_t)b * a.dos.b + (int64_t)head * a.dos.h + (int64_t)q0 * a.dos.s, (int)a.dos.s, a.Sq - 1 - q0, lane);
        lds_dma4(ssm, a.delta + ((int64_t)b * a.H + head) * a.Sq, ((half ? (uint32_t)total : 0u) + (uint32_t)min(q0 + l32, a.Sq - 1)) * 4u);
    };
    if (w < n_it) { request_g(w); request_q(w); }
    wait_vmcnt<0>();         // the compiler's own loads have arrived: no vmcnt wait of its own in the loop
    for (int it = w; it < n_it; it += NW) {
        const int tile = walk.tile(it, a.r), q0 = 32 * tile;
        const bool more = it + NW < n_it;
        if (!walk.sees(tile)) {
            GPTOSS_F32_WAIT(0);
            if (more) { request_g(it + NW); request_q(it + NW); }
            continue;
        }
        GPTOSS_F32_WAIT(F32Tile::kCopies);                             // dO and the statistics are here; Q may be on its way
        f32x16 s, dp;
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) {
            const f32x4 nd = lds_load128f(ssm + 16 * half, 32 * a4);
#pragma unroll
            for (int e = 0; e < 4; ++e) { s[4 * a4 + e] = 0.0f; dp[4 * a4 + e] = nd[e]; }     // dP starts at -delta of its row
        }
        f32_rows_product(dp, gsm, lo, vr);                             // rows = queries, lane = key
        GPTOSS_F32_WAIT(0);
        f32_rows_product(s, qsm, lo, kr);
        const bool interior = j0 + 31 <= q_offset + q0 && q_offset + q0 + 31 - weff < j0 && j0 + 32 <= kv_len && q0 + 32 <= row_lim && !dsrow;
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) {
            const f32x4 l2 = lds_load128f(ssm + 128 + 16 * half, 32 * a4);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int i = 4 * a4 + e;
                float p = exp2f(fmaf(s[i], c, -l2[e]));
                if (!interior) {
                    const int row = q0 + 8 * a4 + 4 * half + e;
                    bool vis = (unsigned)(q_offset + row - key) < (unsigned)weff && key < kv_len && row < row_lim;
                    if (dsrow) vis = vis && key >= dsrow[min(row, a.Sq - 1)];
                    p = vis ? p : 0.0f;
                }
                s[i] = p;
                dp[i] = p * dp[i];                                     // dS (without the softmax scale)
            }
        }
        // dV^T[d][key] += dO^T[d][row] P[row][key];  dK^T[d][key] += Q^T[d][row] dS[row][key]
        f32_cols_product(dv, gsm, lo, s);
        GPTOSS_F32_READS_DONE();
        if (more) request_g(it + NW);
        f32_cols_product(dk, qsm, lo, dp);
        GPTOSS_F32_READS_DONE();
        if (more) request_q(it + NW);
    }

    // the wavefronts' sums, added in wavefront order
    __syncthreads();
    f32_leave_partial(smem + w * (2 * F32Tile::kBytes), dk, lane);
    f32_leave_partial(smem + w * (2 * F32Tile::kBytes) + F32Tile::kBytes, dv, lane);
    __syncthreads();
#pragma unroll
    for (int pass = 0; pass < 16 / NW; ++pass) {
        const int which = 4 * NW * pass / 32, r = (tid >> 4) + 4 * NW * pass % 32, ch = tid & 15, j = j0 + r;
        f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            const f32x4 y = f32_partial(smem + which * F32Tile::kBytes, 2 * F32Tile::kBytes, k, r, ch);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] += y[e];
        }
        if (j < a.Skv) {
            if (out_k) {
                *reinterpret_cast<f32x4 *>((which == 0 ? out_k : out_v) + r * kD + 4 * ch) = x;
            } else {
                const Strides &st = which == 0 ? a.dks : a.dvs;
                const float mul = which == 0 ? a.scale : 1.0f;
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] *= mul;
                *reinterpret_cast<f32x4 *>((which == 0 ? t.dk : t.dv) + (int64_t)b * st.b + (int64_t)g * st.h + (int64_t)j * st.s + 4 * ch) = x;
            }
        }
    }
}
__device__ __forceinline__ void f32_dkdv_workgroup(const KArgs &a, char *smem, int bid) {
    const int g = bid % a.G; bid /= a.G;
    const int bi = bid % a.B; bid /= a.B;
    const int part = bid % a.dkdv_parts, kblk = bid / a.dkdv_parts;       // ascending: most work first
    const int b = rotated_batch_row(bi, kblk, a.B), j0 = 32 * kblk;
    const F32TileSpan span = f32_tiles_of_keys(a, query_offset(a), b, j0, 32, threadIdx.x & 63);
    const int n_tiles = span.t_hi - span.t_lo, slice = (n_tiles + a.dkdv_parts - 1) / a.dkdv_parts;
    const F32TileWalk walk{span.t_lo + part * slice, max(0, min(slice, n_tiles - part * slice)) * a.r};
    const int64_t tensor = (int64_t)a.B * a.G * a.Skv * kD;
    float *out = a.dkdv_parts > 1 ? a.dkdv_partial + 2 * part * tensor + (((int64_t)b * a.G + g) * a.Skv + j0) * kD : nullptr;
    f32_dkdv_keys<4>(a, smem, g, b, j0, walk, out, out ? out + tensor : nullptr);
}
__global__ __launch_bounds__(256, 2) void attn_f32_dkdv_kernel(const KArgs a) {
    __shared__ __attribute__((aligned(1024))) char smem[F32Dkdv::kLdsBytes];
    f32_dkdv_workgroup(a, smem, blockIdx.x);
}

// The slices' partial sums, added in slice order.  One thread per 16-byte output chunk.
__global__ __launch_bounds__(256) void attn_f32_dkdv_reduce_kernel(const KArgs a, int heads) {
    __shared__ float red[1024];
    if ((int)blockIdx.x < heads) { dsinks_of_head<256>(a, blockIdx.x, red); return; }
    const F32Ptrs t = f32_ptrs(a);
    const int64_t rows = (int64_t)a.B * a.G * a.Skv, tensor = rows * kD;
    const int64_t idx = (int64_t)(blockIdx.x - heads) * 256 + threadIdx.x;
    if (idx >= 2 * rows * 16) return;
    const int which = idx >= rows * 16;
    const int64_t rem = idx - (int64_t)which * rows * 16, row = rem >> 4;
    const float *src = a.dkdv_partial + (int64_t)which * tensor + rem * 4;
    f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int part = 0; part < a.dkdv_parts; ++part) {
        const f32x4 y = *reinterpret_cast<const f32x4 *>(src + (int64_t)part * 2 * tensor);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] += y[e];
    }
    const float mul = which == 0 ? a.scale : 1.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] *= mul;
    const int key = (int)(row % a.Skv), bg = (int)(row / a.Skv), g = bg % a.G, b = bg / a.G;
    const Strides &st = which == 0 ? a.dks : a.dvs;
    *reinterpret_cast<f32x4 *>((which == 0 ? t.dk : t.dv) + (int64_t)b * st.b + (int64_t)g * st.h + (int64_t)key * st.s + 4 * (rem & 15)) = x;
}

// ---- backward step 3: dQ ----------------------------------------------------------------
// FUSE_DELTA: the kernel also forms -delta and lse * log2(e) of its rows, in the summation order of
// attn_f32_delta_kernel, and leaves them in the scratch for the kernels that follow.
template <int KS, int NW>
__device__ __forceinline__ void f32_dq_merge(const KArgs &a, const F32Ptrs &t, char *smem, int w, int lane, float mul, const f32x16 (&dq)[2]) {
    using W = F32QueryWork<KS, NW>;
    __syncthreads();
    f32_leave_partial(smem + w * F32Tile::kBytes, dq, lane);
    __syncthreads();
#pragma unroll
    for (int pass = 0; pass < 8 / KS; ++pass) {
        const int i = 4 * NW * pass / 32, r = (threadIdx.x >> 4) + 4 * NW * pass % 32, ch = threadIdx.x & 15;
        const F32Unit u = W::unit(a, i);
        f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const f32x4 y = f32_partial(smem, F32Tile::kBytes, KS * i + k, r, ch);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] += y[e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] *= mul;
        if (u.live && u.q0 + r < a.Sq)
            *reinterpret_cast<f32x4 *>(t.dq + (int64_t)u.b * a.dqs.b + (int64_t)u.head * a.dqs.h + (int64_t)(u.q0 + r) * a.dqs.s + 4 * ch) = x;
    }
}
template <int KS, bool FUSE_DELTA, int NW>
__device__ __forceinline__ void f32_dq_rows(const KArgs &a, char *smem) {
    const int q_offset = query_offset(a);
    const F32Ptrs t = f32_ptrs(a);
    using W = F32QueryWork<KS, NW>;
    const W wk(a, t, q_offset, smem);
    const int lane = wk.lane, l32 = lane & 31, half = lane >> 5, row = wk.q0 + l32;
    const bool row_ok = row < a.Sq;
    int pos;
    unsigned win;
    wk.row_info(a, q_offset, row, pos, win);
    const int64_t total = (int64_t)a.B * a.H * a.Sq;
    const int rowc = min(row, a.Sq - 1);
    const int64_t rid = ((int64_t)wk.b * a.H + wk.head) * a.Sq + rowc;

    if (wk.n_it > 0) { wk.request_v(a, 0); wk.request_k(a, 0); }
    float qr[32], gr[32];
    load_row32(qr, t.q + (int64_t)wk.b * a.qs.b + (int64_t)wk.head * a.qs.h + (int64_t)rowc * a.qs.s + 32 * half, row_ok);
    load_row32(gr, t.d_o + (int64_t)wk.b * a.dos.b + (int64_t)wk.head * a.dos.h + (int64_t)rowc * a.dos.s + 32 * half, row_ok);
    float ndelta, lse2;
    if constexpr (FUSE_DELTA) {
        const float *orow = t.o_in + (int64_t)wk.b * a.os.b + (int64_t)wk.head * a.os.h + (int64_t)rowc * a.os.s + 32 * half;
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const f32x4 ov = *reinterpret_cast<const f32x4 *>(orow + 4 * j);
            x[j] = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[j] = fmaf(ov[e], gr[4 * j + e], x[j]);
        }
        ndelta = -xhalf_sum(((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7])));
        lse2 = a.lse[rid] * kLog2e;
        if (row_ok && half == 0 && wk.w % KS == 0) {       // (a unit past the end holds rows of the first block again: the same values)
            a.delta[rid] = ndelta;
            a.delta[total + rid] = lse2;
        }
    } else {
        ndelta = a.delta[rid];
        lse2 = a.delta[total + rid];
    }
    const F32Offsets lo = make_f32_offsets(lane);
    const float c = a.scale_log2;
    f32x16 dq[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) { dq[0][i] = 0.0f; dq[1][i] = 0.0f; }

    wait_vmcnt<0>();         // the compiler's own loads have arrived: no vmcnt wait of its own in the loop
    for (int it = 0; it < wk.n_it; ++it) {
        const int n0 = wk.first_key(it);
        const bool more = it + 1 < wk.n_it;
        f32x16 s, dp;
#pragma unroll
        for (int i = 0; i < 16; ++i) { s[i] = 0.0f; dp[i] = ndelta; }
        GPTOSS_F32_WAIT(F32Tile::kCopies);         // V is here; K may be on its way
        f32_rows_product(dp, wk.vsm, lo, gr);      // dP^T - delta
        GPTOSS_F32_WAIT(0);
        GPTOSS_F32_READS_DONE();
        if (more) wk.request_v(a, it + 1);
        f32_rows_product(s, wk.ksm, lo, qr);       // S^T
        const bool interior = wk.interior(a, n0);
        const KeyMask km = make_key_mask(pos - n0, win, wk.kv_len - n0, half);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float p = exp2f(fmaf(s[i], c, -lse2));
            if (!interior) p = key_visible(km, 8 * (i >> 2) + (i & 3)) ? p : 0.0f;
            dp[i] = p * dp[i];
        }
        f32_cols_product(dq, wk.ksm, lo, dp);      // dQ^T[d][row] += K^T[d][key] dS^T[key][row]
        GPTOSS_F32_READS_DONE();
        if (more) wk.request_k(a, it + 1);
    }
    f32_dq_merge<KS, NW>(a, t, smem, wk.w, lane, a.scale, dq);
}
template <int KS, bool FUSE_DELTA>
__global__ __launch_bounds__(256, 2) void attn_f32_dq_kernel(const KArgs a) {
    __shared__ __attribute__((aligned(1024))) char smem[8 * F32Tile::kBytes];
    f32_dq_rows<KS, FUSE_DELTA, 4>(a, smem);
}

// dQ (the first workgroups) and dK/dV side by side behind the row statistics, where all of them run at once: the float32 counterpart of
// attn_bwd_both_kernel, with the bits of the two launches.
__global__ __launch_bounds__(256, 2) void attn_f32_both_kernel(const KArgs a, int dq_workgroups) {
    static_assert(F32Dkdv::kLdsBytes >= 8 * F32Tile::kBytes, "one array for both");
    __shared__ __attribute__((aligned(1024))) char smem[F32Dkdv::kLdsBytes];
    if ((int)blockIdx.x < dq_workgroups) f32_dq_rows<4, false, 4>(a, smem);
    else f32_dkdv_workgroup(a, smem, blockIdx.x - dq_workgroups);
}

}  // namespace gptoss
