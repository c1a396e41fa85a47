// float32 attention on the bf16 matrix pipes: every float32 operand as the sum of three bf16 terms.
//
// Why.  The fp32 matrix instruction takes sixteen times as long per product as the bf16 one, and the kernels of attn_f32.h are
// bound by it.  A float32 number IS the sum of three bf16 numbers (the number rounded to nearest, what is left rounded to nearest, the
// rest: 8 + 8 + 8 bits, each term exact), a product of two bf16 numbers is exact in fp32, and the bf16 instruction accumulates in
// fp32.  Of the nine term products six are kept (hi lo, lo hi, mid mid, hi mid, mid hi, hi hi).  With operands in [1, 2) mid is at most 2^-8 and lo
// at most 2^-17, so the three dropped ones are at most 2^-24 together, either sign: half a rounding of the product in the last
// place.  (Terms cut off instead of rounded would lose up to 2^-21 and always towards zero.)  That is 192 cycles of the pipe where the fp32 instruction takes 512.
// The order of the additions matters as much as the terms: an addition to an accumulator rounds at the accumulator's size (the instruction
// adds its 16 products in two groups of eight, each sum rounded once).  S and dP therefore take the small products of the whole contraction first and
// the four hi hi last: eight roundings at full size instead of 48.  And -delta, which is often almost all of dP, is added behind the products.
//
// What the split asks of the numbers.  Terms are exact while they stay normal and nothing overflows: inputs that are 0 or of magnitude
// 2^-100 to 2^24 (SplitCheck), and row statistics that go with them; a workgroup that meets any other (infinities and NaN among them) takes the walk of attn_f32.h
// instead, within the same launch.  Weights are held as 2^24 P (0 or 2^-125 to 2^24: also the terms of denormal ones are) and so is dS.
// (The factor is a product behind the exponential.  In its argument it would cost precision: a float near 24 is 2^-19 apart.)
//
// How.  attn_f32_split_kv_kernel cuts K and V once per call, into records of 32 keys: six planes of 32 rows x 128 bytes, their 16-byte
// chunks swizzled as the LDS tiles of attn_common.h are, so that a copy to LDS is linear and the bf16 fragment reads apply plane by
// plane.  The forward cuts its Q rows in registers; dQ cuts Q and dO and leaves them as records of 32 rows (with the row statistics)
// for dK/dV.  A workgroup is eight wavefronts, one workgroup per compute unit: forward and dQ take four heads x 32 rows, two
// wavefronts each, which walk the key tiles in turn; dK/dV takes four blocks of 32 keys, two wavefronts each, which walk the query
// tiles in turn.  Both add their shares in LDS.  A step stages two tiles (48 KB), the next step's pair under way meanwhile, one
// barrier per step.  Where the records of all batch rows and KV heads would take too much memory, the launches are repeated for some of them
// at a time, over the same scratch (f32_split_plan).
//
// What bounds it (S = 1024, 64 query heads on 8 KV heads, full causal; fp32 instruction / this): forward 101 / 58 us, dQ 134 / 83, dK/dV
// 176 / 94, the whole call 413 / 270; S = 4096 5320 / 3120.  The matrix pipes are busy 42, 45 and 53 % of the cycles: about eight
// vector instructions per MFMA in the forward (cutting the weights is 88 of a tile's 290), and the two wavefronts of a SIMD start each step together.
// Error against float64 (relative 2-norm, S = 1024, fp32 instruction / this), N(0, 1): O 3.0e-7 / 1.3e-7, lse 4.8e-8 / 4.8e-8, dQ 4.4e-7 / 3.4e-7, dK
// 6.0e-7 / 5.1e-7, dV 5.9e-7 / 5.1e-7; all operands in [1, 1 + 2^-7], where dP - delta cancels: dQ 2.2e-3 / 2.1e-3, dK 1.24e-5 / 1.15e-5; powers of two
// times 1 + 2^-7 - 2^-23: O 2.6e-7 / 1.4e-7, dK 5.6e-7 / 4.3e-7; one non-zero number per row: O 7.7e-8 / 7.1e-8, dK 2.85e-7 / 2.85e-7, dV 2.86e-7 / 3.06e-7 (a product is six
// additions to dV, which shows where a sum has few).
#pragma once
#include "attn_f32.h"

namespace gptoss {

struct F32Split {
    static constexpr int kTerms = 3;
    static constexpr int kPlane = 32 * kRowBytes;                      // 32 rows of one term of one tensor
    static constexpr int kKvRecord = 2 * kTerms * kPlane;              // K hi, mid, lo, V hi, mid, lo
    static constexpr int kStatOff = 2 * kTerms * kPlane;
    static constexpr int kQRecord = kStatOff + 2 * 32 * 4;             // Q and dO likewise, 32 x -delta, 32 x lse * log2(e)
    static constexpr int kKeys = 128;                                  // keys of a dK/dV workgroup
    static constexpr int kWaves = 8;
    static constexpr int kWaveCopy = 2 * kTerms * kPlane / 4;          // a tile is copied by four wavefronts
    static constexpr int kRowsLds = kWaves * 2 * F32Tile::kBytes;      // the general walk's tiles (the records' stages are smaller)
    static constexpr int kKeptOff = 4 * kQRecord, kKeptKeys = 15 * 1024, kKeptRows = 6 * 1024;   // behind the stages: operands that do not fit the registers (SplitKept)
    static constexpr int kDkdvLds = kKeptOff + 4 * kKeptKeys;
    static constexpr int kDqLds = kKeptOff + kWaves * kKeptRows;
    static_assert(4 * kKvRecord <= kRowsLds && kRowsLds <= kDqLds && kRowsLds + kWaves * F32Dkdv::kStatBytes <= kDkdvLds, "two stages of two tiles; the general walk");
};
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-24f;       // weights are held as 2^24 P
constexpr float kSplitMostDelta = 0x1p54f;                             // what 64 products of numbers up to 2^24 and 2^24 reach
// The weights are 2^24 exp2(x).  The bare exponential instruction flushes what is below 2^-126: whether a wavefront has none of that.
__device__ __forceinline__ bool split_weights_normal(const f32x16 &x) {
    float lo = fminf(x[0], x[1]);
#pragma unroll
    for (int i = 2; i < 16; i += 2) lo = fminf(fminf(lo, x[i]), x[i + 1]);
    return __builtin_amdgcn_ballot_w64(!(lo >= -125.0f)) == 0ull;
}
__device__ __forceinline__ float split_weight(float x) { return fast_exp2(x) * kSplitScale; }
__device__ __forceinline__ void split_any_weights(f32x16 &x) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        asm volatile("" : "+v"(x[i]));       // (keeps the compiler from doing this for every tile and choosing afterwards)
        x[i] = exp2f(x[i]) * kSplitScale;
    }
}
// Numbers the split does not take: not 0 and below 2^-100, above 2^24, infinite or NaN.
struct SplitCheck {
    uint32_t most = 0, least = ~0u;                                    // of the magnitudes' bits, and of these less one (0: the most)
    __device__ __forceinline__ void look(float x) {
        const uint32_t u = __float_as_uint(x) & 0x7fffffffu;
        most = max(most, u);
        least = min(least, u - 1u);
    }
    __device__ __forceinline__ bool bad() const { return most > 0x4B800000u || least < 0x0D800000u - 1u; }
};

// A pair of numbers as bf16, each to nearest even, in one register; and what they leave of it (exact).
__device__ __forceinline__ uint32_t split_round2(float x, float y) {
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x, y}), bf16x2));
}
__device__ __forceinline__ void split_rest2(float &x, float &y, uint32_t p) {
    x -= __uint_as_float(p << 16);
    y -= __uint_as_float(p & 0xffff0000u);
}
// eight numbers as three bf16 vectors whose sum they are: the number rounded to bf16, what is left rounded to bf16, the rest (exact)
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8 (&t)[3]) {
    u32x4 w[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float u = x[2 * i], v = x[2 * i + 1];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            w[k][i] = split_round2(u, v);
            if (k < 2) split_rest2(u, v, w[k][i]);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) t[k] = as_bf16x8(w[k]);
}
// Registers 8u .. 8u + 7 of a C block, the k slots that a transposed fragment of the same 16-row step holds, cut into terms in twelve
// steps of at most five instructions (an MFMA leaves room for four), a pair of numbers in three.
struct SplitSteps {
    float r[2];
    u32x4 w[3];
    __device__ __forceinline__ void step(const f32x16 &c, int u, int i) {
        const int pair = i / 3, k = i % 3;
        float x = k == 0 ? c[8 * u + 2 * pair] : r[0], y = k == 0 ? c[8 * u + 2 * pair + 1] : r[1];
        const uint32_t p = split_round2(x, y);
        w[k][pair] = p;
        if (k < 2) {
            split_rest2(x, y, p);
            r[0] = x;
            r[1] = y;
        }
    }
    __device__ __forceinline__ void take(bf16x8 (&t)[3]) const {
#pragma unroll
        for (int k = 0; k < 3; ++k) t[k] = as_bf16x8(w[k]);
    }
};
__device__ __forceinline__ void split_cfrag(const f32x16 &c, int u, bf16x8 (&t)[3]) {
    SplitSteps x;
#pragma unroll
    for (int i = 0; i < 12; ++i) x.step(c, u, i);
    x.take(t);
}
// Operands of a lane that do not fit its registers: fragments in LDS, 1 KB each, lane by lane.
struct SplitKept {
    uint32_t at;       // the first one's address for this lane
    __device__ __forceinline__ bf16x8 get(int i) const { return as_bf16x8(lds_load128(at, i * 1024)); }
    __device__ __forceinline__ void put(int i, const bf16x8 x) const {
        *reinterpret_cast<__attribute__((address_space(3))) bf16x8 *>((uintptr_t)(at + i * 1024)) = x;
    }
};
// s += X Y^T over head_dim: X's rows from three planes (OFF bytes behind the addresses `at`), y the lane's row of Y.  24 MFMAs: the five
// small products of the four 16-deep steps, small ones first, then the four products of the first terms, the last step's first
// (its operands are at hand; the others' are read again).  S of N(0, 1) with the six products of a step together: O 2.0e-7 from float64 instead of 1.3e-7, lse 4.82e-8 instead of
// 4.79e-8, the whole call 0.2 % faster.  A fragment's register is loaded with the next step's right behind its last use.  Term p of y in step ks is
// fragment KEPT(p, ks) of `kept`, or in its register where that is negative.
// FLIP: X and Y have changed places (dK/dV, whose tiles are the rows that dQ holds): each pair of products of equal size is added in the other
// order, so that S and dP have the bits that the forward and dQ see.
// work(i) is issued behind MFMA i of the 24.
template <int OFF, bool FLIP, typename Kept, typename Work>
__device__ __forceinline__ void split_rows_product(f32x16 &s, const TileLaneOffsets &at, const bf16x8 (&y)[4][3], const SplitKept &kept, Kept kept_at, Work work) {
    auto load = [&](int ks, int p) __attribute__((always_inline)) { return as_bf16x8(lds_load128(at.nat[ks], OFF + p * F32Split::kPlane)); };
    auto term = [&](int ks, int p) __attribute__((always_inline)) { return kept_at(p, ks) >= 0 ? kept.get(kept_at(p, ks)) : y[ks][p]; };
    auto mac = [&](const bf16x8 &x, const bf16x8 &y_, int i) __attribute__((always_inline)) {
        s = mfma_bf16(x, y_, s);
        work(i);
        GPTOSS_F32_FENCE();
    };
    bf16x8 x2 = load(0, 2), y0 = term(0, 0), x1 = load(0, 1), y1 = term(0, 1), x0 = load(0, 0), y2 = term(0, 2);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const bool more = ks < 3;
        GPTOSS_F32_FENCE();
        if (FLIP) {
            mac(x0, y2, 5 * ks);
            if (more) y2 = term(ks + 1, 2);
            mac(x1, y1, 5 * ks + 1);
            mac(x2, y0, 5 * ks + 2);
            if (more) x2 = load(ks + 1, 2);
            mac(x0, y1, 5 * ks + 3);
            if (more) y1 = term(ks + 1, 1);
            mac(x1, y0, 5 * ks + 4);
            if (more) x1 = load(ks + 1, 1);
        } else {
            mac(x2, y0, 5 * ks);
            if (more) x2 = load(ks + 1, 2);
            mac(x1, y1, 5 * ks + 1);
            mac(x0, y2, 5 * ks + 2);
            if (more) y2 = term(ks + 1, 2);
            mac(x1, y0, 5 * ks + 3);
            if (more) x1 = load(ks + 1, 1);
            mac(x0, y1, 5 * ks + 4);
            if (more) y1 = term(ks + 1, 1);
        }
        if (more) { x0 = load(ks + 1, 0); y0 = term(ks + 1, 0); }
    }
#pragma unroll
    for (int ks = 3; ks >= 0; --ks) {
        bf16x8 next_x = x0, next_y = y0;
        if (ks > 0) { next_x = load(ks - 1, 0); next_y = term(ks - 1, 0); }
        GPTOSS_F32_FENCE();
        mac(x0, y0, 23 - ks);
        x0 = next_x;
        y0 = next_y;
    }
}
constexpr int kInRegister = -1;
struct SplitNoneKept { __device__ __forceinline__ constexpr int operator()(int, int) const { return kInRegister; } };
struct SplitNoWork { __device__ __forceinline__ void operator()(int) const {} };
// acc^T[d][col] += X^T[d][row] p[row][col] over the 32 rows of three planes, six MFMAs per 16 rows and 32 columns, small ones first; p as terms of C registers: the first half's at hand, the
// second half's when work(11) has been issued
template <int OFF, typename Work>
__device__ __forceinline__ void split_cols_product(f32x16 (&acc)[2], const TileLaneOffsets &at, const bf16x8 (&p)[2][3], Work work) {
    auto load = [&](int i, int k) __attribute__((always_inline)) {     // i = 2 u + dblk
        const int u = i >> 1, dblk = i & 1;
        union { struct { s16x4 a, b; } s; bf16x8 v; } f;
        f.s.a = lds_load_tr64(at.tr[dblk][0], OFF + k * F32Split::kPlane + 16 * u * kRowBytes);
        f.s.b = lds_load_tr64(at.tr[dblk][1], OFF + k * F32Split::kPlane + 16 * u * kRowBytes);
        return f.v;
    };
    bf16x8 x2 = load(0, 2), x1 = load(0, 1), x0 = load(0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bool more = i < 3;
        auto mac = [&](const bf16x8 &x, int term, int m) __attribute__((always_inline)) {
            acc[i & 1] = mfma_bf16(x, p[i >> 1][term], acc[i & 1]);
            work(6 * i + m);
            GPTOSS_F32_FENCE();
        };
        GPTOSS_F32_FENCE();
        mac(x2, 0, 0);
        if (more) x2 = load(i + 1, 2);
        mac(x1, 1, 1);
        mac(x0, 2, 2);
        mac(x1, 0, 3);
        if (more) x1 = load(i + 1, 1);
        mac(x0, 1, 4);
        mac(x0, 0, 5);
        if (more) x0 = load(i + 1, 0);
    }
}
// the same with p still to be cut, its first half ahead of the product, its second behind the first twelve MFMAs
template <int OFF>
__device__ __forceinline__ void split_cols_product(f32x16 (&acc)[2], const TileLaneOffsets &at, const f32x16 &p) {
    bf16x8 f[2][3];
    split_cfrag(p, 0, f[0]);
    SplitSteps next;
    split_cols_product<OFF>(acc, at, f, [&](int i) __attribute__((always_inline)) {
        if (i < 12) next.step(p, 1, i);
        if (i == 11) next.take(f[1]);
    });
}
// the lane's 64 floats of a row as B operands of the four 16-deep steps (columns 16 ks + 8 half + 0 .. 7); zero when !valid
__device__ __forceinline__ void split_row(bf16x8 (&y)[4][3], const float *row, bool valid, int half, SplitCheck &check) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
            if (valid) z = *reinterpret_cast<const f32x4 *>(row + 16 * ks + 8 * half + 4 * j);
#pragma unroll
            for (int e = 0; e < 4; ++e) { x[4 * j + e] = z[e]; check.look(z[e]); }
        }
        split8(x, y[ks]);
    }
}
// byte of a plane where chunk c (8 columns) of row r stands
__device__ __forceinline__ int plane_chunk(int r, int c) { return r * kRowBytes + ((c ^ swz(r)) << 4); }
// a wavefront's share of a record: kWaveCopy bytes from `src` to LDS
__device__ __forceinline__ void split_copy(uint32_t dst, const char *src, int lane) {
#pragma unroll
    for (int i = 0; i < F32Split::kWaveCopy / 1024; ++i) lds_dma16(dst + i * 1024, src + i * 1024, (uint32_t)(lane * 16));     // (one lane offset for all of them)
}

// where the records and the partial sums of a batch row's KV head stand among those of the launch
__device__ __forceinline__ int64_t split_row_of(const KArgs &a, int b, int g) { return (int64_t)(b - a.split_b0) * a.split_ng + (g - a.split_g0); }

// The first 32 keys with a record: behind a cache a window's queries see the last ones only (256 queries on 16384 keys, window 128: forward with
// a record for every key 71 us).  The host counts split_tiles of them (split_key_tiles).
__device__ __forceinline__ int split_first_tile(const KArgs &a, int q_offset) { return a.window > 0 ? max(0, q_offset - a.window + 1) / 32 : 0; }
// from the tile of the first query's first key to that of the last query, wherever the queries stand in these
__host__ __device__ inline int split_key_tiles(int Sq, int Skv, int window) {
    const int64_t all = ((int64_t)Skv + 31) / 32, seen = ((int64_t)Sq + window - 2) / 32 + 2;
    return (int)(window > 0 && seen < all ? seen : all);
}
// ---- K and V as records ------------------------------------------------------------------------------------
// One workgroup per (batch, KV head, 32 keys).  Keys that nobody sees (past the tensor, a padded row's length, the last query) are
// zeros.  Bound by memory: 10 bytes moved per number.
__global__ __launch_bounds__(256) void attn_f32_split_kv_kernel(const KArgs a) {
    const F32Ptrs t = f32_ptrs(a);
    const int q_offset = query_offset(a);
    const int nt = a.split_tiles, tile = split_first_tile(a, q_offset) + (int)(blockIdx.x % nt), bg = (int)(blockIdx.x / nt), b = a.split_b0 + bg / a.split_ng, g = a.split_g0 + bg % a.split_ng;
    const int which = threadIdx.x >> 7, r = (threadIdx.x >> 2) & 31, part = threadIdx.x & 3, key = 32 * tile + r;
    int64_t end = min((int64_t)a.Skv, (int64_t)q_offset + a.Sq);
    if (a.seqlens) end = min(end, (int64_t)a.seqlens[b]);
    const float *row = which == 0 ? t.k + (int64_t)b * a.ks.b + (int64_t)g * a.ks.h + (int64_t)key * a.ks.s
                                  : t.v + (int64_t)b * a.vs.b + (int64_t)g * a.vs.h + (int64_t)key * a.vs.s;
    char *rec = a.split_kv + (int64_t)blockIdx.x * F32Split::kKvRecord + which * F32Split::kTerms * F32Split::kPlane;
    SplitCheck check;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
            if (key < end) z = *reinterpret_cast<const f32x4 *>(row + 16 * part + 8 * i + 4 * j);
#pragma unroll
            for (int e = 0; e < 4; ++e) { x[4 * j + e] = z[e]; check.look(z[e]); }
        }
        bf16x8 y[3];
        split8(x, y);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x8 *>(rec + p * F32Split::kPlane + plane_chunk(r, 2 * part + i)) = y[p];
    }
    const int bad = __syncthreads_or(check.bad());
    if (threadIdx.x == 0) a.split_kv_bad[blockIdx.x] = bad;
}

// The key tiles of a forward / dQ workgroup: all four units stand at the same rows, wavefront w takes tile 2 step + w % 2 of them.
struct SplitKeyWalk {
    const char *rec;
    const uint32_t *rec_bad;
    int t_end, t_lo, n, w, lane;
    uint32_t lds;
    __device__ __forceinline__ SplitKeyWalk(const KArgs &a, int q_offset, int b, int g, int t_lo_, int n_, int w_, int lane_, const char *smem)
        : t_lo(t_lo_), n(n_), w(w_), lane(lane_), lds(lds_addr(smem)) {
        const int t_first = split_first_tile(a, q_offset);
        t_end = t_first + a.split_tiles;
        const int64_t first = split_row_of(a, b, g) * a.split_tiles - t_first;       // (tile 0's)
        rec = a.split_kv + first * F32Split::kKvRecord;
        rec_bad = a.split_kv_bad + first;
    }
    __device__ __forceinline__ bool bad() const {
        uint32_t x = 0;
        for (int i = threadIdx.x; i < n; i += 64 * F32Split::kWaves) x |= rec_bad[t_lo + i];
        return x != 0;
    }
    __device__ __forceinline__ int steps() const { return (n + 1) >> 1; }
    // (the tile behind the last one, if there is none, is the last one again)
    __device__ __forceinline__ void request(int step) const {
        const int tile = min(t_lo + 2 * step + (w >> 2), t_end - 1);
        split_copy(lds + ((step & 1) * 2 + (w >> 2)) * F32Split::kKvRecord + (w & 3) * F32Split::kWaveCopy,
                   rec + (int64_t)tile * F32Split::kKvRecord + (w & 3) * F32Split::kWaveCopy, lane);
    }
};
// the step's tiles have landed and every wavefront is done with the step before
__device__ __forceinline__ void split_arrive() {
    wait_vmcnt<0>();
    __syncthreads();
}

// ---- forward ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(512, 2) void attn_f32_split_fwd_kernel(const KArgs a) {
    extern __shared__ __attribute__((aligned(1024))) char f32_split_lds[];
    char *const smem = f32_split_lds;
    const int q_offset = query_offset(a);
    const F32Ptrs t = f32_ptrs(a);
    const F32QueryWork<2, F32Split::kWaves> wk(a, t, q_offset, smem);
    const int lane = wk.lane, w = wk.w, l32 = lane & 31, half = lane >> 5, row = wk.q0 + l32;
    const SplitKeyWalk walk(a, q_offset, wk.b, wk.g, wk.t_lo, wk.n, w, lane, smem);
    if (walk.n > 0) walk.request(0);
    SplitCheck check;
    const bool keys_bad = walk.bad();
    bf16x8 qf[4][3];
    int pos;
    unsigned win;
    wk.row_info(a, q_offset, row, pos, win);
    split_row(qf, t.q + (int64_t)wk.b * a.qs.b + (int64_t)wk.head * a.qs.h + (int64_t)min(row, a.Sq - 1) * a.qs.s, pos >= 0, half, check);      // (what a padded row holds must not matter)
    wait_vmcnt<0>();
    if (__syncthreads_or(keys_bad || check.bad())) {
        f32_fwd_rows<2, F32Split::kWaves>(a, smem);
        return;
    }
    TileLaneOffsets at = tile_offsets_at(make_tile_offsets(lane), walk.lds + (w & 1) * F32Split::kKvRecord);
    const float c = a.scale_log2;
    float m = fast_max(sink_logit(a, wk.head) * kLog2e, kNoLogit), l = 0.0f;
    f32x16 o[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) { o[0][i] = 0.0f; o[1][i] = 0.0f; }
    const int n_steps = walk.steps();
    wait_vmcnt<0>();
    for (int step = 0; step < n_steps; ++step) {
        split_arrive();
        if (step + 1 < n_steps) walk.request(step + 1);
        const int tile = wk.t_lo + 2 * step + (w & 1), n0 = 32 * tile;
        if (tile < wk.t_lo + wk.n) {
            f32x16 s;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 0.0f;
            split_rows_product<0, false>(s, at, qf, SplitKept{}, SplitNoneKept{}, SplitNoWork{});      // S^T: rows = keys, lane = query row
            if (!wk.interior(a, n0)) {
                const KeyMask km = make_key_mask(pos - n0, win, wk.kv_len - n0, half);
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = key_visible(km, 8 * (i >> 2) + (i & 3)) ? s[i] : -INFINITY;
            }
            float mx0 = s[0], mx1 = s[1];
#pragma unroll
            for (int i = 2; i < 16; i += 2) { mx0 = fast_max(mx0, s[i]); mx1 = fast_max(mx1, s[i + 1]); }
            const float m_new = fast_max(m, xhalf_max(fast_max(mx0, mx1)) * c);
            // (a reference that lags behind the maximum by up to 2^8 would save most of these, 6 us at S = 1024, and cost precision: the
            // largest logits' differences from it are then not small)
            if (__builtin_amdgcn_ballot_w64(m_new != m) != 0ull) {
                const float alpha = exp2f(m - m_new);
                m = m_new;
                l *= alpha;
#pragma unroll
                for (int i = 0; i < 16; ++i) { o[0][i] *= alpha; o[1][i] *= alpha; }
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = fmaf(s[i], c, -m);
            if (split_weights_normal(s)) {
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = split_weight(s[i]);
            } else {
                split_any_weights(s);
            }
            float rs[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < 16; ++i) rs[i & 3] += s[i];
            l += (rs[0] + rs[1]) + (rs[2] + rs[3]);
            // O^T[d][row] += V^T[d][key] P^T[key][row], the tile's sum by itself first: O then is rounded once per tile, not twelve times
            f32x16 t_o[2];
#pragma unroll
            for (int i = 0; i < 16; ++i) { t_o[0][i] = 0.0f; t_o[1][i] = 0.0f; }
            split_cols_product<F32Split::kTerms * F32Split::kPlane>(t_o, at, s);
#pragma unroll
            for (int i = 0; i < 16; ++i) { o[0][i] += t_o[0][i]; o[1][i] += t_o[1][i]; }
        }
        tile_offsets_move(at, (step & 1) ? (uint32_t)(-2 * F32Split::kKvRecord) : (uint32_t)(2 * F32Split::kKvRecord));
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) { o[0][i] *= kSplitUnscale; o[1][i] *= kSplitUnscale; }
    f32_fwd_merge<2, F32Split::kWaves>(a, t, smem, w, lane, m, l * kSplitUnscale, o);
}

// ---- dQ, the row statistics, and Q and dO as records -----------------------------------------------------------
__global__ __launch_bounds__(512, 2) void attn_f32_split_dq_kernel(const KArgs a) {
    extern __shared__ __attribute__((aligned(1024))) char f32_split_lds[];
    char *const smem = f32_split_lds;
    const F32Ptrs t = f32_ptrs(a);
    const F32QueryWork<2, F32Split::kWaves> wk(a, t, 0, smem);
    const int lane = wk.lane, w = wk.w, l32 = lane & 31, half = lane >> 5, row = wk.q0 + l32;
    const bool row_ok = row < a.Sq, live = row_ok && row < wk.q_len;       // (what a padded row holds must not matter)
    const int rowc = min(row, a.Sq - 1);
    const SplitKeyWalk walk(a, 0, wk.b, wk.g, wk.t_lo, wk.n, w, lane, smem);
    if (walk.n > 0) walk.request(0);
    const int64_t total = (int64_t)a.B * a.H * a.Sq, rid = ((int64_t)wk.b * a.H + wk.head) * a.Sq + rowc;
    const int64_t rec_i = (split_row_of(a, wk.b, wk.g) * a.r + (wk.head - wk.g * a.r)) * ((a.Sq + 31) / 32) + wk.q0 / 32;
    char *const rec = a.split_q + rec_i * F32Split::kQRecord;
    const float *grow = t.d_o + (int64_t)wk.b * a.dos.b + (int64_t)wk.head * a.dos.h + (int64_t)rowc * a.dos.s;
    SplitCheck check;
    bf16x8 qf[4][3], gf[4][3];
    split_row(qf, t.q + (int64_t)wk.b * a.qs.b + (int64_t)wk.head * a.qs.h + (int64_t)rowc * a.qs.s, live, half, check);
    split_row(gf, grow, live, half, check);
    float ndelta = 0.0f;
    {
        const float *orow = t.o_in + (int64_t)wk.b * a.os.b + (int64_t)wk.head * a.os.h + (int64_t)rowc * a.os.s;
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int d = 16 * (j >> 1) + 8 * half + 4 * (j & 1);
            const f32x4 ov = *reinterpret_cast<const f32x4 *>(orow + d), gv = *reinterpret_cast<const f32x4 *>(grow + d);
            x[j] = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[j] = fmaf(ov[e], gv[e], x[j]);
        }
        ndelta = -xhalf_sum(((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7])));
    }
    const float lse2 = a.lse[rid] * kLog2e;
    // the statistics, too: dS must not overflow where it is held as 2^24 dS (a V outside the limits that only other workgroups see)
    const bool stats_bad = live && !(fabsf(ndelta) <= kSplitMostDelta && fabsf(lse2) < INFINITY);
    // the unit's two wavefronts hold the same rows: one leaves Q and the statistics, the other dO
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            if (w & 1) *reinterpret_cast<bf16x8 *>(rec + (3 + p) * F32Split::kPlane + plane_chunk(l32, 2 * ks + half)) = gf[ks][p];
            else *reinterpret_cast<bf16x8 *>(rec + p * F32Split::kPlane + plane_chunk(l32, 2 * ks + half)) = qf[ks][p];
        }
    const bool rows_bad = __builtin_amdgcn_ballot_w64(check.bad() || stats_bad) != 0ull;
    if (!(w & 1)) {
        reinterpret_cast<float *>(rec + F32Split::kStatOff)[lane] = live ? (half ? lse2 : ndelta) : 0.0f;
        if (lane == 0) a.split_q_bad[rec_i] = rows_bad;
        if (row_ok && half == 0) {
            a.delta[rid] = ndelta;
            a.delta[total + rid] = lse2;
        }
    }
    // the last term of dO and half of Q's stay in LDS (each wavefront a copy of its own)
    const SplitKept kept{walk.lds + F32Split::kKeptOff + w * F32Split::kKeptRows + lane * 16};
    auto kept_q = [](int p, int ks) { return p == 2 && ks >= 2 ? 2 + ks : kInRegister; };
    auto kept_g = [](int p, int ks) { return p == 2 ? ks : kInRegister; };
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        kept.put(kept_g(2, ks), gf[ks][2]);
        if (kept_q(2, ks) >= 0) kept.put(kept_q(2, ks), qf[ks][2]);
    }
    const bool keys_bad = walk.bad();
    if (!live) ndelta = 0.0f;
    wait_vmcnt<0>();
    if (__syncthreads_or(keys_bad || rows_bad)) {
        f32_dq_rows<2, true, F32Split::kWaves>(a, smem);
        return;
    }
    int pos;
    unsigned win;
    wk.row_info(a, 0, row, pos, win);
    TileLaneOffsets at = tile_offsets_at(make_tile_offsets(lane), walk.lds + (w & 1) * F32Split::kKvRecord);
    const float c = a.scale_log2;
    f32x16 dq[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) { dq[0][i] = 0.0f; dq[1][i] = 0.0f; }
    const int n_steps = walk.steps();
    wait_vmcnt<0>();
    for (int step = 0; step < n_steps; ++step) {
        split_arrive();
        if (step + 1 < n_steps) walk.request(step + 1);
        const int tile = wk.t_lo + 2 * step + (w & 1), n0 = 32 * tile;
        if (tile < wk.t_lo + wk.n) {
            f32x16 s, dp;
#pragma unroll
            for (int i = 0; i < 16; ++i) { s[i] = 0.0f; dp[i] = 0.0f; }
            split_rows_product<0, false>(s, at, qf, kept, kept_q, SplitNoWork{});               // S^T
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = fmaf(s[i], c, -lse2);
            // dP^T; the weights behind its MFMAs where all are visible and normal
            constexpr int kV = F32Split::kTerms * F32Split::kPlane;
            if (wk.interior(a, n0) && split_weights_normal(s)) {
                split_rows_product<kV, false>(dp, at, gf, kept, kept_g, [&](int i) __attribute__((always_inline)) { if (i < 16) s[i] = split_weight(s[i]); });
            } else {
                split_any_weights(s);
                const KeyMask km = make_key_mask(pos - n0, win, wk.kv_len - n0, half);
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = key_visible(km, 8 * (i >> 2) + (i & 3)) ? s[i] : 0.0f;
                split_rows_product<kV, false>(dp, at, gf, kept, kept_g, SplitNoWork{});
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) dp[i] = s[i] * (dp[i] + ndelta);
            split_cols_product<0>(dq, at, dp);                                           // dQ^T[d][row] += K^T[d][key] dS^T[key][row]
        }
        tile_offsets_move(at, (step & 1) ? (uint32_t)(-2 * F32Split::kKvRecord) : (uint32_t)(2 * F32Split::kKvRecord));
    }
    f32_dq_merge<2, F32Split::kWaves>(a, t, smem, w, lane, a.scale * kSplitUnscale, dq);
}

// ---- dK, dV ----------------------------------------------------------------------------------------------------
// A key block's walk: pairs of 32-row query tiles, all heads of the group per pair.  The host cuts it into parts of split_steps
// (pair, head) steps, one workgroup each, from the most steps the block can have (padding and documents make it shorter).
__host__ __device__ inline int split_block_steps(int Sq, int window, int r, int block) {
    const int64_t lo = (int64_t)F32Split::kKeys * block, hi = window > 0 ? lo + F32Split::kKeys - 1 + window : Sq;
    const int64_t tiles = ((hi < Sq ? hi : Sq) + 31) / 32 - lo / 32;
    return (int)((tiles + 1) / 2) * r;
}
__host__ __device__ inline int split_block_parts(int Sq, int window, int r, int block, int steps) {
    const int n = (split_block_steps(Sq, window, r, block) + steps - 1) / steps;
    return n < 1 ? 1 : n;
}
// Padded rows and packed documents (split_plan) have shorter walks, which only the device knows: the host's parts of them would be many short ones of the first
// blocks and one long one of the last.  A row's workgroups then divide its walks themselves, into parts of the number of steps that takes the fewest rounds as the
// host counts them, and need no more slots than the host counted.  Backward of 64 heads, us, fp32 instruction / the host's parts / so: 4096 tokens in documents of 100 332 / 515 / 365, of 250 541 / 630 / 455, of 700 1037 / 860 / 740, of 1000 1465 / 1060 / 890; 1024 tokens of 100 108 / 156 / 115, of 1000 350 / 210 / 213; 8 heads on one KV
// head, 4096 of 200 98 / 208 / 84; two rows of 1024 padded to 100 and 150 91 / 162 / 113.  (What is left of documents of 100 is the start of a workgroup per 128 keys and four
// heads, which dQ and the forward have too.)
struct SplitPart { int block, number, steps; };            // (block -1: there is nothing left for this workgroup)
__device__ __forceinline__ int split_walk_steps(const KArgs &a, int b, int block) {
    const int len = a.seqlens ? max(0, min(a.Sq, a.seqlens[b])) : a.Sq, lo = F32Split::kKeys * block, last = min(lo + F32Split::kKeys, len) - 1;
    if (last < lo) return 0;
    int end = a.window > 0 ? min(len, last + a.window) : len;
    if (a.doc_start) {                                     // the first row that does not see the block's last key
        const int32_t *row = a.doc_start + (int64_t)b * a.Sq;
        int from = last + 1;
        while (from < end) {
            const int x = (from + end) >> 1;
            if (row[x] > last) end = x; else from = x + 1;
        }
    }
    return (((end + 31) / 32 - lo / 32 + 1) >> 1) * a.r;
}
template <bool SHORT>
__device__ __forceinline__ SplitPart split_part(const KArgs &a, int b, int64_t bg, int slot, int lane) {
    const int blocks = (a.Skv + F32Split::kKeys - 1) / F32Split::kKeys;
    if (!SHORT || !a.split_plan) {
        int block = 0;
        for (int n; slot >= (n = split_block_parts(a.Sq, a.window, a.r, block, a.split_steps)); ++block) slot -= n;
        return {block, slot, a.split_steps};
    }
    int all = 0, most = 0, mine = 0;
    for (int i = lane; i < blocks; i += 64) {
        mine = split_walk_steps(a, b, i);
        all += mine;
        most = max(most, mine);
    }
#pragma unroll
    for (int d = 1; d < 64; d *= 2) { all += __shfl_xor(all, d); most = max(most, __shfl_xor(most, d)); }
    // rows like this one that make up the launch's work, about: a long row among short ones has more of the chip
    int rows = a.split_nb * a.split_ng;
    if (a.seqlens && a.split_nb > 1) {
        auto size = [&](int row) __attribute__((always_inline)) { const float n = (float)max(1, min(a.Sq, a.seqlens[row])); return a.window > 0 ? n : n * n; };
        float sum = 0.0f;
        for (int i = lane; i < a.split_nb; i += 64) sum += size(a.split_b0 + i);
#pragma unroll
        for (int d = 1; d < 64; d *= 2) sum += __shfl_xor(sum, d);
        rows = (int)fminf((float)a.split_ng * sum / size(b), 0x1p14f);
    }
    int steps = a.split_steps, cost = (rows * a.split_slots + 255) / 256 * (steps + 3);
    auto consider = [&](int rounds, int x) __attribute__((always_inline)) { if (rounds * (x + 3) < cost) { cost = rounds * (x + 3); steps = x; } };
    consider((rows * blocks + 255) / 256, max(most, 1));
    for (int k = 1; k <= 4; ++k) {
        const int n = min(a.split_slots, k * 256 / max(rows, 1)) - blocks;       // (each block may leave one part that is not full)
        if (n > 0) consider(k, max(1, (all + n - 1) / n));
    }
    steps = __builtin_amdgcn_readfirstlane(steps);
    int first = 0;
    for (int i0 = 0; i0 < blocks; i0 += 64) {
        if (blocks > 64) mine = i0 + lane < blocks ? split_walk_steps(a, b, i0 + lane) : 0;
        const int n = i0 + lane < blocks ? max(1, (mine + steps - 1) / steps) : 0;
        int upto = n;
#pragma unroll
        for (int d = 1; d < 64; d *= 2) { const int x = __shfl_up(upto, d); upto += lane >= d ? x : 0; }
        const uint64_t past = __builtin_amdgcn_ballot_w64(first + upto > slot);
        if (past) {
            const int i = __builtin_ctzll(past), parts = __builtin_amdgcn_readlane(n, i), number = slot - (first + __builtin_amdgcn_readlane(upto, i) - parts);
            if (number == 0 && threadIdx.x == 0) {         // (for the sum)
                a.split_plan[2 * (bg * blocks + i0 + i)] = slot;
                a.split_plan[2 * (bg * blocks + i0 + i) + 1] = parts;
            }
            return {i0 + i, number, steps};
        }
        first += __builtin_amdgcn_readlane(upto, 63);
    }
    return {-1, 0, 0};
}
// SHORT: padded rows or packed documents (an instantiation: 1024 rows without either 2 us slower with both)
template <bool SHORT>
__global__ __launch_bounds__(512, 2) void attn_f32_split_dkdv_kernel(const KArgs a) {
    extern __shared__ __attribute__((aligned(1024))) char f32_split_lds[];
    char *const smem = f32_split_lds;
    using C = F32Split;
    const F32Ptrs t = f32_ptrs(a);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, half = lane >> 5;
    int bid = blockIdx.x;
    const int g = bid % a.split_ng + a.split_g0; bid /= a.split_ng;
    const int bi = bid % a.split_nb, slot = bid / a.split_nb;
    const int b = rotated_batch_row(bi, slot, a.split_nb) + a.split_b0;
    const int64_t bg = split_row_of(a, b, g);
    const SplitPart part = split_part<SHORT>(a, b, bg, slot, lane);
    const int block = part.block;
    if (SHORT && block < 0) return;
    const int J0 = C::kKeys * block, j0 = J0 + 32 * (w & 3), key = j0 + l32;
    const int nt = (a.Skv + 31) / 32, nqt = (a.Sq + 31) / 32;
    const F32TileSpan span = f32_tiles_of_keys(a, 0, b, J0, C::kKeys, lane);
    const int t_hi = __builtin_amdgcn_readfirstlane(span.t_hi), t_lo = span.t_lo;
    const int all = ((t_hi - t_lo + 1) >> 1) * a.r;
    const int s0 = part.number * part.steps, n_steps = max(0, min(part.steps, all - s0));
    float *const partial = a.split_partial ? a.split_partial + (bg * a.split_slots + slot) * (2 * C::kKeys * kD) : nullptr;

    const char *const qrec = a.split_q + bg * a.r * nqt * C::kQRecord;
    const uint32_t lds = lds_addr(smem);
    auto request = [&](int step) __attribute__((always_inline)) {
        const int s = s0 + step, tile = min(t_lo + 2 * (s / a.r) + (w >> 2), nqt - 1);
        const char *src = qrec + ((int64_t)(s % a.r) * nqt + tile) * C::kQRecord;
        const uint32_t dst = lds + ((step & 1) * 2 + (w >> 2)) * C::kQRecord;
        split_copy(dst + (w & 3) * C::kWaveCopy, src + (w & 3) * C::kWaveCopy, lane);
        if ((w & 3) == 3) lds_dma4(dst + C::kStatOff, src + C::kStatOff, (uint32_t)(lane * 4));
    };
    // the rows from `lim` on do not see the lane's key: they do not exist, or belong to a later document (found once: with the document starts read per tile and every
    // tile masked, the backward of 4096 tokens in documents of 100 490 us instead of 475, of 400 672 instead of 639)
    int lim = span.row_lim, all_see = lim;                 // (all_see: no key of the wavefront has less)
    if (SHORT && a.doc_start) {
        const int32_t *row = a.doc_start + (int64_t)b * a.Sq;
        int lo = min(key, lim), hi = max(lo, min(lim, 32 * t_hi));
        while (__builtin_amdgcn_ballot_w64(lo < hi) != 0ull) {
            const int x = (lo + hi) >> 1;
            const bool past = row[min(x, a.Sq - 1)] > key;
            if (lo < hi) { if (past) hi = x; else lo = x + 1; }
        }
        lim = all_see = lo;
#pragma unroll
        for (int d = 1; d < 32; d *= 2) all_see = min(all_see, __shfl_xor(all_see, d));
    }
    all_see = __builtin_amdgcn_readfirstlane(all_see);
    if (n_steps > 0) request(0);
    // numbers the split does not take, among the block's keys or the rows of the walk
    uint32_t bad = 0;
    if (n_steps > 0) {
        const int ta = t_lo + 2 * (s0 / a.r), tb = min(t_hi, t_lo + 2 * ((s0 + n_steps - 1) / a.r + 1)), per = tb - ta;
        for (int i = tid; i < per * a.r; i += 64 * C::kWaves) bad |= a.split_q_bad[(bg * a.r + i / per) * nqt + ta + i % per];
        if (tid < 4 && J0 / 32 + tid < nt) bad |= a.split_kv_bad[bg * nt + J0 / 32 + tid];
    }
    bf16x8 kf[4][3], vf[4][3];     // B operands of S and dP
    {
        const char *kv = a.split_kv + (bg * nt + min(j0 / 32, nt - 1)) * C::kKvRecord;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                kf[ks][p] = *reinterpret_cast<const bf16x8 *>(kv + p * C::kPlane + plane_chunk(l32, 2 * ks + half));
                vf[ks][p] = *reinterpret_cast<const bf16x8 *>(kv + (3 + p) * C::kPlane + plane_chunk(l32, 2 * ks + half));
            }
    }
    // what does not fit the registers stays in LDS: K's last term and an eighth of its second, two and a half of V's, one copy for a key block's two wavefronts
    const SplitKept kept{lds + C::kKeptOff + (w & 3) * C::kKeptKeys + lane * 16};
    auto kept_k = [](int p, int ks) { return p == 2 ? ks : p == 1 && ks == 3 ? 14 : kInRegister; };
    auto kept_v = [](int p, int ks) { return p >= 1 ? 4 * p + ks : ks >= 2 ? 10 + ks : kInRegister; };
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            if (!(w >> 2) && kept_k(p, ks) >= 0) kept.put(kept_k(p, ks), kf[ks][p]);
            if ((w >> 2) && kept_v(p, ks) >= 0) kept.put(kept_v(p, ks), vf[ks][p]);
        }
    wait_vmcnt<0>();
    if (__syncthreads_or(bad != 0)) {
        for (int k = 0; k < 4 && J0 + 32 * k < a.Skv; ++k) {
            const F32TileSpan own = f32_tiles_of_keys(a, 0, b, J0 + 32 * k, 32, lane);
            const F32PairWalk walk{t_lo, t_hi, s0, 2 * n_steps, own.t_lo, own.t_hi};
            float *out = partial ? partial + 32 * k * kD : nullptr;
            f32_dkdv_keys<C::kWaves>(a, smem, g, b, J0 + 32 * k, walk, out, out ? out + C::kKeys * kD : nullptr);
            __syncthreads();
        }
        return;
    }
    f32x16 dk[2], dv[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) { dk[0][i] = dk[1][i] = 0.0f; dv[0][i] = dv[1][i] = 0.0f; }
    const int kv_len = a.seqlens ? min(a.Skv, a.seqlens[b]) : a.Skv;
    const int weff = a.window ? a.window : 0x3fffffff;
    TileLaneOffsets at = tile_offsets_at(make_tile_offsets(lane), lds + (w >> 2) * C::kQRecord);
    uint32_t stat = lds + (w >> 2) * C::kQRecord + C::kStatOff + 16 * half;
    const float c = a.scale_log2;
    wait_vmcnt<0>();
    for (int step = 0; step < n_steps; ++step) {
        split_arrive();
        if (step + 1 < n_steps) request(step + 1);
        const int tile = t_lo + 2 * ((s0 + step) / a.r) + (w >> 2), q0 = 32 * tile;
        // (tiles below the wavefront's own keys see none of them)
        if (tile < t_hi && q0 + 31 >= j0 && q0 - weff < j0 + 31 && j0 < kv_len) {
            f32x16 s, dp;
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = dp[i] = 0.0f;
            split_rows_product<0, true>(s, at, kf, kept, kept_k, SplitNoWork{});               // rows = queries, lane = key
#pragma unroll
            for (int a4 = 0; a4 < 4; ++a4) {
                const f32x4 l2 = lds_load128f(stat, 128 + 32 * a4);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[4 * a4 + e] = fmaf(s[4 * a4 + e], c, -l2[e]);
            }
            // dP; behind its MFMAs the weights, where all are visible and normal, and the terms of their first half
            constexpr int kG = C::kTerms * C::kPlane;
            bf16x8 f[2][3];
            SplitSteps cut;
            auto cut_first = [&](int i) __attribute__((always_inline)) {
                if (i >= 12) cut.step(s, 0, i - 12);
                if (i == 23) cut.take(f[0]);
            };
            const bool interior = j0 + 31 <= q0 && q0 + 31 - weff < j0 && j0 + 32 <= kv_len && q0 + 32 <= all_see;
            if (interior && split_weights_normal(s)) {
                split_rows_product<kG, true>(dp, at, vf, kept, kept_v, [&](int i) __attribute__((always_inline)) {
                    if (i < 16) s[i] = split_weight(s[i]);
                    cut_first(i);
                });
            } else {
                split_any_weights(s);
                if (!interior) {
                    // visible: 0 <= row - key < width (hidden from the compiler, which would keep sixteen lane-dependent numbers for it)
                    int first = q0 + 4 * half;
                    asm volatile("" : "+v"(first));
                    const unsigned width = key < kv_len ? (unsigned)max(0, min(weff, lim - key)) : 0u;
#pragma unroll
                    for (int i = 0; i < 16; ++i) s[i] = (unsigned)(first - key + crow(i, 0)) < width ? s[i] : 0.0f;
                }
                split_rows_product<kG, true>(dp, at, vf, kept, kept_v, cut_first);
            }
            // dV^T[d][key] += dO^T[d][row] P[row][key]: the second half of P is cut behind the first MFMAs, the first of dS behind the others
#pragma unroll
            for (int a4 = 0; a4 < 4; ++a4) {
                const f32x4 nd = lds_load128f(stat, 32 * a4);
#pragma unroll
                for (int e = 0; e < 4; ++e) dp[4 * a4 + e] = s[4 * a4 + e] * (dp[4 * a4 + e] + nd[e]);
            }
            split_cols_product<kG>(dv, at, f, [&](int i) __attribute__((always_inline)) {
                if (i < 12) cut.step(s, 1, i); else cut.step(dp, 0, i - 12);
                if (i == 11) cut.take(f[1]);
                if (i == 23) cut.take(f[0]);
            });
            split_cols_product<0>(dk, at, f, [&](int i) __attribute__((always_inline)) {  // dK^T[d][key] += Q^T[d][row] dS[row][key]
                if (i < 12) cut.step(dp, 1, i);
                if (i == 11) cut.take(f[1]);
            });
        }
        const uint32_t move = (step & 1) ? (uint32_t)(-2 * C::kQRecord) : (uint32_t)(2 * C::kQRecord);
        tile_offsets_move(at, move);
        stat += move;
    }
    // the two wavefronts of a key block: their shares added, the tiles of even index first
    __syncthreads();
    f32_leave_partial(smem + w * (2 * F32Tile::kBytes), dk, lane);
    f32_leave_partial(smem + w * (2 * F32Tile::kBytes) + F32Tile::kBytes, dv, lane);
    __syncthreads();
#pragma unroll
    for (int pass = 0; pass < 8; ++pass) {
        const int which = pass & 1, k = pass >> 1, r = tid >> 4, ch = tid & 15, j = J0 + 32 * k + r;
        f32x4 x = f32_partial(smem + which * F32Tile::kBytes, 2 * F32Tile::kBytes, k, r, ch);
        const f32x4 y = f32_partial(smem + which * F32Tile::kBytes, 2 * F32Tile::kBytes, k + 4, r, ch);
        const float mul = (which == 0 && !partial ? a.scale : 1.0f) * kSplitUnscale;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = (x[e] + y[e]) * mul;
        if (j < a.Skv) {
            if (partial) {
                *reinterpret_cast<f32x4 *>(partial + (which * C::kKeys + 32 * k + r) * kD + 4 * ch) = x;
            } else {
                const Strides &st = which == 0 ? a.dks : a.dvs;
                *reinterpret_cast<f32x4 *>((which == 0 ? t.dk : t.dv) + (int64_t)b * st.b + (int64_t)g * st.h + (int64_t)j * st.s + 4 * ch) = x;
            }
        }
    }
}

// The parts of every key block, added in their order (and dSinks in the first blocks).  One thread per 16-byte chunk.
__global__ __launch_bounds__(256) void attn_f32_split_reduce_kernel(const KArgs a, int heads) {
    __shared__ float red[1024];
    if ((int)blockIdx.x < heads) { dsinks_of_head<256>(a, blockIdx.x, red); return; }
    using C = F32Split;
    const F32Ptrs t = f32_ptrs(a);
    const int64_t rows = (int64_t)a.split_nb * a.split_ng * a.Skv, idx = (int64_t)(blockIdx.x - heads) * 256 + threadIdx.x;
    if (idx >= 2 * rows * 16) return;
    const int which = idx >= rows * 16, ch = (int)(idx & 15);
    const int64_t row = (idx - (int64_t)which * rows * 16) >> 4;
    const int key = (int)(row % a.Skv), bg = (int)(row / a.Skv), block = key / C::kKeys;
    const int g = a.split_g0 + bg % a.split_ng, b = a.split_b0 + bg / a.split_ng;
    int slot = 0, n;
    if (a.split_plan) {
        const int *plan = a.split_plan + 2 * ((int64_t)bg * ((a.Skv + C::kKeys - 1) / C::kKeys) + block);
        slot = plan[0];
        n = plan[1];
    } else {
        for (int i = 0; i < block; ++i) slot += split_block_parts(a.Sq, a.window, a.r, i, a.split_steps);
        n = split_block_parts(a.Sq, a.window, a.r, block, a.split_steps);
    }
    const float *src = a.split_partial + ((int64_t)bg * a.split_slots + slot) * (2 * C::kKeys * kD) + (which * C::kKeys + key % C::kKeys) * kD + 4 * ch;
    f32x4 x = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int i = 0; i < n; ++i) {
        const f32x4 y = *reinterpret_cast<const f32x4 *>(src + (int64_t)i * (2 * C::kKeys * kD));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] += y[e];
    }
    const float mul = which == 0 ? a.scale : 1.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] *= mul;
    const Strides &st = which == 0 ? a.dks : a.dvs;
    *reinterpret_cast<f32x4 *>((which == 0 ? t.dk : t.dv) + (int64_t)b * st.b + (int64_t)g * st.h + (int64_t)key * st.s + 4 * ch) = x;
}

}  // namespace gptoss
