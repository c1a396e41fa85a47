// C ABI of the gfx950 GPT-OSS attention library (declared in include/gptoss_attn.h):
// host-side argument validation, launch geometry, and the kernel launches.
// No torch headers, no allocation; the only process-wide state is per-device values that are written once
// (compute-unit count, the LDS attributes of kernels that need more than 64 KB, the address of the built-in scratch).
#include <hip/hip_runtime.h>

#include <atomic>

#include "../../include/gptoss_attn.h"
#include "attn_bwd.h"
#include "attn_bwd_dkdv64.h"
#include "attn_bwd_window.h"
#include "attn_common.h"
#include "attn_decode.h"
#include "attn_f32.h"
#include "attn_f32_split.h"
#include "attn_fwd.h"
#include "attn_fwd_pipe.h"
#include "attn_fwd_window.h"
#include "doc_start.h"
#include "mfma_rate.h"

using namespace gptoss;

namespace {

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// A tensor's rows must start on 16-byte boundaries for the 128-bit accesses.
int check_tensor(const void *p, const gptoss_attn_strides &s, int elem_bytes, int D) {
    if (!p) return GPTOSS_ATTN_ERR_NULL_TENSOR;
    if (!aligned16(p)) return GPTOSS_ATTN_ERR_ALIGNMENT;
    const int64_t per16 = 16 / elem_bytes;
    if (s.b % per16 || s.h % per16 || s.s % per16) return GPTOSS_ATTN_ERR_ALIGNMENT;
    if (s.s < D || s.s > (1 << 24)) return GPTOSS_ATTN_ERR_STRIDE;   // 64 rows x stride is kept in 32 bits by the tile copies
    return GPTOSS_ATTN_OK;
}

Strides cvt(const gptoss_attn_strides &s) { return Strides{s.b, s.h, s.s}; }

// A window that reaches back past the first key from every query position is no window: such a
// call is the full-causal layer and takes exactly its kernels (same bits).
// (Not decidable on the host when the query offset lives in device memory.)
int effective_window(const gptoss_attn_params *p) {
    if (p->q_offset_dev) return p->window;
    return (p->window > 0 && (int64_t)p->window >= (int64_t)p->Sq + p->q_offset) ? 0 : p->window;
}

// Scratch layout: the fp32 row statistics (-delta, then lse * log2 e: 8 bytes per row, rounded up to 16
// bytes), the same statistics in split form (16 bytes per row), then the dK/dV partial sums.
size_t fp32_stats_bytes(const gptoss_attn_params *p) {
    const size_t n = (size_t)2 * sizeof(float) * (size_t)p->B * (size_t)p->H * (size_t)p->Sq;
    return (n + 15) & ~(size_t)15;
}

// Element types of the sink logits and of their gradient (the parameter block has fp32 for both).
struct SinkTypes { bool sinks_bf16 = false, dsinks_bf16 = false; };

KArgs make_args(const gptoss_attn_params *p, SinkTypes ty) {
    KArgs a{};
    a.sinks_bf16 = ty.sinks_bf16;
    a.dsinks_bf16 = ty.dsinks_bf16;
    a.q = static_cast<const bf16 *>(p->q);
    a.k = static_cast<const bf16 *>(p->k);
    a.v = static_cast<const bf16 *>(p->v);
    a.sinks = p->sinks;
    a.seqlens = p->seqlens;
    a.doc_start = p->doc_start;
    a.o = static_cast<bf16 *>(p->o);
    a.lse = p->lse;
    a.d_o = static_cast<const bf16 *>(p->d_o);
    a.dq = static_cast<bf16 *>(p->dq);
    a.dk = static_cast<bf16 *>(p->dk);
    a.dv = static_cast<bf16 *>(p->dv);
    a.dsinks = p->dsinks;
    a.delta = p->delta;
    a.split = reinterpret_cast<u32x4 *>(reinterpret_cast<char *>(p->delta) + fp32_stats_bytes(p));
    a.qs = cvt(p->q_stride); a.ks = cvt(p->k_stride); a.vs = cvt(p->v_stride); a.os = cvt(p->o_stride);
    a.dos = cvt(p->do_stride); a.dqs = cvt(p->dq_stride); a.dks = cvt(p->dk_stride); a.dvs = cvt(p->dv_stride);
    a.B = p->B; a.H = p->H; a.G = p->G; a.Sq = p->Sq; a.Skv = p->Skv;
    a.r = p->H / p->G;
    a.window = effective_window(p);
    a.q_offset = p->q_offset_dev ? 0 : p->q_offset;
    a.q_offset_dev = p->q_offset_dev;
    a.scale = p->scale;
    a.scale_log2 = p->scale * kLog2e;
    a.dkdv_parts = 1;
    a.dkdv_slots = 0;
    a.dkdv_steps = 0;
    a.kv_splits = 1;
    a.fwd_partial = nullptr;
    a.chunk_blocks = 0;
    a.dsink_partial = nullptr;
    a.boundary_partial = nullptr;
    a.split_kv = a.split_q = nullptr;
    a.split_kv_bad = a.split_q_bad = nullptr;
    a.split_steps = a.split_slots = 0;
    a.split_partial = nullptr;
    a.split_plan = nullptr;
    a.split_b0 = a.split_nb = a.split_g0 = a.split_ng = a.split_tiles = 0;
    return a;
}

int hpb_for(int r) { return r >= 4 ? 4 : (r >= 2 ? 2 : 1); }

// 32-row query blocks per wavefront in the forward and dQ kernels.  Two blocks (64 rows)
// halve the LDS fragment traffic per MFMA and win on long key loops (full-causal layers);
// one block (32 rows, three wavefronts per SIMD) wastes less of the narrow band of a
// sliding-window layer and hides its short loops' latency better.
int query_blocks_for(int window) { return (window > 0 && window <= 1024) ? 1 : 2; }

// 32-key blocks per wavefront in the dK/dV kernel
constexpr int kDkdvNB = 1;
constexpr int kDkdvWaves = 4;                        // wavefronts per dK/dV workgroup
constexpr int kDkdvKeys = 32 * kDkdvNB * kDkdvWaves; // keys per dK/dV workgroup

// More key blocks than are cut into equal shares by their number alone.
bool many_key_blocks(const gptoss_attn_params *p) { return (int64_t)p->G * p->B * ((p->Skv + kDkdvKeys - 1) / kDkdvKeys) > 512; }

// Workgroups per key block in the dK/dV kernel.  One workgroup per (batch, KV head, 128 keys) fills
// the 256 CUs (two workgroups each) only from S = 16384 on, and the causal triangle makes the first
// key blocks many times longer than the last; shorter problems cut each key block's query tiles into
// slices so that there are about a thousand workgroups, and sum the slices' fp32 partials afterwards.  A slice
// keeps at least four query tiles of a sliding-window layer (windows of up to 321 keys stay whole, wider ones are cut) and at least
// eight (query tile, head) steps of a full-causal one, which may be a single tile.  Up to 512 blocks the count is rounded
// up (B = 2, S = 383: 78 us uncut, 25 + 5 us in six slices; unpadded short rows then take pieces of other lengths in the same scratch,
// dkdv_pieces_for).  Between 512 and 1024 blocks the first key block of a long row (4096 rows and more) is still longer than the average
// compute unit's share: two slices; a right-padded batch counts half, because its shorter rows leave the longest one alone (dK/dV of B = 4,
// S = 4096, lengths 3309 / 1968 / 1554 / 4079: 715 us uncut, 589 in two slices; B = 2, S = 8192 / 4000: 1437 and 1216).  Several rows of
// 1280 tokens and more (padded: 1024) get the same scratch, for pieces by the walks' lengths (Dkdv64Plan), which cut only the longest
// walks: whole backward and forward of 5 x 1600 564 -> 514 us, 6 x 1500 610 -> 584, 3 x 3000 1074 -> 995, 7 x 1417 645 and 646, 8 x 1300
// 611 -> 602; but 9 x 1100 536 -> 547.  Packed rows: a walk ends with its document, so the longest document's first blocks stand out more,
// and the host does not see the documents: four slices from 256 to 768 blocks of rows of 4096 keys and more.  Whole backward of one row of
// 64 query heads, two slices / four, documents of up to 1500 tokens, up to 4096, 1500 to 6000, and ONE: 8192 tokens 367 / 373, 602 / 568,
// 994 / 924, 1683 / 1689 us; 12288 (768 blocks) 554 / 557, 970 / 963, 1296 / 1254, 3826 / 3712; beyond the line 14000 571 / 593, 872 / 866,
// 1508 / 1501, 4913 / 4875 and 16384 687 / 711, 928 / 941, 1623 / 1631, 6636 / 6690.  (Two rows of 4096, 512 blocks, would rather have two:
// 340 / 359, 526 / 513, 864 / 902, 904 / 919.)
int dkdv_parts_for(const gptoss_attn_params *p, bool padded, bool packed) {
    if (p->dtype == GPTOSS_ATTN_FP32) {
        // A workgroup per 32 keys, two per compute unit at a time.  Up to four slices and a thousand workgroups, so that the long first key
        // blocks of a row do not decide the time; more where that is not two per unit of a 256-CU part: the longest walk, 1.2 us a step, is
        // all there is to such a launch (backward, us in a graph, at most four slices / these: 8 heads on one KV head 300 tokens 55 / 38,
        // 1000 122 / 76, 2 x 1000 134 / 111, on two 1000 83 / 73 (with a thousand workgroups here too 82), 64 on eight 150 45 / 36).  A
        // window's walk is cut by the same rule, into three or more: of 128 8 heads on one 400 tokens 73 / 34, 64 on eight 500 95 / 82;
        // into two 900 108 / 110.
        const int64_t blocks = (int64_t)p->G * p->B * ((p->Skv + 31) / 32), all = (p->Sq + 31) / 32;
        const int window = effective_window(p);
        const int64_t tiles = window > 0 && (window + 62) / 32 + 1 < all ? (window + 62) / 32 + 1 : all;        // that see a block
        int64_t parts = window > 0 ? 1 : 1024 / blocks;
        if (parts > 4) parts = 4;
        if (512 / blocks > (window > 0 ? 2 : parts)) parts = 512 / blocks;
        if (parts > tiles * (p->H / p->G) / 8) parts = tiles * (p->H / p->G) / 8;
        if (parts > tiles) parts = tiles;
        if (parts > 16) parts = 16;
        return parts < 1 ? 1 : (int)parts;
    }
    if (p->dtype != GPTOSS_ATTN_BF16) return 1;
    const int64_t blocks = (int64_t)p->G * p->B * ((p->Skv + kDkdvKeys - 1) / kDkdvKeys);
    const int window = effective_window(p);
    const int64_t rows_seen = window > 0 ? (int64_t)kDkdvKeys + window - 1 : (int64_t)p->Sq;
    const int64_t tiles = ((rows_seen < p->Sq ? rows_seen : p->Sq) + 63) / 64;
    // Rows of one length of up to 1024 tokens: fewer shares, each with 64 KB of partial sums that are written and read again (forward + backward, us,
    // shares for a thousand workgroups / for 768: 8 x 300 tokens 112.6 / 105.5, 6 x 400 118.7 / 112.3, 5 x 621 167.6 / 161.4, 3 x 700 135 / 129, 2 x 900
    // 135 / 131, 4 x 1000 243 / 232; 1 x 1500 160 / 159, but 3 x 1200 226 / 232; padded 5 x 621 117 / 121, 2 x 1555
    // 151 / 155; the 64-key kernel's 1 x 2500 303 / 302, but 2 x 3001 would get two shares instead of three).
    const int64_t workgroups = p->Skv <= 1024 && window == 0 && !padded && !packed ? 768 : 1024;
    int64_t parts = (workgroups + blocks - 1) / blocks;
    // (rows that attn_bwd_dkdv64_kernel takes)
    const bool by_lengths = p->B > 1 && window == 0 && p->Sq == p->Skv && p->q_offset == 0 && !p->q_offset_dev;
    if (many_key_blocks(p)) parts = p->Sq >= (!by_lengths ? 4096 : padded ? 1024 : 1280) && (padded && p->B > 1 ? blocks / 2 : blocks) < 1024 ? 2 : 1;
    if (packed && window == 0 && p->Sq >= 4096 && blocks >= 256 && blocks <= 768 && parts < 4) parts = 4;
    const int64_t steps = window > 0 ? tiles / 4 : tiles * (p->H / p->G) / 8;
    if (parts > steps) parts = steps;
    if (parts > tiles) parts = tiles;
    if (parts > 8) parts = 8;
    return parts < 1 ? 1 : (int)parts;
}

// Pieces of the 32-key kernel's walks (DkdvPieces) instead of equal slices of whole tiles: the shortest ones, of four steps or more, of which
// there are no more than 512 (two workgroups per compute unit of a 256-CU part: in a launch of their own all run at once and end together) and than the
// scratch has slots for.  Taken for one row where they are no longer than the longest slice, for several (whose tiles a piece that starts elsewhere does
// not find in L2) where they are shorter.  dK/dV and the sum of its parts, us, slices / pieces: 2 x 383 tokens 29.8 / 26.9, 2 x 621 47.0 / 37.5,
// 1 x 1024 47.0 / 41.5, 1 x 1900 95 / 83; not taken: 4 x 1000 (pieces as long as the slices) whole call 227 / 234, 3 x 1200 (longer)
// 234 / 243, 4 x 160 (longer) 47 / 52.  Nor for padded or packed rows, whose slices follow the lengths: 1500 and 700 tokens 194 / 210, documents of
// 700, 600 and 500 150 / 164.  From 2048 tokens on the 64-key kernel takes over.
void dkdv_pieces_for(const gptoss_attn_params *p, KArgs &a) {
    if (a.dkdv_parts == 1 || p->seqlens || p->doc_start || effective_window(p) > 0 || p->Sq != p->Skv || p->q_offset != 0 || p->q_offset_dev ||
        p->Skv >= 2048)
        return;
    const int blocks = (p->Skv + kDkdvKeys - 1) / kDkdvKeys, tiles = (p->Sq + kTile - 1) / kTile;
    const int64_t rows = (int64_t)p->G * p->B, slots = (int64_t)a.dkdv_parts * p->Skv / kDkdvKeys;       // (of a row)
    const int64_t most = slots < 512 / rows ? slots : 512 / rows;
    const int slice = (tiles + a.dkdv_parts - 1) / a.dkdv_parts * a.r;
    if (most < blocks) return;
    const int64_t all = (int64_t)blocks * (tiles + 1 - blocks) * a.r;                                    // steps of a row: no shorter pieces than all / most
    for (int steps = (int)(all > 4 * most ? (all + most - 1) / most : 4); steps < slice + (p->B == 1); ++steps) {
        int n = 0;
        for (int i = 0; i < blocks; ++i) n += DkdvPieces::of(a.Sq, a.r, steps, i);
        if (n > most) continue;
        a.dkdv_steps = steps;
        a.dkdv_slots = n;
        return;
    }
}

// workgroups of the forward / dQ launch: (KV head, chunk of HPB query heads, batch, query tile)
int64_t q_outer_grid(const KArgs &a, int hpb, int qb) {
    const int bm = 32 * qb * (4 / hpb);
    const int n_hc = (a.r + hpb - 1) / hpb;
    return (int64_t)a.G * n_hc * a.B * ((a.Sq + bm - 1) / bm);
}
// 32-row query blocks per wavefront of the dQ kernel.  Short problems: 64-row workgroups (two per compute unit) would be few and
// uneven (the key loops grow with the row index); 32-row wavefronts make twice as many, three per SIMD (measured, full causal, B = 1: dQ
// 0.077 -> 0.066 ms at S = 2048, 0.240 -> 0.218 at S = 4096, equal from S = 8192 on, 6 % slower at S = 16384).
int compute_units();
int dq_query_blocks(const KArgs &a) {
    const int qb = query_blocks_for(a.window);
    return qb == 2 && q_outer_grid(a, hpb_for(a.r), 2) <= 4 * (int64_t)compute_units() ? 1 : qb;
}
// Workgroups of attn_bwd_dkdv_kernel.
int64_t dkdv_grid(const KArgs &a) {
    return (int64_t)a.G * a.B * (a.dkdv_steps ? a.dkdv_slots : a.dkdv_parts * ((a.Skv + kDkdvKeys - 1) / kDkdvKeys));
}
bool window_single_pass(const gptoss_attn_params *p);
// Full-causal self-attention goes to attn_bwd_dkdv64_kernel (64 keys per wavefront, one wavefront per SIMD)
// when the shape is the one it is written for (bf16, no window, no offset, Sq == Skv; right-padded batch rows and packed
// documents are fine) and there is enough of it: more than
// 512 key blocks of 128 (then key blocks are whole: at least 257 workgroups of 256 keys, and the same bits as the 32-key
// kernel), or rows of 2048 keys or more that the host cuts into `parts` slices anyway (the same number of slices as the
// 32-key kernel would get, so the scratch is the same; -15 % at S = 2048 ... 8192).
// (The kernel walks Q, dO and the row statistics of one KV head's group of query heads with 32-bit byte
// offsets from the group's first row: head strides must not be negative and the group's span must stay
// below 2^31 bytes; anything else takes the 32-key kernel, and so does what fits both_route.)
bool walk_fits_32_bits(const gptoss_attn_strides &s, int64_t heads, int64_t rows) {
    return s.h >= 0 && ((heads - 1) * s.h + rows * s.s) * 2 < ((int64_t)1 << 31);
}
bool dkdv64_shape(const gptoss_attn_params *p, int parts) {
    const int64_t blocks = (int64_t)p->G * p->B * ((p->Skv + kDkdvKeys - 1) / kDkdvKeys);
    const int64_t heads = p->H / p->G;
    if (!walk_fits_32_bits(p->q_stride, heads, p->Sq) || !walk_fits_32_bits(p->do_stride, heads, p->Sq) ||
        heads * p->Sq * 16 >= ((int64_t)1 << 31))
        return false;
    return p->dtype == GPTOSS_ATTN_BF16 && effective_window(p) == 0 && p->q_offset == 0 && !p->q_offset_dev && p->Sq == p->Skv &&
           p->Sq >= kTile && (blocks > 512 || (parts > 1 && p->Skv >= 2048));
}

// dQ and dK/dV in one launch (attn_bwd_both_kernel), behind one for the row statistics, instead of one after the other.  `a` has the
// backward's dkdv_parts; gets its pieces.
// What it saves is the end of the first launch, where units wait for its longest walks, and the start of the second; what it adds is the
// statistics' own launch, 4 us.  So the line is a number of rounds of workgroups, two per compute unit of a 256-CU part.  Six where the
// same two kernels would run one after the other (dQ's with 32-row wavefronts), as an end is little beside so many rounds: whole backward,
// us in a graph, one after the other / side by side (workgroups), 64 heads on 8 KV heads 512 tokens 38 / 31 (480), 2 x 383 43 / 34 (656),
// 1500 114 / 91 (1248), 2 x 1500 184 / 174 (2656), padded 4 x 1000 143 / 138 (3072).  Three where the other side has
// attn_bwd_dkdv64_kernel, whose steps are cheaper: 8 heads on one 4000 155 / 112 (506), 10000 495 / 441 (1258), 32 on four 3000 188 / 178
// (1520), but 2 x 2048 152 / 160 (2048); documents of 500 to 2500 143 / 141 (1520), 215 / 219 (2048).
// Padded rows of 2048 tokens and more stay apart: attn_bwd_dkdv64_kernel reads no row of the padding, attn_bwd_dkdv_kernel those that
// share a tile with rows that count.
// Which of them starts first: pieces, and slices under a window, are of one length, and what starts last ends last: dQ's last
// walks are short (dK/dV's / dQ's first: 64 on 8 2 x 383 34 / 40, 1500 91 / 101; window 200 98 / 124).  Where the walks of both shrink along the row the
// longest one starts first: a step (query tile, head) of dK/dV takes 1.9 us, a key tile of dQ 1.1 (8 on two, slices of half a
// row's steps, 4000 101 / 94, 8000 289 / 261, padded 4 x 1000 51 / 48; on one, of a row's, 4000 112 / 124, but 5000 171 / 151).
constexpr int64_t kBothRound = 512;
struct BothRoute { bool taken, dq_first; };
BothRoute both_route(const gptoss_attn_params *p, KArgs &a) {
    if (p->dtype != GPTOSS_ATTN_BF16 || a.r < 4 || window_single_pass(p) || dq_query_blocks(a) != 1) return {false, false};
    if (p->seqlens && p->Skv >= 2048) return {false, false};
    dkdv_pieces_for(p, a);
    const int64_t rounds = dkdv64_shape(p, a.dkdv_parts) ? 3 : 6;
    const int64_t q_tiles = (p->Sq + kTile - 1) / kTile, k_tiles = (p->Skv + kTile - 1) / kTile;
    const int64_t slice = (q_tiles + a.dkdv_parts - 1) / a.dkdv_parts * a.r;
    return {q_outer_grid(a, 4, 1) + dkdv_grid(a) <= rounds * kBothRound, !a.dkdv_steps && a.window == 0 && 11 * k_tiles > 19 * slice};
}

bool dkdv64_route(const gptoss_attn_params *p, int parts) {
    if (!dkdv64_shape(p, parts)) return false;
    KArgs a = make_args(p, {});
    a.dkdv_parts = parts;
    return parts == 1 || !both_route(p, a).taken;
}

// The hand-pipelined forward kernel (attn_fwd_pipe.h) takes full-causal rows whose groups of query heads fill its four
// wavefronts; self-attention of whole tiles without padding or packing has an instantiation of its own.
bool fwd_pipe_route(const gptoss_attn_params *p) {
    return p->dtype == GPTOSS_ATTN_BF16 && effective_window(p) == 0 && (p->H / p->G) % 4 == 0 && p->Skv >= kTile;
}
bool fwd_pipe_plain(const gptoss_attn_params *p) {
    return p->Sq == p->Skv && p->Sq % kTile == 0 && !p->seqlens && !p->doc_start && p->q_offset == 0 && !p->q_offset_dev;
}

// Shares of the keys per query block where the workgroups (64 queries of four heads) are too few to fill the chip (no packing): two per compute
// unit of a 256-CU part, at least eight tiles each, as a share starts and ends and is added.  From the shapes alone, so that the
// scratch (68 KB a workgroup) does not depend on where the queries stand.  us, whole / in shares, 64 heads on 8 KV heads:
//  * New queries on a cache, up to 512 workgroups in three shares and more (35 MB at most): 100 queries on 4096 keys 62 / 30, 300 on 12000
//    167 / 82; two shares that just fill the chip are not worth their sum, 1024 on 8192 134 / 137.
//  * More workgroups than compute units, but not two each, make some units take twice as long as the others (a unit is no faster with
//    two).  On long caches shares end with a full or half full round of two per unit: three for 257 to 341 workgroups (69 MB), two to
//    384 and four for 171 to 192 (52): 1268 queries on 16000 keys 398 / 319, on 4000 97 / 97; 1500 on 9000 228 / 211, on 4000 99 / 101; 704 on 16000
//    219 / 190, on 5000 75 / 77; 400 workgroups 412 / 437, 200 of 32 heads 130 / 143.
//  * Self-attention has more rows to add: up to four groups of four heads from 20 tiles on (8 heads on one KV head 1300 tokens 23.4 / 21.3,
//    4000 60 / 41, but 2 x 1024 19.2 / 20.4, six groups of 1600 28 / 31), and four workgroups per unit from 128 tiles on (69 MB), whose walks differ
//    most: 8200 tokens 117 / 91, 12000 191 / 164 (with two per unit whole), but 4000 60 / 46.
int fwd_pipe_splits(const gptoss_attn_params *p) {
    const bool self = p->Skv <= p->Sq;
    const int64_t groups = (int64_t)p->G * (p->H / p->G / 4) * p->B, wgs = groups * ((p->Sq + kTile - 1) / kTile);
    const int64_t tiles = (p->Skv + kTile - 1) / kTile;
    if (self && (groups > 4 || tiles < 20)) return 1;
    int64_t n = (self && tiles >= 128 ? 1024 : 512) / wgs;
    if (n > tiles / 8) n = tiles / 8;
    if (n > 16) n = 16;
    if (!self && n < 3 && tiles >= 96) {
        if (wgs > 256) n = wgs <= 1024 / 3 ? 3 : wgs <= 768 / 2 ? 2 : 1;
        else n = wgs <= 768 / 4 && tiles >= 128 ? 4 : 1;
        return (int)n;
    }
    return n < (self ? 2 : 3) ? 1 : (int)n;
}

// The one-pass forward of sliding-window layers (attn_fwd_window.h): a window of 32, 64, 96 or 128 keys, all four wavefronts of
// a workgroup with a head of their own.  Self-attention of whole 32-row blocks without packing has an instantiation of its own.
bool fwd_window_route(const gptoss_attn_params *p) {
    const int w = effective_window(p);
    // lane offsets are 32-bit: up to 160 rows of K / V, 32 of Q and O; the grid's y and z dimensions end at 65535
    const int64_t row_limit = (int64_t)1 << 22;
    if (p->k_stride.s >= row_limit || p->v_stride.s >= row_limit || p->q_stride.s >= row_limit || p->o_stride.s >= row_limit) return false;
    if ((int64_t)(p->H / p->G / 4) * p->B > 65535 || (p->Sq + 31) / 32 > 65535) return false;
    return p->dtype == GPTOSS_ATTN_BF16 && w >= 32 && w <= 128 && w % 32 == 0 && (p->H / p->G) % 4 == 0;
}
bool fwd_window_plain(const gptoss_attn_params *p) {
    return !p->doc_start && p->q_offset == 0 && !p->q_offset_dev && p->Sq == p->Skv && p->Sq % 32 == 0;
}

// A few queries on a long cache (attn_decode.h): all (query, head) pairs of a KV head fit two 32-column blocks.
bool decode_route(const gptoss_attn_params *p) {
    return p->dtype == GPTOSS_ATTN_BF16 && !p->doc_start && (int64_t)p->Sq * (p->H / p->G) <= Decode::kMaxPairs;
}
int64_t decode_keys(const gptoss_attn_params *p) {
    return p->window > 0 && (int64_t)p->window + p->Sq < p->Skv ? (int64_t)p->window + p->Sq : p->Skv;
}
// The keys of a KV head walked by one workgroup of eight wavefronts, no slices to add and one launch less.  Where the cache comes from HBM
// (us a call, sliced / whole, 8 query heads per KV head), B G = 8: 257 keys 12.5 / 10.6, 1024 12.4 / 11.1, 1500 12.4 / 13.6, 2049 12.4 / 16.7;
// B G = 128: 1024 14.1 / 13.0, 2049 20.9 / 20.1, 4096 32.8 / 34.3, 8192 55.7 / 65.5; B G = 256: 1000 20.1 / 17.1; two column blocks, B G =
// 8: 600 12.6 / 11.7, 1000 12.6 / 14.6.  (A cache that is still in the last-level cache moves the line up to 3000 keys, but a decoding step
// reads all layers' weights between two calls on one cache.)  512 groups fill the chip unsliced.
bool decode_whole(const gptoss_attn_params *p) {
    const int64_t groups = (int64_t)p->B * p->G, pairs = (int64_t)p->Sq * (p->H / p->G);
    return groups < 512 && decode_keys(p) <= (pairs > 32 ? 640 : 1024);
}
// Slices of the keys: about two workgroups per compute unit of a 256-CU part (so that the scratch does not depend on the
// device), each wavefront of a slice with a tile of its own at least.
int decode_splits(const gptoss_attn_params *p) {
    if (decode_whole(p)) return 1;
    const int64_t keys = decode_keys(p);
    const int64_t groups = (int64_t)p->B * p->G;
    int64_t n = (512 + groups - 1) / groups;
    const int64_t most = keys / (4 * Decode::kKeys);
    if (n > most) n = most;
    return (int)(n < 1 ? 1 : n);
}

// float32 forward and dQ: wavefronts that share a unit (32 query rows of one head).  Few units: four, so that the chip fills and
// a row's keys are walked four at a time (64 heads, S = 256: forward 15 us; 18 with two, 29 with one); more than 1024: two (S = 1024: 101 us
// forward, 136 dQ; 100 and 136 with four, 121 and 164 with one), and for a window's handful of tiles one (window 128, S =
// 1024: 36 and 47 us; 40 and 53 with two, 49 and 68 with four).
int f32_key_splits(const KArgs &a) {
    const int64_t units = (int64_t)a.B * a.H * ((a.Sq + 31) / 32);
    return units <= 1024 ? 4 : (a.window > 0 && a.window <= 512 ? 1 : 2);
}
int64_t f32_grid(const KArgs &a, int ks) {
    const int64_t units = (int64_t)a.r * a.B * ((a.Sq + 31) / 32);      // per KV head; 4 / ks of them per workgroup
    return (int64_t)a.G * ((units + 4 / ks - 1) / (4 / ks));
}

// ---- float32 on the bf16 matrix pipes (attn_f32_split.h) -----------------------------------------
// Taken where the caller has scratch for the records, four consecutive heads share a KV head (the four units of a workgroup then stand
// at the same rows), the backward for self-attention without an offset, and where it is the faster one: it costs a launch and fills the
// chip with workgroups of eight wavefronts, one per compute unit.  Self-attention takes it in both directions or in neither (with lse of
// the one and S of the other dQ of operands next to a bf16 number was 1.09 times as far from float64 as with the fp32 instruction alone).
// fp32 instruction / this, us in a graph, 64 query heads on 8 KV heads, forward and backward: 320 rows 23 + 82 / 25 + 70, 448 33 + 110 / 31
// + 80, 1024 100 + 310 / 66 + 200, 4096 5320 / 3120; 8 heads on one KV head 2048 rows (128 workgroups) 63 + 249 / 79 + 165; a window is a
// handful of tiles per workgroup, whose start and end then decide: of 128, 320 rows 22 + 88 / 21 + 63, 640 33 + 103 / 35 + 91, 800 (400
// workgroups) 36 + 107 / 39 + 102, 1024 147 / 150; of 383, 800 63 + 220 / 50 + 136; of 64, 448 21 + 69 / 20 + 61, but 640 26 + 74 / 33 + 83
// (windows below 96 would rather have the line at 256 workgroups). Queries on a cache, forward: 256 (128 workgroups) on 2048 80 / 84, on
// 4096 154 / 154, on 16384 600 / 566; 320 on 1024 59 / 48, 1024 on 8192 1121 / 647; with a window of 128, 320 on 16384 23 / 21, 448 26 /
// 22, 576 34 / 36, 256 (128 workgroups) 15 / 21; of 64, 320 17 / 19, 448 21 / 20; of 192, 576 43 / 41; of 400, 800 76 / 56.
bool f32_split_route(const gptoss_attn_params *p, bool bwd) {
    if (p->dtype != GPTOSS_ATTN_FP32 || p->B <= 0 || p->G <= 0 || p->H <= 0 || p->H % p->G || (p->H / p->G) % 4 || p->Skv <= 0) return false;
    const bool self = p->Sq == p->Skv && p->q_offset == 0 && !p->q_offset_dev;       // (both directions take it, or neither)
    if (bwd && !self) return false;
    const int64_t wgs = (int64_t)(p->H / 4) * p->B * (((int64_t)p->Sq + 31) / 32);
    const int window = effective_window(p);
    if (window > 0 && window < 384 && wgs > (!self && window < 160 ? 256 : 400)) return false;
    if (!self && window > 0) return p->Sq >= 192 && wgs >= (window < 96 ? 224 : 160);
    return p->Sq >= 192 && (wgs >= 160 || (wgs >= 128 && p->Skv >= 2048));
}
// Steps per dK/dV workgroup, `rows` batch rows and KV heads at once: the count whose rounds of workgroups take the least time on 256 compute units, one
// workgroup each (so that the scratch does not depend on the device), a workgroup's start and end counted as three steps.  At most four
// rounds: each workgroup of a cut key block leaves 64 KB.  Of the counts from the longest walk's down to four, a thirty-second apart, the smallest
// that needs no more than k rounds is the best of k rounds: found by halving, as the caller asks for the scratch's size and the call itself asks again
// (all counts one by one / so, 1024 tokens 1.1 / 0.4 us, 4096 4.0 / 2.0, 16384 17 / 8).
struct F32SplitParts { int steps, slots; bool cut; };
F32SplitParts f32_split_parts(const gptoss_attn_params *p, int64_t rows) {
    const int window = effective_window(p), r = p->H / p->G, blocks = (p->Skv + F32Split::kKeys - 1) / F32Split::kKeys;
    const int64_t cus = 256;
    int steps[640], n = 0;                                 // (from 2^31 down: 609)
    for (int x = split_block_steps(p->Sq, window, r, 0); n == 0 || x >= 4; x -= 1 + x / 32) steps[n++] = x;
    auto slots_of = [&](int i) {
        int slots = 0;
        for (int k = 0; k < blocks; ++k) slots += split_block_parts(p->Sq, window, r, k, steps[i]);
        return slots;
    };
    F32SplitParts best{steps[0], blocks, false};
    int64_t rounds = (rows * blocks + cus - 1) / cus, best_cost = rounds * (steps[0] + 3);
    for (int first = 0; rounds <= 4; ++rounds) {
        int last = first, slots = 0;                       // the last count of at most so many rounds, from `first` on
        for (int lo = first, hi = n - 1; lo <= hi;) {
            const int mid = (lo + hi) / 2, m = slots_of(mid);
            if (rows * m <= rounds * cus) { last = mid; slots = m; lo = mid + 1; } else hi = mid - 1;
        }
        if (slots && rounds * (steps[last] + 3) < best_cost) {
            best = {steps[last], slots, slots > blocks};
            best_cost = rounds * (steps[last] + 3);
        }
        first = last;
    }
    return best;
}
// How a call runs: nb batch rows by ng KV heads at a time, and what is where in the scratch: which K / V records are bad, these records; for
// the backward the same of Q / dO, then the parts' sums.  The records are one and a half to two and a half times as large as what they are made of, and
// the scratch is the caller's memory: kF32SplitRecords bytes of them at most (and 64 MB of parts' sums), in even shares; a KV head of one row
// that needs more has no such route.  Forward + backward of 64 heads on 8 KV heads, everything at once / so, us (and MB at the peak, outputs
// included; the left figures with terms cut off instead of rounded, 1.5 % faster at 1024 tokens): 4096 tokens 3200 (529) / 3275 (450),
// window 512 985 / 1010, 4 x 2000 3415 (913) / 3499 (579), 8192 12070 (1046) / 12310 (604), 16384 47300 (2106) / 49400 (911).  128 MB:
// window 512 another 7 % slower, the others alike.
constexpr size_t kF32SplitRecords = (size_t)256 << 20;
struct F32SplitPlan { int nb, ng, tiles; size_t kv, q_bad, q, plan, partial, bytes; F32SplitParts parts; };
F32SplitPlan f32_split_plan(const gptoss_attn_params *p, bool bwd) {
    auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
    auto share = [](int n, size_t most) { const int times = (int)((n + most - 1) / most); return (n + times - 1) / times; };
    F32SplitPlan s{};
    if (!f32_split_route(p, bwd)) return s;
    s.tiles = split_key_tiles(p->Sq, p->Skv, effective_window(p));
    const size_t n_kv = (size_t)s.tiles, n_q = (size_t)(p->H / p->G) * ((p->Sq + 31) / 32);      // of a KV head
    const size_t most = kF32SplitRecords / (n_kv * F32Split::kKvRecord + (bwd ? n_q * F32Split::kQRecord : 0));
    if (most == 0) return s;
    s.nb = most > (size_t)p->G ? share(p->B, most / p->G) : 1;
    s.ng = share(p->G, most);
    if (most >= (size_t)p->B) {                            // all batch rows, some of the KV heads, where that is more even: backward of 3 x 2000 padded 1135 -> 1044 us
        const int ng = share(p->G, most / p->B);
        const int by_rows = (p->B + s.nb - 1) / s.nb * ((p->G + s.ng - 1) / s.ng), by_heads = (p->G + ng - 1) / ng;
        if (by_heads < by_rows || (by_heads == by_rows && (int64_t)p->B * ng < (int64_t)s.nb * s.ng)) { s.nb = p->B; s.ng = ng; }
    }
    const size_t rows = (size_t)s.nb * s.ng;
    s.kv = up(4 * rows * n_kv);
    s.bytes = s.kv + rows * n_kv * F32Split::kKvRecord;
    if (!bwd) return s;
    s.q_bad = s.bytes;
    s.q = s.q_bad + up(4 * rows * n_q);
    s.plan = s.q + rows * n_q * F32Split::kQRecord;
    s.parts = f32_split_parts(p, (int64_t)rows);
    s.partial = s.plan + (s.parts.cut ? up(2 * sizeof(int) * rows * ((p->Skv + F32Split::kKeys - 1) / F32Split::kKeys)) : 0);
    s.bytes = s.partial + (s.parts.cut ? rows * s.parts.slots * (2 * F32Split::kKeys * kD * sizeof(float)) : 0);
    return s;
}
void f32_split_args(KArgs &a, const F32SplitPlan &s, void *scratch) {
    char *base = static_cast<char *>(scratch);
    a.split_kv_bad = reinterpret_cast<uint32_t *>(base);
    a.split_kv = base + s.kv;
    a.split_q_bad = reinterpret_cast<uint32_t *>(base + s.q_bad);
    a.split_q = base + s.q;
    a.split_tiles = s.tiles;
    a.split_steps = s.parts.steps;
    a.split_slots = s.parts.slots;
    a.split_partial = s.parts.cut ? reinterpret_cast<float *>(base + s.partial) : nullptr;
    a.split_plan = s.parts.cut && (a.seqlens || a.doc_start) ? reinterpret_cast<int *>(base + s.plan) : nullptr;
}
// step(last) for every share of the batch rows and KV heads, set in `a`
template <typename Step>
int f32_split_shares(KArgs &a, const F32SplitPlan &s, Step step) {
    for (a.split_b0 = 0; a.split_b0 < a.B; a.split_b0 += s.nb)
        for (a.split_g0 = 0; a.split_g0 < a.G; a.split_g0 += s.ng) {
            a.split_nb = s.nb < a.B - a.split_b0 ? s.nb : a.B - a.split_b0;
            a.split_ng = s.ng < a.G - a.split_g0 ? s.ng : a.G - a.split_g0;
            const int rc = step(a.split_b0 + s.nb >= a.B && a.split_g0 + s.ng >= a.G);
            if (rc) return rc;
        }
    return GPTOSS_ATTN_OK;
}

// One launch.  hipLaunchKernel reports this launch's own status, so an error some earlier call of the
// thread left in the runtime's sticky state is neither reported here nor cleared.  A grid beyond the
// x-dimension limit is refused on the host.
template <typename Kernel>
int launch(Kernel kernel, int64_t workgroups, int threads, hipStream_t st, const KArgs &a, size_t dynamic_lds = 0) {
    if (workgroups <= 0 || workgroups > 0x7fffffff) return GPTOSS_ATTN_ERR_SHAPE;
    void *args[] = {const_cast<KArgs *>(&a)};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(kernel), dim3((unsigned)workgroups), dim3((unsigned)threads),
                                         args, dynamic_lds, st);
    return e == hipSuccess ? GPTOSS_ATTN_OK : static_cast<int>(e);
}

// The same for a three-dimensional grid of 256-thread workgroups (the caller has checked the y and z limits).
template <typename Kernel>
int launch3(Kernel kernel, dim3 grid, hipStream_t st, const KArgs &a) {
    if (grid.x == 0 || grid.y == 0 || grid.z == 0 || grid.y > 65535 || grid.z > 65535) return GPTOSS_ATTN_ERR_SHAPE;
    void *args[] = {const_cast<KArgs *>(&a)};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, dim3(256), args, 0, st);
    return e == hipSuccess ? GPTOSS_ATTN_OK : static_cast<int>(e);
}

// The sum of the partials of cut key blocks; dSinks, where it is still to be done, in the first blocks of the same launch.
template <typename Kernel>
int launch_reduce(Kernel kernel, int64_t chunks, hipStream_t st, KArgs a, bool with_dsinks) {
    int heads = with_dsinks ? a.H : 0;
    const int64_t blocks = (chunks + 255) / 256 + heads;
    if (blocks > 0x7fffffff) return GPTOSS_ATTN_ERR_SHAPE;
    void *args[] = {&a, &heads};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(kernel), dim3((unsigned)blocks), dim3(256), args, 0, st);
    return e == hipSuccess ? GPTOSS_ATTN_OK : static_cast<int>(e);
}

// ---- single-pass backward of sliding-window layers (attn_bwd_window.h) ------------------------
// Taken for bf16 self-attention (Sq == Skv, no offset, no packed rows) with a window of at most
// 128 and 2..16 query heads per KV head (WinCfg::kMaxGroup: the kernel's LDS holds dSinks slots for
// that many); everything else keeps the dK/dV + dQ kernel pair.
bool window_single_pass(const gptoss_attn_params *p) {
    const int r = p->G > 0 ? p->H / p->G : 0;
    const int window = effective_window(p);
    return p->dtype == GPTOSS_ATTN_BF16 && window > 0 && window <= WinCfg::kMaxWindow && !p->doc_start &&
           p->q_offset == 0 && !p->q_offset_dev && p->Sq == p->Skv && r >= 2 && r <= WinCfg::kMaxGroup;
}

constexpr int kMaxDevices = 64;

// Compute units of the current device (looked up once per device).
int compute_units() {
    static std::atomic<int> cus[kMaxDevices];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
    int n = cus[dev].load(std::memory_order_acquire);
    if (n <= 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cus[dev].store(n, std::memory_order_release);
    }
    return n;
}

// Query blocks per workgroup, 4 to 32: the count whose rounds of workgroups (one per compute unit at a time) take the least time,
// a workgroup's own start counted as four steps; of equals the larger (fewer seams).
int window_chunk_blocks(const gptoss_attn_params *p, int cus) {
    const int64_t n_blocks = (p->Sq + WinCfg::kRows - 1) / WinCfg::kRows, rows = (int64_t)p->G * p->B;
    const int pairs = (p->H / p->G + 1) / 2;
    if (cus <= 0) cus = 256;
    int best = WinCfg::kBack;
    int64_t best_cost = 0;
    for (int c = WinCfg::kBack; c <= 32; ++c) {
        const int64_t rounds = (rows * ((n_blocks + c - 1) / c) + cus - 1) / cus, cost = rounds * (pairs * c + 4);
        if (c == WinCfg::kBack || cost <= best_cost) { best = c; best_cost = cost; }
        if (c >= n_blocks) break;
    }
    return best;
}

// A kernel that uses more than 64 KB of LDS has to be told so once per device.
template <auto Kernel>
int lds_attribute(int bytes) {
    static std::atomic<bool> done[kMaxDevices];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return static_cast<int>(e);
    const bool tracked = dev >= 0 && dev < kMaxDevices;
    if (!tracked || !done[dev].load(std::memory_order_acquire)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) return static_cast<int>(e);
        if (tracked) done[dev].store(true, std::memory_order_release);
    }
    return GPTOSS_ATTN_OK;
}

// Scratch of the single-pass window backward: dSinks partial sums [B][chunk][H] (room for two words each: the size that callers have known), then (rounded up
// to 16 bytes) the fp32 dK / dV shares of the four key blocks on each seam between chunks.
struct WindowScratch { int chunk_blocks, n_chunks; size_t sink_bytes, seam_bytes; };

WindowScratch window_scratch_for(const gptoss_attn_params *p, int chunk_blocks) {
    WindowScratch w;
    w.chunk_blocks = chunk_blocks;
    const int n_blocks = (p->Sq + WinCfg::kRows - 1) / WinCfg::kRows;
    w.n_chunks = (n_blocks + w.chunk_blocks - 1) / w.chunk_blocks;
    w.sink_bytes = (((size_t)p->B * w.n_chunks * p->H * 2 * sizeof(float)) + 15) & ~(size_t)15;
    w.seam_bytes = (size_t)p->B * p->G * (w.n_chunks - 1) * WinCfg::kBack * 2 * (2 * WinCfg::kRows * kD) * sizeof(float);
    return w;
}

WindowScratch window_scratch(const gptoss_attn_params *p, int cus) { return window_scratch_for(p, window_chunk_blocks(p, cus)); }

// seam_sums: neighbouring chunks exchange fp32 shares through the scratch (needs window_scratch bytes);
// otherwise each chunk walks four query blocks past its end and nothing but the dSinks sums is kept.
int launch_window_bwd(const gptoss_attn_params *p, hipStream_t st, bool seam_sums, SinkTypes ty) {
    int rc = lds_attribute<&attn_bwd_window_kernel>(WinCfg::kLdsBytes);
    if (rc) return rc;
    KArgs a = make_args(p, ty);
    const WindowScratch ws = window_scratch(p, compute_units());
    a.scale_log2 = (p->scale > WinCfg::kMinScale ? p->scale : WinCfg::kMinScale) * kLog2e;
    a.chunk_blocks = ws.chunk_blocks;
    a.dsink_partial = p->delta;
    if (seam_sums && ws.n_chunks > 1)
        a.boundary_partial = reinterpret_cast<float *>(reinterpret_cast<char *>(p->delta) + ws.sink_bytes);
    rc = launch(attn_bwd_window_kernel, (int64_t)a.G * a.B * ws.n_chunks, 64 * WinCfg::NWAVES, st, a, WinCfg::kLdsBytes);
    if (rc) return rc;
    // seam blocks and dSinks in one small launch
    const int64_t seam_chunks = a.boundary_partial ? (int64_t)a.B * a.G * (ws.n_chunks - 1) * WinCfg::kBack * 2 * WinCfg::kRows * 8 : 0;
    const int seam_blocks = (int)((seam_chunks + 255) / 256);
    const int sink_blocks = a.dsinks ? a.H : 0;
    if (seam_blocks + sink_blocks == 0) return GPTOSS_ATTN_OK;
    int n_chunks = ws.n_chunks, sb = seam_blocks;
    void *args[] = {&a, &n_chunks, &sb};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(attn_bwd_window_finish_kernel),
                                         dim3((unsigned)(seam_blocks + sink_blocks)), dim3(256), args, 0, st);
    return e == hipSuccess ? GPTOSS_ATTN_OK : static_cast<int>(e);
}

int launch_f32_split_kv(const KArgs &a, hipStream_t st) { return launch(attn_f32_split_kv_kernel, (int64_t)a.split_nb * a.split_ng * a.split_tiles, 256, st, a); }
int64_t f32_split_grid(const KArgs &a) { return (int64_t)a.split_ng * (a.r / 4) * a.split_nb * ((a.Sq + 31) / 32); }

int launch_f32_split_fwd(const gptoss_attn_params *p, hipStream_t st, SinkTypes ty, const F32SplitPlan &plan, void *scratch) {
    KArgs a = make_args(p, ty);
    f32_split_args(a, plan, scratch);
    const int rc = lds_attribute<&attn_f32_split_fwd_kernel>(F32Split::kRowsLds);
    if (rc) return rc;
    return f32_split_shares(a, plan, [&](bool) {
        const int s = launch_f32_split_kv(a, st);
        return s ? s : launch(attn_f32_split_fwd_kernel, f32_split_grid(a), 512, st, a, F32Split::kRowsLds);
    });
}

int launch_f32_split_bwd(const gptoss_attn_params *p, hipStream_t st, SinkTypes ty, const F32SplitPlan &plan, void *scratch) {
    KArgs a = make_args(p, ty);
    f32_split_args(a, plan, scratch);
    int rc = lds_attribute<&attn_f32_split_dq_kernel>(F32Split::kDqLds);
    const bool lengths = a.seqlens || a.doc_start;
    if (rc || (rc = lengths ? lds_attribute<&attn_f32_split_dkdv_kernel<true>>(F32Split::kDkdvLds) : lds_attribute<&attn_f32_split_dkdv_kernel<false>>(F32Split::kDkdvLds))) return rc;
    return f32_split_shares(a, plan, [&](bool last) {
        int s = launch_f32_split_kv(a, st);
        if (s || (s = launch(attn_f32_split_dq_kernel, f32_split_grid(a), 512, st, a, F32Split::kDqLds))) return s;
        const bool with_dsinks = last && a.dsinks;         // (every row's statistics are there)
        if (!a.split_partial && with_dsinks && (s = launch(attn_bwd_dsinks_kernel, a.H, 1024, st, a))) return s;
        s = launch(lengths ? attn_f32_split_dkdv_kernel<true> : attn_f32_split_dkdv_kernel<false>, (int64_t)a.split_ng * a.split_nb * a.split_slots, 512, st, a, F32Split::kDkdvLds);
        if (s || !a.split_partial) return s;
        return launch_reduce(attn_f32_split_reduce_kernel, (int64_t)2 * a.split_nb * a.split_ng * a.Skv * 16, st, a, with_dsinks);
    });
}

template <int NQB, int NW>
int launch_decode(int64_t workgroups, hipStream_t st, const KArgs &a) {
    constexpr int lds = decode_lds_bytes<NQB, NW>();
    const int rc = lds > 64 * 1024 ? lds_attribute<&attn_decode_kernel<NQB, NW>>(lds) : GPTOSS_ATTN_OK;
    return rc ? rc : launch(attn_decode_kernel<NQB, NW>, workgroups, 64 * NW, st, a, lds);
}

// one launch of a synthetic instruction stream (mfma_rate.h): one workgroup per compute unit
template <int MIX>
int64_t launch_stream_probe(int waves_per_simd, int iters, float *sink, hipStream_t st) {
    const void *fn = reinterpret_cast<const void *>(stream_probe_kernel<MIX>);
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kStreamProbeLdsBytes);
    if (e != hipSuccess) return -static_cast<int64_t>(e) - 1000;
    const int blocks = compute_units();
    void *args[] = {&sink, &iters};
    e = hipLaunchKernel(fn, dim3((unsigned)blocks), dim3(256u * waves_per_simd), args, kStreamProbeLdsBytes, st);
    if (e != hipSuccess) return -static_cast<int64_t>(e) - 1000;
    return (int64_t)blocks * 4 * waves_per_simd * iters * kStreamProbeMfmas;     // MFMA instructions the launch executes
}

}  // namespace

extern "C" {

int gptoss_attn_version(void) { return GPTOSS_ATTN_ABI_VERSION; }

const char *gptoss_attn_status_string(int status) {
    switch (status) {
        case GPTOSS_ATTN_OK: return "ok";
        case GPTOSS_ATTN_ERR_NULL_PARAMS: return "params pointer is NULL";
        case GPTOSS_ATTN_ERR_NULL_TENSOR: return "a required tensor pointer is NULL";
        case GPTOSS_ATTN_ERR_HEAD_DIM: return "head_dim must be 64";
        case GPTOSS_ATTN_ERR_HEADS: return "H and G must be positive and H divisible by G";
        case GPTOSS_ATTN_ERR_SHAPE: return "B, Sq, Skv must be positive; window, q_offset non-negative; positions and window at most 2^30; scale positive and finite; doc_start needs Sq == Skv and q_offset == 0; at most 2^31-1 workgroups";
        case GPTOSS_ATTN_ERR_DTYPE: return "unsupported dtype";
        case GPTOSS_ATTN_ERR_ALIGNMENT: return "tensor base or stride is not 16-byte aligned";
        case GPTOSS_ATTN_ERR_STRIDE: return "sequence stride smaller than head_dim or larger than 2^24 elements";
        case GPTOSS_ATTN_ERR_ABI: return "struct_size does not match this library";
        case GPTOSS_ATTN_ERR_WORKSPACE: return "the problem needs more scratch than the library's built-in array holds (gptoss_attn_static_scratch_bytes)";
        default: return status > 0 ? "HIP runtime error (status is the hipError_t)" : "unknown status";
    }
}

int gptoss_attn_validate(const gptoss_attn_params *p, int need_bwd) {
    if (!p) return GPTOSS_ATTN_ERR_NULL_PARAMS;
    if (p->struct_size != sizeof(gptoss_attn_params)) return GPTOSS_ATTN_ERR_ABI;
    if (p->dtype != GPTOSS_ATTN_BF16 && p->dtype != GPTOSS_ATTN_FP32) return GPTOSS_ATTN_ERR_DTYPE;
    if (p->D != kD) return GPTOSS_ATTN_ERR_HEAD_DIM;
    if (p->H <= 0 || p->G <= 0 || p->H % p->G) return GPTOSS_ATTN_ERR_HEADS;
    if (p->B <= 0 || p->Sq <= 0 || p->Skv <= 0 || p->window < 0 || (!p->q_offset_dev && p->q_offset < 0)) return GPTOSS_ATTN_ERR_SHAPE;
    // positions are 32-bit in the kernels and +-2^30 marks "no window" / "dead row"
    if ((int64_t)p->Sq + (p->q_offset_dev ? 0 : p->q_offset) > (1 << 30) || p->Skv > (1 << 30) || p->window > (1 << 30)) return GPTOSS_ATTN_ERR_SHAPE;
    if (!(p->scale > 0.0f) || !(p->scale < 3.0e38f)) return GPTOSS_ATTN_ERR_SHAPE;
    if (p->doc_start && (p->Sq != p->Skv || p->q_offset != 0 || p->q_offset_dev)) return GPTOSS_ATTN_ERR_SHAPE;
    if (p->q_offset_dev && (reinterpret_cast<uintptr_t>(p->q_offset_dev) & 3)) return GPTOSS_ATTN_ERR_ALIGNMENT;
    const int eb = p->dtype == GPTOSS_ATTN_FP32 ? 4 : 2;
    int rc;
    if ((rc = check_tensor(p->q, p->q_stride, eb, p->D))) return rc;
    if ((rc = check_tensor(p->k, p->k_stride, eb, p->D))) return rc;
    if ((rc = check_tensor(p->v, p->v_stride, eb, p->D))) return rc;
    if ((rc = check_tensor(p->o, p->o_stride, eb, p->D))) return rc;
    if (!p->lse) return GPTOSS_ATTN_ERR_NULL_TENSOR;
    if (need_bwd) {
        if ((rc = check_tensor(p->d_o, p->do_stride, eb, p->D))) return rc;
        if ((rc = check_tensor(p->dq, p->dq_stride, eb, p->D))) return rc;
        if ((rc = check_tensor(p->dk, p->dk_stride, eb, p->D))) return rc;
        if ((rc = check_tensor(p->dv, p->dv_stride, eb, p->D))) return rc;
        if (!p->delta) return GPTOSS_ATTN_ERR_NULL_TENSOR;
        if (!aligned16(p->delta)) return GPTOSS_ATTN_ERR_ALIGNMENT;   // the dK/dV partial sums use 16-byte accesses
    }
    return GPTOSS_ATTN_OK;
}

// Bytes of the row-statistics part of the scratch; dK/dV partials follow.
static size_t stats_bytes(const gptoss_attn_params *p) {
    return fp32_stats_bytes(p) + (size_t)16 * (size_t)p->B * (size_t)p->H * (size_t)p->Sq;
}

// dK/dV partial sums of `parts` slices
static size_t partials_bytes(const gptoss_attn_params *p, int parts) {
    return parts > 1 ? (size_t)parts * 2 * sizeof(float) * (size_t)p->B * (size_t)p->G * (size_t)p->Skv * kD : 0;
}

size_t gptoss_attn_fwd_workspace_bytes(const gptoss_attn_params *p) {
    // (asked before anything has looked at the shapes: heads the forward will refuse would divide by zero below)
    if (!p || p->B <= 0 || p->H <= 0 || p->G <= 0 || p->H % p->G || p->Sq <= 0 || p->Skv <= 0) return 0;
    if (decode_route(p)) {
        const int splits = decode_splits(p);
        if (splits > 1) return (size_t)p->B * p->G * splits * decode_partial_floats(p->Sq * (p->H / p->G)) * sizeof(float);
    } else if (fwd_pipe_route(p) && !p->doc_start) {
        const int splits = fwd_pipe_splits(p);
        if (splits > 1) return (size_t)splits * p->B * p->H * p->Sq * (kD + 2) * sizeof(float);
    }
    return 0;
}

// The backward's scratch with `parts` slices of the key blocks.
static size_t bwd_bytes(const gptoss_attn_params *p, int parts) {
    size_t n = stats_bytes(p);
    if (p->G > 0 && p->Skv > 0) {
        n += partials_bytes(p, parts);
        if (window_single_pass(p)) {
            // gptoss_attn_bwd takes this route and lays its own scratch over the same bytes.  The layout
            // follows the compute-unit count of the device that is current at launch time; the size
            // returned is that of the shortest chunks (the most seams), which covers every device.
            const WindowScratch ws = window_scratch_for(p, WinCfg::kBack);
            if (ws.sink_bytes + ws.seam_bytes > n) n = ws.sink_bytes + ws.seam_bytes;
        }
    }
    return n;
}

size_t gptoss_attn_bwd_workspace_bytes(const gptoss_attn_params *p) {
    if (!p || p->B <= 0 || p->H <= 0 || p->Sq <= 0) return 0;
    return bwd_bytes(p, p->G > 0 && p->Skv > 0 ? dkdv_parts_for(p, p->seqlens != nullptr, p->doc_start != nullptr) : 1);
}

size_t gptoss_attn_workspace_bytes(const gptoss_attn_params *p) {
    if (!p || p->B <= 0 || p->H <= 0 || p->Sq <= 0) return 0;
    // with or without lengths of padded rows and documents: who asks may not have filled these in yet
    int parts = 1;
    for (int kind = 0; kind < 4 && p->G > 0 && p->Skv > 0; ++kind) {
        const int n = dkdv_parts_for(p, kind & 1, kind & 2);
        if (n > parts) parts = n;
    }
    const size_t n = bwd_bytes(p, parts), fwd = gptoss_attn_fwd_workspace_bytes(p);
    return fwd > n ? fwd : n;
}

size_t gptoss_attn_split_bytes(const gptoss_attn_params *p, int backward) {
    return p ? f32_split_plan(p, backward != 0).bytes : 0;
}

// scratch: see gptoss_attn_fwd_scratch (NULL or too little: the keys are not cut)
static int forward(const gptoss_attn_params *p, void *stream, SinkTypes ty, void *scratch, size_t scratch_bytes) {
    const int rc = gptoss_attn_validate(p, 0);
    if (rc) return rc;
    if (!aligned16(scratch)) return GPTOSS_ATTN_ERR_ALIGNMENT;
    const bool cut = scratch && scratch_bytes >= gptoss_attn_fwd_workspace_bytes(p);
    KArgs a = make_args(p, ty);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (decode_route(p)) {
        if (cut) { a.kv_splits = decode_splits(p); a.fwd_partial = static_cast<float *>(scratch); }
        const int pairs = a.Sq * a.r;
        const int64_t wgs = (int64_t)a.G * a.B * a.kv_splits;
        if (decode_whole(p)) return pairs <= 32 ? launch_decode<1, 8>(wgs, st, a) : launch_decode<2, 8>(wgs, st, a);
        const int s = pairs <= 32 ? launch_decode<1, 4>(wgs, st, a) : launch_decode<2, 4>(wgs, st, a);
        if (s || a.kv_splits == 1) return s;
        return launch(attn_decode_combine_kernel, ((int64_t)a.B * a.G * pairs + 3) / 4, 256, st, a);
    }
    if (p->dtype == GPTOSS_ATTN_FP32) {
        const F32SplitPlan plan = f32_split_plan(p, false);
        if (plan.bytes && scratch && scratch_bytes >= plan.bytes) return launch_f32_split_fwd(p, st, ty, plan, scratch);
        const int ks = f32_key_splits(a);
        const int64_t grid32 = f32_grid(a, ks);
        return ks == 4 ? launch(attn_f32_fwd_kernel<4>, grid32, 256, st, a) : ks == 2 ? launch(attn_f32_fwd_kernel<2>, grid32, 256, st, a) : launch(attn_f32_fwd_kernel<1>, grid32, 256, st, a);
    }
    const int hpb = hpb_for(a.r), qb = query_blocks_for(a.window);
    const int64_t grid = q_outer_grid(a, hpb, qb);
    if (fwd_window_route(p)) {
        // two 32-row query blocks per workgroup (K / V rows staged once for both) where that still leaves every compute
        // unit several rounds of workgroups, else one
        const int64_t pairs = (int64_t)a.G * (a.r / 4) * a.B * ((a.Sq + 63) / 64);
        const bool by_pairs = a.Sq > 32 && pairs >= 8 * (int64_t)compute_units();
        const dim3 wgrid((unsigned)a.G, (unsigned)((a.r / 4) * a.B), (unsigned)(by_pairs ? (a.Sq + 63) / 64 : (a.Sq + 31) / 32));
        const bool plain = fwd_window_plain(p);
#define GPTOSS_LAUNCH_WIN(WH) (plain ? launch3(attn_fwd_window_kernel<WH, false>, wgrid, st, a) : launch3(attn_fwd_window_kernel<WH, true>, wgrid, st, a))
        switch (a.window / 32) {
            case 1: return GPTOSS_LAUNCH_WIN(1);
            case 2: return GPTOSS_LAUNCH_WIN(2);
            case 3: return GPTOSS_LAUNCH_WIN(3);
            default: return GPTOSS_LAUNCH_WIN(4);
        }
#undef GPTOSS_LAUNCH_WIN
    }
    if (fwd_pipe_route(p)) {
        const int splits = cut && !a.doc_start ? fwd_pipe_splits(p) : 1;
        if (splits > 1) {
            a.kv_splits = splits;
            a.fwd_partial = static_cast<float *>(scratch);
            const int s = launch(attn_fwd_pipe_kernel<true, false>, grid * splits, 256, st, a);
            return s ? s : launch(attn_fwd_combine_kernel, ((int64_t)a.B * a.H * a.Sq + 31) / 32, 256, st, a);
        }
        return fwd_pipe_plain(p) ? launch(attn_fwd_pipe_kernel<false, false>, grid, 256, st, a)
               : a.doc_start     ? launch(attn_fwd_pipe_kernel<true, true>, grid, 256, st, a)
                                 : launch(attn_fwd_pipe_kernel<true, false>, grid, 256, st, a);
    }
#define GPTOSS_LAUNCH_FWD(HPB, QB) launch(attn_fwd_kernel<HPB, QB>, grid, 256, st, a)
    if (qb == 2) return hpb == 4 ? GPTOSS_LAUNCH_FWD(4, 2) : hpb == 2 ? GPTOSS_LAUNCH_FWD(2, 2) : GPTOSS_LAUNCH_FWD(1, 2);
    return hpb == 4 ? GPTOSS_LAUNCH_FWD(4, 1) : hpb == 2 ? GPTOSS_LAUNCH_FWD(2, 1) : GPTOSS_LAUNCH_FWD(1, 1);
#undef GPTOSS_LAUNCH_FWD
}

int gptoss_attn_fwd(const gptoss_attn_params *p, void *stream) { return forward(p, stream, {}, nullptr, 0); }

static bool sink_dtype_ok(int dtype) { return dtype == GPTOSS_ATTN_FP32 || dtype == GPTOSS_ATTN_BF16; }

int gptoss_attn_fwd_sinks(const gptoss_attn_params *p, int sinks_dtype, void *stream) {
    if (!sink_dtype_ok(sinks_dtype)) return GPTOSS_ATTN_ERR_DTYPE;
    return forward(p, stream, {sinks_dtype == GPTOSS_ATTN_BF16, false}, nullptr, 0);
}

int gptoss_attn_fwd_scratch(const gptoss_attn_params *p, int sinks_dtype, void *scratch, size_t scratch_bytes, void *stream) {
    if (!sink_dtype_ok(sinks_dtype)) return GPTOSS_ATTN_ERR_DTYPE;
    return forward(p, stream, {sinks_dtype == GPTOSS_ATTN_BF16, false}, scratch, scratch_bytes);
}

int gptoss_attn_bwd_preprocess(const gptoss_attn_params *p, void *stream) {
    const int rc = gptoss_attn_validate(p, 1);
    if (rc) return rc;
    const KArgs a = make_args(p, {});
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t rows = (int64_t)a.B * a.H * a.Sq;
    int s = p->dtype == GPTOSS_ATTN_FP32 ? launch(attn_f32_delta_kernel, (rows + 15) / 16, 256, st, a)
                                         : launch(attn_bwd_delta_kernel, (rows + 127) / 128, 256, st, a);
    if (s == GPTOSS_ATTN_OK && a.dsinks) s = launch(attn_bwd_dsinks_kernel, a.H, 1024, st, a);
    return s;
}

static int launch_dkdv_sum(const KArgs &a, hipStream_t st, bool with_dsinks) {
    if (a.dkdv_steps) return launch_reduce(attn_bwd_dkdv_pieces_reduce_kernel, (int64_t)2 * a.B * a.G * ((a.Skv + 31) / 32) * 256, st, a, with_dsinks);
    return launch_reduce(attn_bwd_dkdv_reduce_kernel, (int64_t)2 * a.B * a.G * ((a.Skv + 31) / 32) * 256, st, a, with_dsinks);
}

// The dK/dV launch (and the sum of the partials when key blocks are cut).  whole_blocks: never cut a
// key block, so that nothing beyond the row statistics is kept in the scratch.  with_dsinks: dSinks too, from the row statistics.
static int launch_dkdv(const gptoss_attn_params *p, void *stream, bool whole_blocks, bool with_dsinks, SinkTypes ty) {
    const int rc = gptoss_attn_validate(p, 1);
    if (rc) return rc;
    KArgs a = make_args(p, ty);
    hipStream_t st = static_cast<hipStream_t>(stream);
    a.dkdv_parts = whole_blocks ? 1 : dkdv_parts_for(p, p->seqlens != nullptr, p->doc_start != nullptr);
    a.dkdv_partial = reinterpret_cast<float *>(reinterpret_cast<char *>(p->delta) + stats_bytes(p));
    if (with_dsinks && a.dkdv_parts == 1) {
        const int s = launch(attn_bwd_dsinks_kernel, a.H, 1024, st, a);
        if (s) return s;
    }
    if (p->dtype == GPTOSS_ATTN_FP32) {
        const int s = launch(attn_f32_dkdv_kernel, (int64_t)a.B * a.G * a.dkdv_parts * ((a.Skv + 31) / 32), 256, st, a);
        if (s || a.dkdv_parts == 1) return s;
        return launch_reduce(attn_f32_dkdv_reduce_kernel, (int64_t)2 * a.B * a.G * a.Skv * 16, st, a, with_dsinks);
    }
    if (dkdv64_route(p, a.dkdv_parts)) {
        const int64_t blocks = (int64_t)a.B * ((a.Skv + Dkdv64::BN - 1) / Dkdv64::BN);      // of a KV head
        // padded and packed rows, several rows of one length whose blocks would stay whole otherwise, and few enough equal shares that the
        // longest of them decides: pieces by the walks' lengths, at most as many as there are slots for partial sums (Dkdv64Plan; the
        // kernels hold kMaxBlocks lengths, nearly twice what dkdv_parts_for leaves) (not packed rows of up to four heads per KV head whose
        // equal shares run all at once: these are four heads of a tile or two, and finding the lengths takes longer than the better
        // division saves.  Backward of 8 heads on two KV heads, equal shares / by lengths, us: 4096 tokens in documents of 100 43 / 50, of
        // 300 54 / 58, of 3000 132 / 135, of 95, 1502 and 222 94 / 92; 8192 (512 shares) of 300 82 / 67; eight heads on one, 4096 of 300 62
        // / 59) (Few shares, rows of one length, the same in a graph: 8 heads on one KV head 6000 tokens 293 / 263 (192 shares), 8000 337 /
        // 294 (256), 16 on one 5000 358 / 324, 32 on four 2200 142 / 130 (288), 8 on two 5000 201 / 195 (320); 32 on four 3000 187 / 195
        // (384), 8 on one 12000 567 / 587 (376), 2 x 6000 343 / 370 (384): with several rounds the shares even out by themselves, and equal
        // ones keep in step.)
        const bool one_round = !a.seqlens && a.doc_start && a.r <= 4 && a.G * blocks * a.dkdv_parts <= 256;
        const bool by_lengths = a.dkdv_parts > 1 && blocks <= Dkdv64Plan::kMaxBlocks && !one_round &&
                                (a.seqlens || a.doc_start || (a.B > 1 && a.Sq < 4096 && many_key_blocks(p)) || a.G * blocks * a.dkdv_parts <= 320);
        if (by_lengths) a.dkdv_slots = (int)((int64_t)a.dkdv_parts * a.B * a.Skv / Dkdv64::BN);
        const int64_t grid64 = a.G * (by_lengths ? a.dkdv_slots : blocks * a.dkdv_parts);
        const bool plain = !by_lengths && !a.seqlens && !a.doc_start && a.Sq % kTile == 0;
        const int s = plain ? launch(attn_bwd_dkdv64_kernel<false>, grid64, 256, st, a) : launch(attn_bwd_dkdv64_kernel<true>, grid64, 256, st, a);
        if (s || a.dkdv_parts == 1) return s;
        if (by_lengths)
            return dkdv64_reduce_chunks(a.G * blocks) == 4 ? launch_reduce(attn_bwd_dkdv64_reduce_kernel<4>, a.G * blocks * 4 * 256, st, a, with_dsinks)
                                                           : launch_reduce(attn_bwd_dkdv64_reduce_kernel<1>, a.G * blocks * 16 * 256, st, a, with_dsinks);
        return launch_reduce(attn_bwd_dkdv_reduce_kernel, (int64_t)2 * a.B * a.G * ((a.Skv + 31) / 32) * 256, st, a, with_dsinks);
    }
    dkdv_pieces_for(p, a);
    const int64_t grid = dkdv_grid(a);
    const int s = a.doc_start ? launch(attn_bwd_dkdv_kernel<kDkdvWaves, kDkdvNB, true>, grid, 64 * kDkdvWaves, st, a)
                 : a.dkdv_steps ? launch(attn_bwd_dkdv_kernel<kDkdvWaves, kDkdvNB, false, true>, grid, 64 * kDkdvWaves, st, a)
                              : launch(attn_bwd_dkdv_kernel<kDkdvWaves, kDkdvNB, false>, grid, 64 * kDkdvWaves, st, a);
    if (s || a.dkdv_parts == 1) return s;
    return launch_dkdv_sum(a, st, with_dsinks);
}

// The same for float32: dQ's workgroups come first.  Two launches / one, us as above (workgroups): 8 heads on one KV head 300 tokens 38 /
// 24, 1000 76 / 67 (730), 1500 141 / 102 (846), on two 500 41 / 31, 2 x 700 76 / 61 (792), 2 x 1000 111 / 104 (1024); 64 on eight 64 29 /
// 22, 150 36 / 30 (520); window 128, 8 on one 400 34 / 23.  Not 4 x 700 122 / 132 (1144); rows of a few tiles start and end rather than
// walk, 64 on eight 180 39.7 / 40.6 (672), 2 x 100 37 / 38 (768).
static int64_t f32_dkdv_grid(const KArgs &a) { return (int64_t)a.B * a.G * a.dkdv_parts * ((a.Skv + 31) / 32); }
static bool f32_both_route(const KArgs &a, int dtype) {
    return dtype == GPTOSS_ATTN_FP32 && f32_key_splits(a) == 4 && f32_grid(a, 4) + f32_dkdv_grid(a) <= (a.Sq > 256 ? 1024 : 640);
}
static int launch_f32_both(KArgs &a, hipStream_t st) {
    int s = launch(attn_f32_delta_kernel, ((int64_t)a.B * a.H * a.Sq + 15) / 16, 256, st, a);
    if (s) return s;
    int first = (int)f32_grid(a, 4);
    void *args[] = {&a, &first};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(attn_f32_both_kernel), dim3((unsigned)(first + f32_dkdv_grid(a))), dim3(256), args, 0, st);
    if (e != hipSuccess) return static_cast<int>(e);
    if (a.dkdv_parts > 1) return launch_reduce(attn_f32_dkdv_reduce_kernel, (int64_t)2 * a.B * a.G * a.Skv * 16, st, a, a.dsinks != nullptr);
    return a.dsinks ? launch(attn_bwd_dsinks_kernel, a.H, 1024, st, a) : GPTOSS_ATTN_OK;
}

// dQ and dK/dV side by side, behind the row statistics.
static int launch_both(KArgs &a, hipStream_t st, bool dq_first) {
    int s = launch(attn_bwd_delta_kernel, ((int64_t)a.B * a.H * a.Sq + 127) / 128, 256, st, a);
    if (s) return s;
    const void *kernel = a.doc_start    ? reinterpret_cast<const void *>(attn_bwd_both_kernel<true, false>)
                         : a.dkdv_steps ? reinterpret_cast<const void *>(attn_bwd_both_kernel<false, true>)
                                        : reinterpret_cast<const void *>(attn_bwd_both_kernel<false, false>);
    int dkdv = (int)dkdv_grid(a), dq = (int)q_outer_grid(a, 4, 1), dkdv_at = dq_first ? dq : 0, dq_at = dq_first ? 0 : dkdv;
    void *args[] = {&a, &dkdv_at, &dq_at};
    const hipError_t e = hipLaunchKernel(kernel, dim3((unsigned)(dkdv + dq)), dim3(256), args, 0, st);
    if (e != hipSuccess) return static_cast<int>(e);
    if (a.dkdv_parts > 1) return launch_dkdv_sum(a, st, a.dsinks != nullptr);
    return a.dsinks ? launch(attn_bwd_dsinks_kernel, a.H, 1024, st, a) : GPTOSS_ATTN_OK;
}

int gptoss_attn_bwd_dkdv(const gptoss_attn_params *p, void *stream) { return launch_dkdv(p, stream, false, false, {}); }

// The dQ launch; fuse_delta: the kernel also produces the row statistics (see attn_bwd_dq_kernel).
static int launch_dq(const gptoss_attn_params *p, void *stream, int fuse_delta) {
    const int rc = gptoss_attn_validate(p, 1);
    if (rc) return rc;
    const KArgs a = make_args(p, {});
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (p->dtype == GPTOSS_ATTN_FP32) {
        const int ks = f32_key_splits(a);
        const int64_t grid32 = f32_grid(a, ks);
#define GPTOSS_LAUNCH_DQ(KS) (fuse_delta ? launch(attn_f32_dq_kernel<KS, true>, grid32, 256, st, a) : launch(attn_f32_dq_kernel<KS, false>, grid32, 256, st, a))
        return ks == 4 ? GPTOSS_LAUNCH_DQ(4) : ks == 2 ? GPTOSS_LAUNCH_DQ(2) : GPTOSS_LAUNCH_DQ(1);
#undef GPTOSS_LAUNCH_DQ
    }
    const int hpb = hpb_for(a.r);
    const int qb = dq_query_blocks(a);
    const int64_t grid = q_outer_grid(a, hpb, qb);
#define GPTOSS_LAUNCH_DQ(HPB, QB) \
    (fuse_delta ? launch(attn_bwd_dq_kernel<HPB, QB, true>, grid, 256, st, a) : launch(attn_bwd_dq_kernel<HPB, QB, false>, grid, 256, st, a))
    if (qb == 2) return hpb == 4 ? GPTOSS_LAUNCH_DQ(4, 2) : hpb == 2 ? GPTOSS_LAUNCH_DQ(2, 2) : GPTOSS_LAUNCH_DQ(1, 2);
    return hpb == 4 ? GPTOSS_LAUNCH_DQ(4, 1) : hpb == 2 ? GPTOSS_LAUNCH_DQ(2, 1) : GPTOSS_LAUNCH_DQ(1, 1);
#undef GPTOSS_LAUNCH_DQ
}

int gptoss_attn_bwd_dq(const gptoss_attn_params *p, void *stream) { return launch_dq(p, stream, 0); }

// The whole backward: the dQ kernel computes the row statistics on the way (no separate
// pass over O and dO), then dK/dV and dSinks read them from the scratch buffer.  The results are
// bit-identical to gptoss_attn_bwd_preprocess + gptoss_attn_bwd_dkdv + gptoss_attn_bwd_dq, but for the two routes in front: float32 with
// scratch (attn_f32_split.h) and the single-pass window kernel agree with these within the rounding of their sums.
static int bwd_all(const gptoss_attn_params *p, void *stream, bool whole_blocks, SinkTypes ty, void *scratch = nullptr, size_t scratch_bytes = 0) {
    int rc = gptoss_attn_validate(p, 1);
    if (rc) return rc;
    if (!aligned16(scratch)) return GPTOSS_ATTN_ERR_ALIGNMENT;
    if (scratch) {
        const F32SplitPlan plan = f32_split_plan(p, true);
        if (plan.bytes && scratch_bytes >= plan.bytes) return launch_f32_split_bwd(p, static_cast<hipStream_t>(stream), ty, plan, scratch);
    }
    if (window_single_pass(p)) return launch_window_bwd(p, static_cast<hipStream_t>(stream), !whole_blocks, ty);
    if (!whole_blocks) {
        KArgs a = make_args(p, ty);
        a.dkdv_parts = dkdv_parts_for(p, p->seqlens != nullptr, p->doc_start != nullptr);
        a.dkdv_partial = reinterpret_cast<float *>(reinterpret_cast<char *>(p->delta) + stats_bytes(p));
        if (f32_both_route(a, p->dtype)) return launch_f32_both(a, static_cast<hipStream_t>(stream));
        const BothRoute both = both_route(p, a);
        if (both.taken) return launch_both(a, static_cast<hipStream_t>(stream), both.dq_first);
    }
    rc = launch_dq(p, stream, 1);
    if (rc) return rc;
    return launch_dkdv(p, stream, whole_blocks, p->dsinks != nullptr, ty);
}

int gptoss_attn_bwd(const gptoss_attn_params *p, void *stream) { return bwd_all(p, stream, false, {}); }

int gptoss_attn_bwd_sinks(const gptoss_attn_params *p, int sinks_dtype, int dsinks_dtype, void *stream) {
    if (!sink_dtype_ok(sinks_dtype) || !sink_dtype_ok(dsinks_dtype)) return GPTOSS_ATTN_ERR_DTYPE;
    return bwd_all(p, stream, false, {sinks_dtype == GPTOSS_ATTN_BF16, dsinks_dtype == GPTOSS_ATTN_BF16});
}

int gptoss_attn_bwd_scratch(const gptoss_attn_params *p, int sinks_dtype, int dsinks_dtype, void *scratch, size_t scratch_bytes, void *stream) {
    if (!sink_dtype_ok(sinks_dtype) || !sink_dtype_ok(dsinks_dtype)) return GPTOSS_ATTN_ERR_DTYPE;
    return bwd_all(p, stream, false, {sinks_dtype == GPTOSS_ATTN_BF16, dsinks_dtype == GPTOSS_ATTN_BF16}, scratch, scratch_bytes);
}

// ---- the backward for callers that cannot allocate ------------------------------------------
// Same kernels as gptoss_attn_bwd; the row statistics live in a device array that is part of the
// library image instead of a caller-provided workspace.  Each GPU has its own copy of the array
// at its own address, looked up once per device.
namespace {
constexpr size_t kStaticScratchBytes = GPTOSS_ATTN_STATIC_SCRATCH_BYTES;
}
static __device__ __align__(256) float scratch[kStaticScratchBytes / sizeof(float)];
static std::atomic<float *> scratch_ptr[kMaxDevices];     // device address of `scratch`, per device; NULL = not looked up yet

static int static_scratch(float **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return static_cast<int>(e);
    if (dev < 0 || dev >= kMaxDevices) return GPTOSS_ATTN_ERR_WORKSPACE;
    float *ptr = scratch_ptr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        // with the device current, the symbol resolves to this device's copy; two threads racing
        // here look up the same address
        e = hipGetSymbolAddress(reinterpret_cast<void **>(&ptr), HIP_SYMBOL(scratch));
        if (e != hipSuccess) return static_cast<int>(e);
        if (!ptr) return GPTOSS_ATTN_ERR_WORKSPACE;
        scratch_ptr[dev].store(ptr, std::memory_order_release);
    }
    *out = ptr;
    return GPTOSS_ATTN_OK;
}

size_t gptoss_attn_static_scratch_bytes(void) { return kStaticScratchBytes; }

int gptoss_attn_bwd_static(const gptoss_attn_params *p, void *stream) {
    if (!p) return GPTOSS_ATTN_ERR_NULL_PARAMS;
    if (p->struct_size != sizeof(gptoss_attn_params)) return GPTOSS_ATTN_ERR_ABI;
    gptoss_attn_params q = *p;
    q.delta = reinterpret_cast<float *>(static_cast<uintptr_t>(256));   // stands in for the scratch while the other arguments are checked
    int rc = gptoss_attn_validate(&q, 1);
    if (rc) return rc;
    if (stats_bytes(&q) > kStaticScratchBytes) return GPTOSS_ATTN_ERR_WORKSPACE;
    rc = static_scratch(&q.delta);
    if (rc) return rc;
    return bwd_all(&q, stream, true, {});
}

// ---- packed rows (doc_start.h) ----------------------------------------------------------------
int gptoss_attn_doc_start(const void *position_ids, int id_bytes, int B, int S, int64_t row_stride, int32_t *doc_start, void *stream) {
    if (!position_ids || !doc_start) return GPTOSS_ATTN_ERR_NULL_TENSOR;
    if (id_bytes != 4 && id_bytes != 8) return GPTOSS_ATTN_ERR_DTYPE;
    if (B <= 0 || B > 65535 || S <= 0 || S > (1 << 30)) return GPTOSS_ATTN_ERR_SHAPE;
    if ((reinterpret_cast<uintptr_t>(position_ids) & (id_bytes - 1)) || (reinterpret_cast<uintptr_t>(doc_start) & 3)) return GPTOSS_ATTN_ERR_ALIGNMENT;
    const dim3 grid((unsigned)((S + kDocTokens - 1) / kDocTokens), (unsigned)B);
    void *args[] = {&position_ids, &row_stride, &S, &doc_start};
    const void *kernel = id_bytes == 8 ? reinterpret_cast<const void *>(doc_start_kernel<int64_t>) : reinterpret_cast<const void *>(doc_start_kernel<int32_t>);
    const hipError_t e = hipLaunchKernel(kernel, grid, dim3(256), args, 0, static_cast<hipStream_t>(stream));
    return e == hipSuccess ? GPTOSS_ATTN_OK : static_cast<int>(e);
}

// ---- measurement aid (mfma_rate.h) -----------------------------------------------------------
int64_t gptoss_attn_mfma_rate_probe(const void *operands, size_t operand_bytes, int iters, float *sink, size_t sink_floats,
                                    void *stream) {
    if (!operands || !sink || operand_bytes < 16 || iters <= 0 || !aligned16(operands)) return GPTOSS_ATTN_ERR_NULL_TENSOR;
    const int64_t blocks = (int64_t)2 * compute_units();       // two workgroups of four wavefronts per compute unit
    if ((size_t)blocks * 256 > sink_floats || operand_bytes / 16 > 0xffffffffu) return GPTOSS_ATTN_ERR_SHAPE;
    const u32x4 *ops = static_cast<const u32x4 *>(operands);
    uint32_t n_vec = (uint32_t)(operand_bytes / 16);
    void *args[] = {&ops, &n_vec, &iters, &sink};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(mfma_rate_kernel), dim3((unsigned)blocks), dim3(256), args, 0,
                                         static_cast<hipStream_t>(stream));
    if (e != hipSuccess) return -static_cast<int64_t>(e) - 1000;
    return blocks * 4 * (int64_t)iters * kMfmaRatePerIter;      // MFMA instructions the launch executes
}

int64_t gptoss_attn_stream_probe(int mix, int waves_per_simd, int iters, float *sink, size_t sink_floats, void *stream) {
    if (!sink || iters <= 0 || mix < 0 || mix >= kStreamMixes || waves_per_simd < 1 || waves_per_simd > 3) return GPTOSS_ATTN_ERR_SHAPE;
    if ((size_t)compute_units() * 256 * waves_per_simd > sink_floats) return GPTOSS_ATTN_ERR_SHAPE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (mix) {
        case kStreamMfmaOnly: return launch_stream_probe<kStreamMfmaOnly>(waves_per_simd, iters, sink, st);
        case kStreamFwdUniform: return launch_stream_probe<kStreamFwdUniform>(waves_per_simd, iters, sink, st);
        case kStreamFwdClumped: return launch_stream_probe<kStreamFwdClumped>(waves_per_simd, iters, sink, st);
        case kStreamDqUniform: return launch_stream_probe<kStreamDqUniform>(waves_per_simd, iters, sink, st);
        case kStreamDqClumped: return launch_stream_probe<kStreamDqClumped>(waves_per_simd, iters, sink, st);
        default: return launch_stream_probe<kStreamDkdvUniform>(waves_per_simd, iters, sink, st);
    }
}

}  // extern "C"
