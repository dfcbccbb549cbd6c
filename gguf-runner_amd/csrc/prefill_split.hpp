// Key-split prefill launches (short chunks over long caches): the plan, shared by
// the host and the kernels.
//
// A launch whose (query head, query block) workgroups leave most CUs idle is cut
// along the keys instead.  The kv_mul query heads of a KV head are packed into
// the rows of a query block (row r of KV head g is token r / kv_mul, query head
// g * kv_mul + r % kv_mul: a 16-token chunk fills its 32-row waves, and a K / V
// tile is read once for the whole group), and every block's range of BN-key tiles
// is cut into pieces of `ct` tiles, one workgroup each.  A workgroup writes its
// unnormalised f32 O^T accumulators and each row's (maximum, sum) as partials,
// in the register layout of the MFMA accumulators; the combine kernel merges them.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

namespace gr {

struct PrefillSplit {
    int n_splits = 0;        // pieces of the longest block; 0: not split
    int ct = 0;              // tiles per piece
    int n_qb = 0;            // query blocks per KV head
    int bm = 0, bn = 0;      // rows per block, keys per tile
    int64_t tiles = 0;       // tiles of all blocks
    int wgs = 0;             // workgroups with tiles
    float* ws_o = nullptr;   // [g][query block][piece][row group of 32][d / 32][4][lane][4]
    float* ws_ml = nullptr;  // [g][query block][piece][row group of 32][m | l][lane]
};

// Keys [lo, hi) that the tokens tok0 .. tok1 of a chunk see (hi exclusive).
__host__ __device__ inline int pf_key_lo(int p0, int tok0, int window, int bidirectional) {
    int lo = window > 0 ? p0 + tok0 + 1 - window : 0;
    if (bidirectional && lo > p0) lo = p0;
    return lo > 0 ? lo : 0;
}
__host__ __device__ inline int pf_key_hi(int p0, int tok1, int n_tokens, int bidirectional) {
    return bidirectional ? p0 + n_tokens : p0 + tok1 + 1;
}

// Tiles of query block qb of a split launch.
__host__ __device__ inline int pf_split_tiles(int qb, int bm, int bn, int n_tokens, int kv_mul, int p0, int window,
                                              int bidirectional) {
    const int rows = n_tokens * kv_mul;
    const int last = (qb + 1) * bm < rows ? (qb + 1) * bm - 1 : rows - 1;
    const int first = pf_key_lo(p0, qb * bm / kv_mul, window, bidirectional) / bn * bn;
    return (pf_key_hi(p0, last / kv_mul, n_tokens, bidirectional) - first + bn - 1) / bn;
}

// Workgroup b of a split launch.  It runs on XCD b % 8, and the XCDs share the KV
// heads: one XCD takes n_kv / 8 heads, or 8 / n_kv XCDs take the query blocks of one
// head in turn (so that a head's tiles stay in few L2s and the short and the long
// blocks of a first chunk spread evenly); other head counts go round the XCDs item
// by item.  qb may come out past the last block: an idle workgroup.
struct PfSplitItem {
    int g, piece, qb;
};
__host__ __device__ inline int pf_split_xcds(int n_kv) { return n_kv % 8 == 0 ? 1 : (8 % n_kv == 0 ? 8 / n_kv : 0); }
__host__ __device__ inline int pf_split_grid(int n_kv, int n_qb, int n_splits) {
    const int r = pf_split_xcds(n_kv);
    if (r == 0) return n_kv * n_qb * n_splits;
    return 8 * ((n_kv * r + 7) / 8) * ((n_qb + r - 1) / r) * n_splits;
}
__host__ __device__ inline PfSplitItem pf_split_item(int b, int n_kv, int n_qb, int n_splits) {
    const int r = pf_split_xcds(n_kv);
    if (r == 0) return {b / (n_qb * n_splits), b / n_qb % n_splits, b % n_qb};
    const int per = (n_qb + r - 1) / r;  // blocks of a head on one XCD
    const int x = b & 7, i = b >> 3;
    return {x / r + i / (per * n_splits) * 8, i / per % n_splits, i % per * r + x % r};
}

// Partial slots (workgroups) a split launch may have, for `slots` resident
// workgroups: causal blocks of a first chunk are half empty in the
// [block][piece] index, so twice the resident number.
constexpr int kPfSplitSlots = 2;
constexpr size_t pf_split_ws_bytes(int slots, int bm, int head_dim) {
    return (size_t)kPfSplitSlots * slots * bm * (head_dim + 4) * 4;
}

// Bytes of a plan's partials, and their carving: ws_ml, then ws_o.
inline size_t pf_split_part_bytes(const PrefillSplit& s, int n_kv, int head_dim) {
    return (size_t)s.n_qb * n_kv * s.n_splits * s.bm * (head_dim + 4) * 4;
}
inline void pf_split_carve(PrefillSplit& s, int n_kv, void* ws) {
    s.ws_ml = (float*)ws;
    s.ws_o = s.ws_ml + (size_t)s.n_qb * n_kv * s.n_splits * s.bm * 4;
}

// The smallest piece of at least min_ct tiles whose workgroups all fit the
// `slots` the GPU holds at once (0 splits if there is none worth having: pieces
// as long as the blocks).  Both counts only fall as pieces grow: the piece is found by
// bisection, over block lengths computed once.
inline PrefillSplit pf_split_plan(int n_tokens, int n_heads, int n_kv, int p0, int window, int bidirectional, int bm,
                                  int bn, int slots, int min_ct) {
    PrefillSplit s;
    const int kv_mul = n_heads / n_kv;
    s.bm = bm, s.bn = bn;
    s.n_qb = (int)(((int64_t)n_tokens * kv_mul + bm - 1) / bm);
    if ((int64_t)s.n_qb * n_kv >= slots) return s;  // one piece a block fills the slots
    std::vector<int> tiles(s.n_qb);
    int longest = 0;
    int64_t total = 0;
    for (int qb = 0; qb < s.n_qb; qb++) {
        const int t = pf_split_tiles(qb, bm, bn, n_tokens, kv_mul, p0, window, bidirectional);
        tiles[qb] = t;
        longest = t > longest ? t : longest;
        total += t;
    }
    auto pieces = [&](int ct) {  // workgroups per KV head
        int64_t n = 0;
        for (int t : tiles) n += (t + ct - 1) / ct;
        return n;
    };
    auto fits = [&](int ct) {
        return pieces(ct) * n_kv <= slots &&
               (int64_t)s.n_qb * n_kv * ((longest + ct - 1) / ct) <= kPfSplitSlots * (int64_t)slots;
    };
    int lo = (int)((total * n_kv + slots - 1) / slots), hi = longest;  // pieces of `longest` fit
    if (lo < min_ct) lo = min_ct;
    while (lo < hi) {
        const int ct = lo + (hi - lo) / 2;
        if (fits(ct)) hi = ct;
        else lo = ct + 1;
    }
    if (lo >= longest) return s;
    s.ct = lo;
    s.tiles = total * n_kv;
    s.wgs = (int)(pieces(lo) * n_kv);
    s.n_splits = (longest + lo - 1) / lo;
    return s;
}

// What a cut must save in a launch's longest workgroup beyond the general cost below, in
// tiles: the combine launch and its partials are a fixed cost that short caches do not earn.
struct PfSplitSaving {
    float whole = 1e30f;      // keys of the unsplit launch's longest workgroup, in tiles
    float launch = 0.0f;      // the combine launch
    float per_group = 0.0f;   // per 32 rows of partials
    float partials = 0.0f;    // and at most for them
};

// The plan if it is worth having against an unsplit launch that takes `whole` tiles of
// time (its longest workgroup): at least one piece and its share of all tiles on `cus`
// CUs, 1.1 for the uneven finish, a tile for the combine launch and per_wg per
// workgroup for its partials; and `saving`.  Most launches that lose show it without a
// plan, by the keys their rows see and a piece per block (a plan of 8192 tokens costs the
// host some us).
inline PrefillSplit pf_split_choose(int n_tokens, int n_heads, int n_kv, int p0, int window, int bidirectional, int bm,
                                    int bn, int slots, int min_ct, float whole, int cus, float per_wg,
                                    PfSplitSaving saving = {}) {
    const int64_t n_qb = ((int64_t)n_tokens * (n_heads / n_kv) + bm - 1) / bm;
    int64_t seen = 0;  // keys that the tokens see, causal (an image block's see more)
    const int64_t n = n_tokens, in = window > 0 ? (window > p0 ? (window - p0 < n ? window - p0 : n) : 0) : n;
    seen = in * p0 + in * (in + 1) / 2 + (n - in) * window;
    const float least = 1.1f * ((float)(seen * n_heads) / ((float)bm * bn * cus)) + 1.0f + per_wg * (float)(n_qb * n_kv);
    if (least * 0.999f >= whole) return {};
    const PrefillSplit s = pf_split_plan(n_tokens, n_heads, n_kv, p0, window, bidirectional, bm, bn, slots, min_ct);
    if (s.n_splits == 0) return s;
    const float share = (float)s.tiles / cus;
    const float cost = 1.1f * (share > s.ct ? share : (float)s.ct) + 1.0f + per_wg * s.wgs;
    const int64_t groups = ((int64_t)n_tokens * (n_heads / n_kv) + 31) / 32 * n_kv * s.n_splits;
    const float written = saving.per_group * (float)groups;
    const bool saves = saving.whole > (float)s.ct + saving.launch + (written < saving.partials ? written : saving.partials);
    return cost < whole && saves ? s : PrefillSplit{};
}

// The 16-bit launches (prefill.hip).  Resident workgroups of the split kernels (two per CU
// at d <= 128, one at 256), the rows and keys of their tiles, the cost per workgroup, and
// what a cut of one query block's launch must save.
constexpr int kPfCUs = 256;
struct PfSplitShape {
    int slots, bm, bn;
    float per_wg, launch, per_group, partials;
};
constexpr PfSplitShape pf_split_shape(int head_dim) {
    return head_dim == 64    ? PfSplitShape{2 * kPfCUs, 128, 128, 0.017f, 3.0f, 0.004f, 100.0f}
           : head_dim == 128 ? PfSplitShape{2 * kPfCUs, 128, 64, 0.03f, 0.0f, 0.0125f, 5.0f}
                             : PfSplitShape{kPfCUs, 128, 32, 0.06f, 3.0f, 0.0f, 0.0f};
}

// Split or not: in tiles of 128 rows x BN keys, the unsplit launch takes its longest
// pair of blocks (it has at most one workgroup per CU here); the split one as
// pf_split_choose says.  A launch of one query block is the shortest there is, and the
// combine launch (3.7 us) and the partials must come out of its keys: PfSplitShape's
// saving (the constants differ with the tile's time, and at d128 the unsplit kernel also
// prepares Q); with two blocks or more, which the unsplit workgroups run in turn, 1.5
// tiles.  Fitted to 2051 launches that the general cost splits (fifteen head shapes, 2 to
// 2400 tokens after 0 to 5000, f16 and bf16): the side taken is slower than the other by
// at most 7%, in 99 of 100 by less than 2%.  By the general cost alone 140 of them were more
// than 2% slower split, up to 32%: 14 / 2 heads d64, 16 tokens after 250 11.3 us, split
// 14.9; 32 / 8 heads d128, 88 after 250 17.9, split 19.9.  (What it leaves whole
// could still gain: 32 / 8 heads d128, 700 tokens after 130 42.6, split 34.2.)
// MI355X, us per call (prep included), unsplit -> split: 32 / 8 heads d128, 64 tokens after
// 4000 78.5 -> 29, 512 after 8000 302 -> 92, 1500 after 8000 325 -> 267; 14 / 2 heads d64,
// 203 after 4000 83 -> 25, 1500 after 8000 167 -> 80; 8 / 4 heads d256, 512 after 8000 543
// -> 61.  Not split: 1500 tokens from 0, d128 54 (63 split); 4096 from 0, d64 58 (73 split).
inline PrefillSplit pf_split_16bit_plan(int n_tokens, int n_heads, int n_kv, int head_dim, int p0, int window,
                                        int bidirectional) {
    const PfSplitShape sh = pf_split_shape(head_dim);
    if (n_tokens <= 0) return {};
    const int n_qb = (n_tokens - 1) / sh.bm + 1;
    if ((int64_t)n_heads * ((n_qb + 1) / 2) > kPfCUs) return {};
    float whole = 0.0f, keys = 0.0f;
    auto add = [&](int qb) {
        const int last = (qb + 1) * sh.bm < n_tokens ? (qb + 1) * sh.bm - 1 : n_tokens - 1;
        whole += (float)pf_split_tiles(qb, sh.bm, sh.bn, n_tokens, 1, p0, window, bidirectional);
        keys += (float)(pf_key_hi(p0, last, n_tokens, bidirectional) - pf_key_lo(p0, qb * sh.bm, window, bidirectional));
    };
    add(n_qb - 1);
    if (n_qb > 1) add(0);
    const PfSplitSaving saving = n_qb > 1 ? PfSplitSaving{keys / sh.bn, 1.5f, 0.0f, 0.0f}
                                          : PfSplitSaving{keys / sh.bn, sh.launch, sh.per_group, sh.partials};
    return pf_split_choose(n_tokens, n_heads, n_kv, p0, window, bidirectional, sh.bm, sh.bn, sh.slots, 128 / sh.bn, whole,
                           kPfCUs, sh.per_wg, saving);
}

}  // namespace gr
