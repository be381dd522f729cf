// qfm_prefill_layout.h -- the prefill workspace carve-up, in one place.
//
// Plain C++ (no HIP): the launcher, the workspace sizing and the workspace
// view all take their offsets from pf_layout(), and the CPU tests replay it
// (tests/test_prefill_layout.py) for every token count, format, shape and
// tile width to check that the regions are disjoint, inside the workspace,
// and large enough for everything the planning and GEMM kernels index.
#pragma once
#include <stddef.h>

namespace qfm {

// Regions of the prefill workspace, in address order.
enum PfRegion {
    kPfLg,        // fp32 [slices][T][E] approximate router logits (slice 0 ends as the view's logits)
    kPfXnorm,     // fp32 [T] ||x_t||
    kPfWnorm,     // fp32 [E] ||w_e||
    kPfWb16,      // bf16 [E][H] router weights
    kPfSel,       // int [T][K]
    kPfWts,       // fp32 [T][K]
    kPfGam,       // fp32 [T] shared-expert gate
    kPfCtr,       // int [8] {candidate overflows, gate/up items, down items, ...}
    kPfOff,       // int [E + 2] group offsets
    kPfBlk,       // int [nblk][E] per counting block histograms
    kPfItemsGu,   // int4 [max_mt * nt_gu] gate/up work items, each at the index of the block that runs it
    kPfItemsDn,   // int4 [max_mt * nt_dn] down work items, likewise
    kPfTok,       // int [P] pair -> token
    kPfSlot,      // int [P] pair -> partial slot
    kPfPwt,       // fp32 [P] pair weight
    kPfHid,       // bf16 [P][I] hidden rows
    kPfPart,      // fp16 [P][H] owned partials, each 64-column group scaled by 2^k
    kPfPartK,     // int8 [P][H / 64] the k of each partial group
    kPfXsum,      // fp32 [T] sum(x_t)
    kPfHsum,      // fp32 [P][nt_gu] hidden row sums per gate/up n-tile
    kPfX16,       // fp16 [T][H] x rows scaled by 2^k (INT8 gate/up)
    kPfX16sum,    // fp32 [T]
    kPfX16isc,    // fp32 [T]
    kPfCount
};

struct PfLayout {
    size_t off[kPfCount], bytes[kPfCount];
    size_t total;              // bytes from the first region to the end of the last
    size_t P;                  // pairs: T * (K + shared)
    size_t max_mt;             // bound on the 128-row m-tiles over all groups (a multiple of 8)
    int nt_gu, nt_dn;          // n-tiles of the gate/up and down GEMMs
    int nblk;                  // counting / scatter blocks
};

// T tokens; (H, I, E, K) the configuration; has_sh: shared expert present;
// gu_rows: weight rows per gate/up tile (gate and up interleaved: I / (gu_rows
// / 2) n-tiles); dn_cols: output columns per down tile; bm: rows per m-tile;
// slices: router GEMM k-slices; pairs_per_blk: pairs per counting block.
inline PfLayout pf_layout(int T, int H, int I, int E, int K, bool has_sh, int gu_rows, int dn_cols, int bm,
                          int slices, int pairs_per_blk) {
    PfLayout L{};
    auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
    const size_t t = (size_t)T;
    L.P = t * (size_t)(K + (has_sh ? 1 : 0));
    L.nt_gu = I / (gu_rows / 2);
    L.nt_dn = H / dn_cols;
    L.nblk = (int)((t * K + pairs_per_blk - 1) / pairs_per_blk);
    // every group of c rows takes ceil(c / bm) <= c / bm + 1 m-tiles: at most
    // P / bm + (E + 1) over the E routed groups and the shared one
    L.max_mt = (L.P / bm + E + 2 + 7) / 8 * 8;
    const size_t want[kPfCount] = {
        (size_t)slices * t * E * 4, t * 4, (size_t)E * 4, (size_t)E * H * 2, t * K * 4, t * K * 4, t * 4, 8 * 4,
        (size_t)(E + 2) * 4, (size_t)L.nblk * E * 4, L.max_mt * L.nt_gu * 16, L.max_mt * L.nt_dn * 16,
        L.P * 4, L.P * 4, L.P * 4, L.P * I * 2, L.P * H * 2, L.P * (size_t)(H / 64), t * 4, L.P * L.nt_gu * 4,
        t * H * 2, t * 4, t * 4};
    size_t o = 0;
    for (int r = 0; r < kPfCount; r++) {
        L.off[r] = o;
        L.bytes[r] = want[r];
        o += al(want[r]);
    }
    L.total = o;
    return L;
}

// The middle path's work items: an expert's rows, 16 mid_token_tiles at a time
// (the figures are at launch_mid), and the most that T rows can make: one per
// distinct expert, one more per full item, the shared expert's. The launcher
// refuses a call whose bound exceeds the item region before it launches
// anything, and the plan kernel stores none beyond the region.
inline int mid_token_tiles(int T, int E, int K, int I, bool f4) { return T * K / E < 24 || f4 || I > 512 ? 1 : 4; }
inline int mid_items_bound(int T, int E, int K, bool has_sh, int token_tiles) {
    const int mt = 16 * token_tiles, tk = T * K;
    return (E < tk ? E : tk) + tk / mt + (has_sh ? (T + mt - 1) / mt : 0);
}

constexpr int kPfTileRows = 128;       // rows of a tile of the grouped GEMMs

// The largest call of the middle path, in rows; at a larger top_k than 10 also in
// pairs, as it is an expert's rows that decide, unless the result is fp32, which
// keeps the items' hidden rows (below) as long as the rows allow. us per layer, the middle path /
// 128-row tiles: 2048/512 INT8 1500 rows 507 / 620, 2560/640 INT8 1500 rows 841 /
// 932, NVFP4 2048/512 458 / 686, 2560/640 723 / 991; it grows by 0.13, 0.30, 0.19
// and 0.28 us a row, the tiles by 0.04 to 0.07. Top-16, 2800 rows of 2048/512:
// INT8 940 / 737, NVFP4 1059 / 784.
constexpr int mid_rows_max(int I, bool f4) { return I <= 512 ? 2800 : f4 ? 2500 : 1800; }
inline bool mid_takes(int T, int K, int I, bool f4, bool f32) {
    return T <= mid_rows_max(I, f4) && (f32 || T * K <= 10 * mid_rows_max(I, f4));
}

// Few rows an expert: weights read once, nontemporal (the figures are at ld_w).
inline bool mid_reads_once(int T, int E, int K, bool f4) { return T * K / E < (f4 ? 8 : 12); }

// Which form of the expert GEMMs a middle call runs is known once the selection
// is: a router that crowds its rows on few experts makes many items of one
// expert, and each reads and converts its weights again, where a 128-row tile
// does it once. The tiles hold the hidden rows in 8 bits (bf16), the items in 11;
// a bf16 result rounds to about the same (error against 64 bits 0.0024 and
// 0.0017), an fp32 result does not (0.0017 and 0.0003) and keeps the items. For
// bf16 results, from mid_offers_tiles on, the tile GEMMs are launched behind the
// middle ones, and k_mid_plan leaves one pair of them without work (2.5 us each):
// the tiles run where tiles * tile + base < groups * group + (items - groups) *
// item, in units of 10 ns (groups: experts with a row, items: mid_token_tiles).
// Fitted to calls of both forms with router biases of spread 0 to 3 and with all
// rows on ten experts, 256 to 2800 rows; the choice is within 2% of the faster
// form in 363 of 368 of them and within 11% in all.
struct MidCost { int group, item, tile, base; };
inline bool mid_offers_tiles(int T, int I, bool f32) { return !f32 && T >= (I > 512 ? 256 : 384); }
inline MidCost mid_cost(int I, bool f4, int token_tiles, bool once) {
    if (f4) return I > 512 ? MidCost{0, 30, 99, 1000} : MidCost{0, 18, 68, 1300};
    if (I > 512) return once ? MidCost{0, 54, 67, 2400} : MidCost{0, 31, 65, 1700};
    return token_tiles > 1 ? MidCost{45, 58, 68, -800} : once ? MidCost{10, 30, 50, 2000} : MidCost{0, 19, 41, 2200};
}

// Slices of H in the router GEMM. Few m-tiles do not fill the chip, so K is cut
// (1021 rows: 31 -> 13 us in four). One slice writes the logits' own region;
// more lie in the partials' region (part_bytes), which the down GEMM writes
// later and which has room for four, at top_k 1 without a shared expert for two.
inline int pf_router_slices(int T, int E, size_t part_bytes) {
    const size_t room = part_bytes / ((size_t)T * E * 4);
    return T <= 2048 && room >= 4 ? 4 : T <= 4096 && room >= 2 ? 2 : 1;
}

// Four waves a token in k_pf_select (a block each), else one: while the blocks of
// all tokens are resident at once, 4 on each of the 256 CUs, and at H = 2560,
// whose rows leave less latency to hide, up to 800 (us at 700 / 900 / 1024 / 1025
// rows: 2048 four waves 21.3 / 23.2 / 22.6 / 27.3, one 25.6 / 24.6 / 22.4 / 22.6;
// 2560 four 22.7 / 27.0 / 27.4 / 29.8, one 25.2 / 25.2 / 25.0 / 25.1). Only where
// its input and output logits are two buffers: with one slice they are the same,
// and a wave would read logits that another wave of its token has already stored
// with the bias added.
inline bool pf_select_split(int T, int H, int slices) { return T <= (H == 2048 ? 1024 : 800) && slices > 1; }

}  // namespace qfm
