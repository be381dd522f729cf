// Host-only view of the prefill workspace carve-up for tests/test_prefill_layout.py:
// exposes pf_layout (qwen-3-ocho_amd/csrc/qfm_prefill_layout.h) through a C ABI.
#include "../qwen-3-ocho_amd/csrc/qfm_prefill_layout.h"

extern "C" int pf_layout_c(int T, int H, int I, int E, int K, int has_sh, int gu_rows, int dn_cols, int bm, int slices,
                           int pairs_per_blk, unsigned long long *off, unsigned long long *bytes,
                           unsigned long long *meta) {
    const qfm::PfLayout L = qfm::pf_layout(T, H, I, E, K, has_sh != 0, gu_rows, dn_cols, bm, slices, pairs_per_blk);
    for (int r = 0; r < qfm::kPfCount; r++) {
        off[r] = L.off[r];
        bytes[r] = L.bytes[r];
    }
    meta[0] = L.total; meta[1] = L.P; meta[2] = L.max_mt;
    meta[3] = (unsigned long long)L.nt_gu; meta[4] = (unsigned long long)L.nt_dn; meta[5] = (unsigned long long)L.nblk;
    return qfm::kPfCount;
}

extern "C" int pf_router_slices_c(int T, int E, unsigned long long part_bytes) {
    return qfm::pf_router_slices(T, E, part_bytes);
}
extern "C" int pf_select_split_c(int T, int H, int slices) { return qfm::pf_select_split(T, H, slices); }
extern "C" int mid_token_tiles_c(int T, int E, int K, int I, int f4) { return qfm::mid_token_tiles(T, E, K, I, f4 != 0); }
extern "C" int mid_items_bound_c(int T, int E, int K, int has_sh, int token_tiles) {
    return qfm::mid_items_bound(T, E, K, has_sh != 0, token_tiles);
}
extern "C" int mid_takes_c(int T, int K, int I, int f4, int f32) { return qfm::mid_takes(T, K, I, f4 != 0, f32 != 0); }
extern "C" int mid_offers_tiles_c(int T, int I, int f32) { return qfm::mid_offers_tiles(T, I, f32 != 0); }
extern "C" int mid_picks_tiles_c(int groups, int items, int tiles, int T, int E, int K, int I, int f4) {
    const qfm::MidCost c =
        qfm::mid_cost(I, f4 != 0, qfm::mid_token_tiles(T, E, K, I, f4 != 0), qfm::mid_reads_once(T, E, K, f4 != 0));
    return tiles * c.tile + c.base < groups * c.group + (items - groups) * c.item;
}
