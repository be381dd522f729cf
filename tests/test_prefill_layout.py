"""Host-only checks of the prefill workspace carve-up (no GPU).

pf_layout (qwen-3-ocho_amd/csrc/qfm_prefill_layout.h) is the single source of
the prefill workspace offsets: the launcher, the workspace sizing and the
workspace view all read it. These tests compile it on the host and replay it
for token counts 9..16384, both arena formats, both shapes, with and without
the shared expert, and gate/up / down tile widths 64..256, checking that

* the regions are 256-byte aligned, in order, disjoint and inside the total;
* every region holds what the kernels index in it (items, pairs, partials,
  row sums) for the worst routing the bound admits;
* k_pf_plan's m-tile count never exceeds the bound the work lists and the
  GEMM grids are sized for, over adversarial, uniform and skewed routings,
  and every work item it writes lies inside its group;
* the library's own qfm_workspace_bytes equals the layout with the tile
  widths it is built with.
"""
import ctypes as C
import os
import subprocess
import tempfile

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NREG = 23
NAMES = ["lg", "xnorm", "wnorm", "wb16", "sel", "wts", "gam", "ctr", "off", "blk", "items_gu", "items_dn",
         "p_tok", "p_slot", "p_wt", "hid", "part", "partk", "xsum", "hsum", "x16", "x16sum", "x16isc"]
BM, SLICES, PAIRS_PER_BLK = 128, 1, 4096
GU_I8, GU_F4, DN_I8 = 256, 256, 128           # the tile widths the library is built with


@pytest.fixture(scope="module")
def shim():
    d = tempfile.mkdtemp(prefix="pflayout")
    so = os.path.join(d, "libpflayout.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", so,
                    os.path.join(ROOT, "tests", "prefill_layout_shim.cpp")], check=True)
    lib = C.CDLL(so)
    lib.pf_layout_c.restype = C.c_int
    return lib


def layout(shim, T, H, I, E, K, has_sh, gu, dn):
    off = (C.c_ulonglong * NREG)()
    by = (C.c_ulonglong * NREG)()
    meta = (C.c_ulonglong * 6)()
    n = shim.pf_layout_c(T, H, I, E, K, int(has_sh), gu, dn, BM, SLICES, PAIRS_PER_BLK, off, by, meta)
    assert n == NREG
    return (np.array(off[:], np.int64), np.array(by[:], np.int64),
            dict(total=meta[0], P=meta[1], max_mt=meta[2], nt_gu=meta[3], nt_dn=meta[4], nblk=meta[5]))


def plan_items(counts, nt):
    """k_pf_plan's work list for group row counts `counts`: (group, row0, rows, n)
    per m-tile and n-tile, in the kernel's order."""
    mt = (counts + BM - 1) // BM
    first = np.concatenate([[0], np.cumsum(mt)[:-1]])
    mtot = int(mt.sum())
    items = []
    for m in range(mtot):
        g = int(np.searchsorted(first, m, side="right") - 1)     # last group whose first m-tile <= m
        row0 = (m - int(first[g])) * BM
        rows = min(BM, int(counts[g]) - row0)
        items.extend((g, row0, rows, n) for n in range(nt))
    return mtot, items


TS = [9, 10, 37, 100, 128, 129, 300, 1000, 4095, 4096, 8037, 8038, 8192, 16384]
SHAPES = [(2048, 512), (2560, 640)]


@pytest.mark.parametrize("H,I", SHAPES)
@pytest.mark.parametrize("has_sh", [True, False])
@pytest.mark.parametrize("gu,dn", [(GU_I8, DN_I8), (GU_F4, GU_F4), (128, 64), (256, 256), (512, 128), (128, 256)])
def test_regions_disjoint_and_sized(shim, H, I, has_sh, gu, dn):
    E, K = 512, 10
    for T in TS:
        off, by, m = layout(shim, T, H, I, E, K, has_sh, gu, dn)
        assert (off % 256 == 0).all(), T
        ends = off + by
        assert (ends[:-1] <= off[1:]).all(), (T, [NAMES[i] for i in np.nonzero(ends[:-1] > off[1:])[0]])
        assert ends[-1] <= m["total"]
        S = K + (1 if has_sh else 0)
        P = T * S
        assert m["P"] == P
        nt_gu, nt_dn = I // (gu // 2), H // dn
        assert (m["nt_gu"], m["nt_dn"]) == (nt_gu, nt_dn)
        assert m["max_mt"] % 8 == 0                       # the XCD tile maps cover [0, max_mt * nt) exactly
        need = dict(lg=SLICES * T * E * 4, sel=T * K * 4, wts=T * K * 4, ctr=32, off=(E + 2) * 4,
                    blk=m["nblk"] * E * 4, items_gu=m["max_mt"] * nt_gu * 16, items_dn=m["max_mt"] * nt_dn * 16,
                    p_tok=P * 4, p_slot=P * 4, p_wt=P * 4, hid=P * I * 2, part=P * H * 2, partk=P * (H // 64),
                    hsum=P * nt_gu * 4,
                    x16=T * H * 2, x16sum=T * 4, x16isc=T * 4, wb16=E * H * 2)
        for k, v in need.items():
            assert by[NAMES.index(k)] >= v, (T, k, by[NAMES.index(k)], v)
        assert m["nblk"] * PAIRS_PER_BLK >= T * K
        # the m-tile bound: every group of c rows needs ceil(c / BM) <= c / BM + 1 tiles
        assert m["max_mt"] >= P // BM + E + 1


def _routings(T, K, E, rng):
    """Per-expert routed counts (each token picks K distinct experts): uniform,
    skewed, and the adversary that maximizes m-tiles (BM + 1 rows per expert)."""
    out = []
    for skew in (0.0, 1.5, 4.0):
        p = np.exp(skew * rng.standard_normal(E))
        p /= p.sum()
        cnt = np.zeros(E, np.int64)
        for _ in range(T):
            cnt[rng.choice(E, K, replace=False, p=p)] += 1
        out.append(cnt)
    adv = np.zeros(E, np.int64)
    left = T * K
    for e in range(E):                                    # BM + 1 rows each while pairs last, never above T
        c = min(BM + 1, T, left)
        adv[e] = c
        left -= c
    if left > 0:                                          # the rest spread (count <= T per expert)
        for e in range(E):
            add = min(T - adv[e], left)
            adv[e] += add
            left -= add
    out.append(adv)
    return out


@pytest.mark.parametrize("H,I", SHAPES)
@pytest.mark.parametrize("gu,dn", [(GU_I8, DN_I8), (GU_F4, GU_F4), (128, 64), (256, 256)])
def test_plan_fits_the_bounds(shim, H, I, gu, dn):
    E, K = 512, 10
    rng = np.random.default_rng(5)
    for T in (9, 37, 300, 2000, 8038):
        for has_sh in (True, False):
            off, by, m = layout(shim, T, H, I, E, K, has_sh, gu, dn)
            for cnt in _routings(T, K, E, rng):
                assert cnt.sum() == T * K and cnt.max() <= T
                groups = np.concatenate([cnt, [T] if has_sh else []]).astype(np.int64)
                for nt, cap in ((m["nt_gu"], by[NAMES.index("items_gu")] // 16),
                                (m["nt_dn"], by[NAMES.index("items_dn")] // 16)):
                    mtot, items = plan_items(groups, nt)
                    assert mtot <= m["max_mt"], (T, mtot, m["max_mt"])
                    assert len(items) <= cap
                    for g, row0, rows, n in items:
                        assert 0 < rows <= BM and row0 + rows <= groups[g] and 0 <= n < nt


@pytest.mark.parametrize("H,I,f4,top", [(2048, 512, 0, 2800), (2048, 512, 1, 2800), (2560, 640, 0, 1800),
                                        (2560, 640, 1, 2500)])
def test_middle_rows_fit_the_regions(shim, H, I, f4, top):
    """Calls of 9 to `top` rows (mid_rows_max) keep their own contents in the
    same regions: one item list whose bound (one item per distinct expert, one
    more per full mt rows, the shared expert's) launch_mid refuses to exceed,
    8-byte pairs over the token and slot regions, an int8 exponent per 64 hidden
    values in the row-sum region, and beyond 600 rows the K slices of the router
    logits in the partials' region (room for four but
    at top_k 1 without a shared expert)."""
    E = 512
    for K in (1, 2, 9, 10, 16):
        for has_sh in (True, False):
            for T in [9, 10, 31, 32, 33, 127, 128, 129, 600, 601, 819, 820, 1229, 1230, 2047, 2048, top - 1, top]:
                if T > top:
                    continue
                off, by, m = layout(shim, T, H, I, E, K, has_sh, GU_F4 if f4 else GU_I8, GU_F4 if f4 else DN_I8)
                r = dict(zip(NAMES, zip(off, by)))
                P = T * (K + has_sh)
                mt = 16 if T * K // E < 24 or f4 or I > 512 else 64
                items = min(E, T * K) + T * K // mt + (-(-T // mt) if has_sh else 0)
                assert items * 16 <= r["items_gu"][1], (K, has_sh, T)
                assert r["p_tok"][0] + 8 * P <= r["p_slot"][0] + r["p_slot"][1] and r["p_tok"][0] % 8 == 0
                assert P * (I // 64) <= r["hsum"][1]
                room = r["part"][1] // (T * E * 4)
                slices = 4 if T <= 2048 and room >= 4 else 2 if T <= 4096 and room >= 2 else 1
                assert slices == 1 or slices * T * E * 4 <= r["part"][1]
                assert room >= (4 if K + has_sh > 1 else 2)


@pytest.mark.parametrize("H,I,f4,top", [(2048, 512, 0, 2800), (2048, 512, 1, 2800), (2560, 640, 0, 1800),
                                        (2560, 640, 1, 2500)])
def test_middle_items_never_exceed_their_bound(shim, H, I, f4, top):
    """The item bound that the launcher checks before its first launch holds for
    every routing (uniform, skewed, all rows on one expert, one row more than
    whole items on as many experts as possible), and lies within the region that
    the plan kernel is given as its limit."""
    E = 512
    rng = np.random.default_rng(6)
    for K in (1, 10, 16):
        for T in (9, 16, 17, 129, 600, 1229, top):
            if T > top:
                continue
            for has_sh in (True, False):
                by = layout(shim, T, H, I, E, K, has_sh, GU_F4 if f4 else GU_I8, GU_F4 if f4 else DN_I8)[1]
                nt = shim.mid_token_tiles_c(T, E, K, I, f4)
                bound = shim.mid_items_bound_c(T, E, K, int(has_sh), nt)
                assert bound <= by[NAMES.index("items_gu")] // 16
                mt = 16 * nt
                routings = _routings(T, K, E, rng) if K > 1 else []
                one = np.zeros(E, np.int64)
                one[:K] = T
                spread = np.zeros(E, np.int64)                 # a row over whole items wherever rows are left
                left = T * K
                for e in range(E):
                    spread[e] = min(T, mt + 1 if left >= mt + 1 + (E - 1 - e) else 1, left)
                    left -= spread[e]
                spread[:K] += left // K
                for cnt in routings + [one, spread]:
                    items = int(((cnt + mt - 1) // mt).sum()) + (-(-T // mt) if has_sh else 0)
                    assert items <= bound, (K, T, has_sh, items, bound)


@pytest.mark.parametrize("H,I,f4,top", [(2048, 512, 0, 2800), (2048, 512, 1, 2800), (2560, 640, 0, 1800),
                                        (2560, 640, 1, 2500)])
def test_middle_path_by_pairs_and_routing(shim, H, I, f4, top):
    """The middle path ends at `top` rows and, at a larger top_k and for bf16
    results, at as many pairs as top-10 makes there. Inside, a plan that takes the 128-row tiles fits their
    work lists whatever the routing, rows crowded on ten experts take them (from
    the first call that offers them on), and evenly spread rows take the items up
    to the largest call."""
    E = 512
    rng = np.random.default_rng(8)
    first = 256 if I > 512 else 384
    for f32 in (0, 1):
        assert shim.mid_takes_c(top, 10, I, f4, f32) and not shim.mid_takes_c(top + 1, 10, I, f4, f32)
        assert shim.mid_takes_c(top, 1, I, f4, f32) and not shim.mid_takes_c(top + 1, 1, I, f4, f32)
        assert shim.mid_takes_c(10 * top // 16, 16, I, f4, f32)
        assert bool(shim.mid_takes_c(10 * top // 16 + 1, 16, I, f4, f32)) == bool(f32)   # fp32 results: by rows alone
        assert not shim.mid_takes_c(top + 1, 16, I, f4, f32)
    assert not shim.mid_offers_tiles_c(first - 1, I, 0) and shim.mid_offers_tiles_c(first, I, 0)
    assert not shim.mid_offers_tiles_c(first, I, 1) and not shim.mid_offers_tiles_c(top, I, 1)
    for T in (first, 600, 601, 1229, top):
        for K in (10, 16):
            if not shim.mid_takes_c(T, K, I, f4, 0):
                continue
            m = layout(shim, T, H, I, E, K, True, GU_F4 if f4 else GU_I8, GU_F4 if f4 else DN_I8)[2]
            mt = 16 * shim.mid_token_tiles_c(T, E, K, I, f4)
            ten, even = np.zeros(E, np.int64), np.full(E, T * K // E, np.int64)
            ten[:K], even[:T * K % E] = T, T * K // E + 1
            for cnt in [ten, even] + _routings(T, K, E, rng):
                g = np.append(cnt, T)
                n = [int((-(-g // per)).sum()) for per in (mt, BM)]
                assert n[1] <= m["max_mt"]
                pick = shim.mid_picks_tiles_c(int((g > 0).sum()), n[0], n[1], T, E, K, I, f4)
                assert pick if cnt is ten else not pick if cnt is even else True, (T, K, n)


@pytest.mark.parametrize("H,I,f4", [(2048, 512, 0), (2048, 512, 1), (2560, 640, 0), (2560, 640, 1)])
def test_selection_waves_never_share_a_logits_buffer(shim, H, I, f4):
    """k_pf_select reads the router GEMM's slices and stores their sum plus the
    bias. One slice lies in the output's own region, where a second wave of the
    same token would race with the first one's stores: four waves a token only
    over two or more slices, and those fit the region that they borrow."""
    E = 512
    assert not any(shim.pf_select_split_c(T, H, 1) for T in range(9, 2000))
    for K in (1, 2, 9, 10, 16):
        for has_sh in (True, False):
            for T in [9, 600, 601, 800, 801, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 16384]:
                off, by, m = layout(shim, T, H, I, E, K, has_sh, GU_F4 if f4 else GU_I8, GU_F4 if f4 else DN_I8)
                part, lg = by[NAMES.index("part")], by[NAMES.index("lg")]
                n = shim.pf_router_slices_c(T, E, C.c_ulonglong(int(part)))
                assert n in (1, 2, 4) and n * T * E * 4 <= (part if n > 1 else lg)
                assert not shim.pf_select_split_c(T, H, n) or n > 1


def test_library_sizes_match_the_layout(shim):
    """qfm_workspace_bytes (M > 8) = the workspace's tag header (256 bytes of row
    tags, 8 rows x E 8-byte logit words and 8 rows x (K + 1) slots x H 8-byte
    partial words, kept by the M <= 8 forward) + the larger of the INT8 and
    NVFP4 layouts with the shared expert, at the tile widths the library is
    built with."""
    import qfm
    lib = qfm.load()
    for H, I in SHAPES:
        hdr = 256 + 8 * 512 * 8 + 8 * 11 * H * 8
        qfm.init(H, I, 512, 10, 1, 1)
        for T in TS:
            a = layout(shim, T, H, I, 512, 10, True, GU_I8, DN_I8)[2]["total"]
            b = layout(shim, T, H, I, 512, 10, True, GU_F4, GU_F4)[2]["total"]
            assert lib.qfm_workspace_bytes(T) == hdr + max(a, b), (H, T)
    qfm.init(2048, 512, 512, 10, 1, 1)
