"""GPU parity on the edge cases of the decode formats and the selection:

* X8 quantization on exact ties (v = (k + 1/2) s): round half to even, bit-exact;
* middle-row tokens whose x row is zero: every expert is a candidate (the exact
  form of the ranking's bound), ties go to the lowest expert index, and the
  workspace counter reports those tokens (the MFMA router's own overflow:
  test_gpu_routing.py);
* middle rows around whole items, crowded on few experts (the 128-row tiles then
  take them) and at their upper edge, and the 128-row tiles' own path from its
  shortest calls on, at both shapes;
* fork rows (M <= 8) whose experts coincide, all rows on the same ten experts
  or a mix of shared and private ones (each distinct expert's pair range
  staged past its first two rows);
* selection on constructed near-ties: router rows whose bf16 roundings coincide
  (here at 33 rows through the exact router; through the MFMA logits, which cannot
  order them: test_gpu_routing.py);
* every E4M3 block-scale byte 0x00..0xFF (bytes >= 0x80 are large unsigned
  scales, 0x7F is +inf, as the reference decodes them) through every NVFP4
  path: the fused fork-row kernels, the middle rows' items, the 128-row tiles and
  the reference-named M=1 / M=8 tiers, against the oracle's dequantization of the
  same codes and scale bytes.
"""
import ctypes as C
import sys

import numpy as np
import pytest

import _oracle as orc
import qfm

pytestmark = pytest.mark.gpu

TOL = 1e-2
H, I, E, K = 2048, 512, 512, 10


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def lib():
    L = qfm.load()
    qfm.init(H, I, E, K, 1, 1)
    assert qfm.device_info()["arch"].startswith("gfx950")
    return L


def _rel(y, r):
    return float(np.abs(y - r).max() / np.abs(r).max())


def _sync(lib):
    qfm.check(lib.qfm_device_sync(), "sync")
    qfm.status_check()


def _forward(lib, lay, x_bits, st):
    """qfm_moe_forward on bf16 rows x_bits [M][H]; returns y (fp32 of the bf16
    output), sel, wts and the prefill counters (None for M <= 8)."""
    M = x_bits.shape[0]
    dx, dy = qfm.DevBuf.from_array(x_bits), qfm.DevBuf(M * H * 2)
    wsb = lib.qfm_workspace_bytes(M)
    ws = qfm.DevBuf(wsb)
    qfm.check(lib.qfm_moe_forward(C.byref(lay), dx.ptr, M, dy.ptr, ws.ptr, wsb, st.h), "forward")
    st.sync()
    view = qfm.QfmWsView()
    lib.qfm_workspace_view(ws.ptr, M, C.byref(view))
    out = dict(y=orc.bf16_to_f32(dy.download(np.uint16, (M, H))), sel=qfm.d2h(view.sel, np.int32, (M, K)),
               wts=qfm.d2h(view.wts, np.float32, (M, K)))
    out["counters"] = qfm.d2h(view.counters, np.int32, 3) if view.counters else None
    return out


# ------------------------------------------------------------------ X8 ties
def test_x8_ties_bit_exact(lib):
    """qf8_i8_x8 rounds exact ties half to even like the reference's rintf
    (qf8_moe_i8.hip:66): absmax 127 gives the scale 1.0 exactly."""
    _say("x8 ties")
    ties = np.array([0.5, 1.5, 2.5, 3.5, -0.5, -1.5, -2.5, 126.5, -126.5, 5.5, 6.5, -7.5], np.float32)
    v = np.zeros(128, np.float32)
    for blk, sgn in ((0, 1), (1, -1), (2, 1), (3, -1)):
        v[32 * blk] = 127.0 * sgn
        v[32 * blk + 1:32 * blk + 1 + ties.size] = sgn * ties
    dv, dq, ds = qfm.DevBuf.from_array(v), qfm.DevBuf(v.size), qfm.DevBuf(v.size // 32 * 4)
    qfm.check(lib.qf8_i8_x8_ex(dv.ptr, dq.ptr, ds.ptr, v.size, None), "x8")
    _sync(lib)
    q, s = orc.x8_quant(v)
    gq = dq.download(np.int8, v.size)
    assert np.array_equal(gq, q)
    assert np.array_equal(ds.download(np.float32, v.size // 32).view(np.uint32), s.view(np.uint32))
    assert np.array_equal(gq[1:1 + ties.size], np.rint(ties).astype(np.int8))


# ------------------------------------------------------------------ middle rows: zero rows
@pytest.mark.parametrize("bias", [False, True])
def test_prefill_zero_rows_fallback(lib, bias):
    """Zero x rows of a middle call (k_mid_topk): without a router bias every logit
    is 0, all 512 experts share the ranking's prefix bound (its exact form), and the
    selection is experts 0..9 (ties to the lower index) with equal weights; the
    counter reports exactly those rows. With a bias the logits are the bias values
    and the selection is their top 10."""
    T, seed, layer, xl = 40, 2, 31, 77
    zero = [0, 5, 17, 39]
    _say("prefill zero rows, bias", bias)
    qfm.init(H, I, E, K, 1, 1)
    st = qfm.Stream()
    L = qfm.SynthLayer(qfm.QFM_FMT_INT8, seed, layer, with_bias=bias, stream=st)
    x = orc.fill("gauss_bf16", seed, xl, orc.T_X, 0, T * H).reshape(T, H)
    x[zero] = 0
    g = _forward(lib, L.s.layer, x, st)
    r = orc.moe_layer_grouped(H, I, E, K, T, seed, layer, xl, use_bias=int(bias), x=x)
    assert np.array_equal(g["sel"], r["sel"])
    assert np.allclose(g["wts"], r["w"], rtol=2e-6, atol=1e-7)
    if not bias:
        assert np.array_equal(g["sel"][zero], np.tile(np.arange(K), (len(zero), 1)))
        assert np.allclose(g["wts"][zero], 0.1, rtol=1e-6)
        assert g["counters"][0] == len(zero), g["counters"]
    else:
        assert g["counters"][0] == 0, g["counters"]
    assert not g["y"][zero].any() and not r["y"][zero].any()     # zero rows: every expert outputs 0
    rel = max(_rel(g["y"][t], r["y"][t]) for t in range(T) if t not in zero)
    _say("  max rel err", rel, "fallback rows", int(g["counters"][0]))
    assert rel <= TOL
    L.destroy()
    st.destroy()


# ------------------------------------------------------------------ prefill: tile boundaries
@pytest.mark.parametrize("T,fmt", [(128, 0), (129, 0), (256, 1), (383, 0)])
def test_prefill_tile_boundaries(lib, T, fmt):
    """A router bias of +64 on experts 100..109 (and -64 elsewhere) sends every
    token to exactly those ten experts: eleven groups (with the shared one) of
    T rows each, i.e. whole 16-row items (T = 128, 256), one spare row (129), or 15
    rows over (383), and 502 experts with no rows at all (the 128-row tiles of such
    calls begin at 384 rows: test_middle_rows_crowded, test_tiles_beyond_middle).
    Routing bit-exact and every output row against the grouped fp64 oracle given
    the same bias."""
    seed, layer, xl = 4, 23, 91
    _say("prefill tile boundaries T", T, "fmt", fmt)
    qfm.init(H, I, E, K, 1, 1)
    st = qfm.Stream()
    L = qfm.SynthLayer(fmt, seed, layer, with_bias=True, stream=st)
    st.sync()                      # the generator writes the layer on st: finish before overwriting the bias
    bias = np.full(E, -64.0, np.float32)
    bias[100:110] = 64.0 + np.arange(10, dtype=np.float32) * 0.25
    qfm.check(lib.qfm_memcpy_h2d(L.s.layer.router_bias, bias.ctypes.data, bias.nbytes), "bias")
    x = orc.fill("gauss_bf16", seed, xl, orc.T_X, 0, T * H).reshape(T, H)
    g = _forward(lib, L.s.layer, x, st)
    r = orc.moe_layer_grouped(H, I, E, K, T, seed, layer, xl, use_bias=1, x=x, fmt=fmt, bias=bias)
    assert set(np.unique(g["sel"])) == set(range(100, 110))
    assert np.array_equal(g["sel"], r["sel"])
    assert np.allclose(g["wts"], r["w"], rtol=2e-6, atol=1e-7)
    rel = max(_rel(g["y"][t], r["y"][t]) for t in range(T))
    _say("  max rel err", rel, "counters", g["counters"])
    assert rel <= TOL
    L.destroy()
    st.destroy()


# ------------------------------------------------------------------ NVFP4, one row
@pytest.mark.parametrize("hidden,inter,k,shared,gated,f32", [
    (2048, 512, 1, True, 1, False), (2048, 512, 4, False, 1, True), (2048, 512, 5, True, 0, True),
    (2048, 512, 16, True, 1, False), (2560, 640, 3, True, 1, True), (2560, 640, 4, False, 1, False),
    (2560, 640, 13, True, 0, False), (2560, 640, 16, True, 1, True)])
def test_nvfp4_one_row_steps(lib, hidden, inter, k, shared, gated, f32):
    """One NVFP4 row: the down launch deals the k experts' I / 32 chunks to 64
    lanes in 1 to 5 steps (k around whole steps: 4 x 16 chunks fill one exactly,
    3 and 4 x 20 lie either side of it, 16 x 20 fill five), with the shared expert
    gated, ungated and absent, into bf16 and fp32 rows. Routing bit-exact; y within TOL of the fp64 oracle (hidden values
    and x enter the dots as scaled fp16, 2^-12 each; bf16 result 2^-9)."""
    _say("nvfp4 one row H", hidden, "K", k, "shared", shared, "gated", gated, "f32", f32)
    qfm.init(hidden, inter, E, k, 1, gated)
    st = qfm.Stream()
    seed, layer, xl = 9, 5, 70
    L = qfm.SynthLayer(qfm.QFM_FMT_NVFP4, seed, layer, stream=st)
    lay = qfm.QfmLayer.from_buffer_copy(L.s.layer)
    if not shared:
        lay.sh_gate, lay.sh_up, lay.sh_down, lay.sh_gate_inp = qfm.Qf8I8Mat(), qfm.Qf8I8Mat(), qfm.Qf8I8Mat(), None
    x = orc.fill("gauss_bf16", seed, xl, orc.T_X, 0, hidden).reshape(1, hidden)
    dx, dy = qfm.DevBuf.from_array(x), qfm.DevBuf(hidden * 4)
    wsb = lib.qfm_workspace_bytes(1)
    ws = qfm.DevBuf(wsb)
    fwd = lib.qfm_moe_forward_f32 if f32 else lib.qfm_moe_forward
    for _ in range(2):                                   # the second call on a used workspace
        qfm.check(fwd(C.byref(lay), dx.ptr, 1, dy.ptr, ws.ptr, wsb, st.h), "forward")
    st.sync()
    view = qfm.QfmWsView()
    lib.qfm_workspace_view(ws.ptr, 1, C.byref(view))
    y = dy.download(np.float32, (hidden,)) if f32 else orc.bf16_to_f32(dy.download(np.uint16, (hidden,)))
    zero = None if shared else (np.zeros((inter, hidden)), np.zeros((inter, hidden)), np.zeros((hidden, inter)))
    r = orc.moe_layer_grouped(hidden, inter, E, k, 1, seed, layer, xl, x=x, fmt=1, gated=gated, shared=zero)
    assert np.array_equal(qfm.d2h(view.sel, np.int32, (1, k)), r["sel"])
    assert np.allclose(qfm.d2h(view.wts, np.float32, (1, k)), r["w"], rtol=2e-6, atol=1e-7)
    assert _rel(y, r["y"][0]) <= TOL
    L.destroy()
    st.destroy()
    qfm.init(H, I, E, K, 1, 1)


# ------------------------------------------------------------------ middle row counts
@pytest.mark.parametrize("hidden,inter,T,fmt,hot", [
    (2048, 512, 9, 1, 0), (2048, 512, 16, 0, 16), (2048, 512, 33, 1, 17), (2560, 640, 31, 0, 33), (2560, 640, 17, 1, 1),
    (2560, 640, 65, 1, 65), (2560, 640, 601, 0, 65), (2048, 512, 1300, 0, 65)])
def test_middle_rows(lib, hidden, inter, T, fmt, hot):
    """9 to 2800 rows (2560/640: 1800 INT8, 2500 NVFP4) run as weight-streaming
    items of 16 (2048/512 INT8 from 24 rows an expert: 64) rows per expert.
    `hot` rows are copies of row 0, so that its ten experts get at least that
    many rows: counts at and around whole items, beside experts with one row and
    with none. Routing bit-exact, the exact logits in the workspace view, and y
    within TOL of the grouped fp64 oracle (16-bit hidden values and partials)."""
    _say("middle rows H", hidden, "T", T, "fmt", fmt, "hot", hot)
    qfm.init(hidden, inter, E, K, 1, 1)
    st = qfm.Stream()
    seed, layer, xl = 6, 3, 60
    L = qfm.SynthLayer(fmt, seed, layer, stream=st)
    x = orc.fill("gauss_bf16", seed, xl, orc.T_X, 0, T * hidden).reshape(T, hidden)
    x[:hot] = x[0]
    dx, dy = qfm.DevBuf.from_array(x), qfm.DevBuf(T * hidden * 2)
    wsb = lib.qfm_workspace_bytes(T)
    ws = qfm.DevBuf(wsb)
    for _ in range(2):                                   # the second call on a used workspace
        qfm.check(lib.qfm_moe_forward(C.byref(L.s.layer), dx.ptr, T, dy.ptr, ws.ptr, wsb, st.h), "forward")
    st.sync()
    view = qfm.QfmWsView()
    lib.qfm_workspace_view(ws.ptr, T, C.byref(view))
    y = orc.bf16_to_f32(dy.download(np.uint16, (T, hidden)))
    r = orc.moe_layer_grouped(hidden, inter, E, K, T, seed, layer, xl, x=x, fmt=fmt)
    assert np.array_equal(qfm.d2h(view.sel, np.int32, (T, K)), r["sel"])
    assert np.allclose(qfm.d2h(view.wts, np.float32, (T, K)), r["w"], rtol=2e-6, atol=1e-7)
    if T <= 600:                                         # (beyond: approximate logits, exact ones for the candidates)
        W = orc.fill("gauss", seed, layer, orc.T_ROUTER, 0, E * hidden, scale=0.02).reshape(E, hidden)
        rows = [0, T // 2, T - 1]
        lg = qfm.d2h(view.logits, np.float32, (T, E))
        assert np.array_equal(lg[rows].view(np.uint32), orc.router_logits(W, x[rows]).view(np.uint32))
    rel = max(_rel(y[t], r["y"][t]) for t in range(T))
    _say("  max rel err", rel)
    assert rel <= TOL
    L.destroy()
    st.destroy()
    qfm.init(H, I, E, K, 1, 1)


@pytest.mark.parametrize("fmt", [0, 1])
def test_middle_rows_upper_edge(lib, fmt):
    """The largest middle call and the smallest prefill call on the same rows:
    the same routing, and y rows that differ by the two paths' 16-bit roundings
    only (hidden values 2^-9 against 2^-12, partials and y alike: well below
    TOL of the largest value)."""
    _say("middle rows, upper edge, fmt", fmt)
    qfm.init(H, I, E, K, 1, 1)
    st = qfm.Stream()
    T = 2800
    L = qfm.SynthLayer(fmt, 8, 2, stream=st)
    x = orc.fill("gauss_bf16", 8, 61, orc.T_X, 0, (T + 1) * H).reshape(T + 1, H)
    a, b = _forward(lib, L.s.layer, x[:T], st), _forward(lib, L.s.layer, x, st)
    assert np.array_equal(a["sel"], b["sel"][:T]) and np.allclose(a["wts"], b["wts"][:T], rtol=2e-6, atol=1e-7)
    assert max(_rel(a["y"][t], b["y"][t]) for t in range(T)) <= TOL
    L.destroy()
    st.destroy()


def _gemm_blocks(sel, T, hidden, inter, fmt, shared, tiles):
    """Blocks of gate/up and down work of a call with this selection: the middle
    path's items, or 128-row tiles."""
    cnt = np.bincount(sel.ravel(), minlength=E)
    four = fmt == 0 and inter <= 512 and sel.size // E >= 24
    per = 128 if tiles else 64 if four else 16
    n = int((-(-cnt // per)).sum()) + (-(-T // per) if shared else 0)
    if tiles:
        return [n * (inter // 128), n * (hidden // (256 if fmt else 128))]
    return [n * (inter // 64), n * (hidden // (512 if four else 256))]


@pytest.mark.parametrize("hidden,inter,T,fmt,k,shared,gated,tiles", [
    (2560, 640, 256, 0, 10, True, 1, True), (2560, 640, 257, 1, 10, True, 0, True), (2560, 640, 255, 0, 10, True, 1, False),
    (2048, 512, 384, 1, 10, False, 1, True), (2048, 512, 511, 0, 10, True, 1, True), (2048, 512, 640, 0, 4, True, 0, True),
    (2560, 640, 769, 0, 10, False, 1, True), (2560, 640, 895, 1, 16, True, 1, True), (2048, 512, 1281, 0, 10, True, 1, True),
    (2048, 512, 1281, 1, 10, True, 1, True)])
def test_middle_rows_crowded(lib, hidden, inter, T, fmt, k, shared, gated, tiles):
    """Middle calls whose rows all go to the same k experts (a router bias of +64
    on them): from 256 (2560/640) or 384 rows on the plan leaves such a call to the
    128-row tiles, read from its own pairs; the groups hold T rows each, whole
    tiles, one row more and one fewer. Below, items of 16 rows. The counters say
    which ran; an fp32 result keeps the items. Up to 600 rows the row sums of x that the tiles correct their offsets
    with come from k_mid_router, beyond from the MFMA router's prep launch.
    Routing bit-exact, y within TOL of the grouped fp64 oracle; crowded calls and
    calls with spread rows in turn on one workspace, each repeats its first result
    bit for bit."""
    _say("middle rows crowded H", hidden, "T", T, "fmt", fmt, "K", k, "shared", shared, "gated", gated)
    qfm.init(hidden, inter, E, k, 1, gated)
    st = qfm.Stream()
    seed, layer, xl = 4, 23, 92
    L = qfm.SynthLayer(fmt, seed, layer, with_bias=True, stream=st)
    st.sync()
    bias = np.full(E, -64.0, np.float32)
    bias[100:100 + k] = 64.0 + np.arange(k, dtype=np.float32) * 0.25
    dbias = qfm.DevBuf.from_array(bias)
    lay = qfm.QfmLayer.from_buffer_copy(L.s.layer)
    if not shared:
        lay.sh_gate, lay.sh_up, lay.sh_down, lay.sh_gate_inp = qfm.Qf8I8Mat(), qfm.Qf8I8Mat(), qfm.Qf8I8Mat(), None
    x = orc.fill("gauss_bf16", seed, xl, orc.T_X, 0, T * hidden).reshape(T, hidden)
    dx, dy = qfm.DevBuf.from_array(x), qfm.DevBuf(T * hidden * 2)
    wsb = lib.qfm_workspace_bytes(T)
    ws = qfm.DevBuf(wsb)
    view = qfm.QfmWsView()
    ys = []
    for crowd in (False, True, False, True):
        lay.router_bias = dbias.ptr if crowd else None
        qfm.check(lib.qfm_moe_forward(C.byref(lay), dx.ptr, T, dy.ptr, ws.ptr, wsb, st.h), "forward")
        st.sync()
        lib.qfm_workspace_view(ws.ptr, T, C.byref(view))
        sel = qfm.d2h(view.sel, np.int32, (T, k))
        counters = qfm.d2h(view.counters, np.int32, 3).tolist()
        assert counters[1:] == _gemm_blocks(sel, T, hidden, inter, fmt, shared, tiles and crowd), (crowd, counters)
        ys.append(dy.download(np.uint16, (T, hidden)))
    zero = None if shared else (np.zeros((inter, hidden)), np.zeros((inter, hidden)), np.zeros((hidden, inter)))
    r = orc.moe_layer_grouped(hidden, inter, E, k, T, seed, layer, xl, use_bias=1, x=x, fmt=fmt, bias=bias, gated=gated,
                              shared=zero)
    assert np.array_equal(sel, r["sel"]) and set(np.unique(sel)) == set(range(100, 100 + k))
    assert np.allclose(qfm.d2h(view.wts, np.float32, (T, k)), r["w"], rtol=2e-6, atol=1e-7)
    y = orc.bf16_to_f32(ys[1])
    rel = max(_rel(y[t], r["y"][t]) for t in range(T))
    _say("  max rel err", rel)
    assert rel <= TOL
    assert np.array_equal(ys[0], ys[2]) and np.array_equal(ys[1], ys[3])
    dy32 = qfm.DevBuf(T * hidden * 4)
    qfm.check(lib.qfm_moe_forward_f32(C.byref(lay), dx.ptr, T, dy32.ptr, ws.ptr, wsb, st.h), "forward f32")
    st.sync()
    counters = qfm.d2h(view.counters, np.int32, 3).tolist()
    assert counters[1:] == _gemm_blocks(sel, T, hidden, inter, fmt, shared, False)
    y = dy32.download(np.float32, (T, hidden)).astype(np.float64)
    err = float(np.linalg.norm(y - r["y"]) / np.linalg.norm(r["y"]))
    _say("  fp32 result: error (2-norm)", err)
    # hidden rows rounded to 11 bits (2^-12 of a value) and partials to 11 bits of their
    # 64 columns' largest, 3 times the root mean square: 4 x 2^-12 (bf16 hidden rows: 1.7e-3)
    assert err <= 4 * 2.0 ** -12
    L.destroy()
    st.destroy()
    qfm.init(H, I, E, K, 1, 1)


@pytest.mark.parametrize("hidden,inter,T,fmt,shared,gated,hot", [
    (2560, 640, 1801, 0, True, 1, 10), (2560, 640, 1919, 0, True, 0, 24), (2560, 640, 2501, 1, True, 0, 24),
    (2560, 640, 2817, 1, False, 1, 10), (2048, 512, 2944, 0, False, 1, 10), (2048, 512, 2943, 1, True, 1, 24),
    (2048, 512, 2945, 0, True, 0, 24)])
def test_tiles_beyond_middle(lib, hidden, inter, T, fmt, shared, gated, hot):
    """The shortest calls of the 128-row tiles' own path (a block per tile) and
    row counts around whole tiles, at both shapes and formats, gated, ungated and
    without a shared expert. A bias of +64 on `hot` experts sends every row to ten
    of them: groups of T rows (ten) or of uneven sizes, few experts for the fp64
    oracle. The counters say that the tiles ran."""
    _say("tiles beyond middle H", hidden, "T", T, "fmt", fmt, "shared", shared, "gated", gated, "hot", hot)
    qfm.init(hidden, inter, E, K, 1, gated)
    st = qfm.Stream()
    seed, layer, xl = 4, 24, 95
    L = qfm.SynthLayer(fmt, seed, layer, with_bias=True, stream=st)
    st.sync()
    bias = np.full(E, -64.0, np.float32)
    bias[100:100 + hot] = 64.0
    qfm.check(lib.qfm_memcpy_h2d(L.s.layer.router_bias, bias.ctypes.data, bias.nbytes), "bias")
    lay = qfm.QfmLayer.from_buffer_copy(L.s.layer)
    if not shared:
        lay.sh_gate, lay.sh_up, lay.sh_down, lay.sh_gate_inp = qfm.Qf8I8Mat(), qfm.Qf8I8Mat(), qfm.Qf8I8Mat(), None
    x = orc.fill("gauss_bf16", seed, xl, orc.T_X, 0, T * hidden).reshape(T, hidden)
    dx, dy = qfm.DevBuf.from_array(x), qfm.DevBuf(T * hidden * 4)
    wsb = lib.qfm_workspace_bytes(T)
    ws = qfm.DevBuf(wsb)
    qfm.check(lib.qfm_moe_forward_f32(C.byref(lay), dx.ptr, T, dy.ptr, ws.ptr, wsb, st.h), "forward")
    st.sync()
    view = qfm.QfmWsView()
    lib.qfm_workspace_view(ws.ptr, T, C.byref(view))
    sel = qfm.d2h(view.sel, np.int32, (T, K))
    assert qfm.d2h(view.counters, np.int32, 3).tolist()[1:] == _gemm_blocks(sel, T, hidden, inter, fmt, shared, True)
    zero = None if shared else (np.zeros((inter, hidden)), np.zeros((inter, hidden)), np.zeros((hidden, inter)))
    r = orc.moe_layer_grouped(hidden, inter, E, K, T, seed, layer, xl, use_bias=1, x=x, fmt=fmt, bias=bias, gated=gated,
                              shared=zero)
    assert np.array_equal(sel, r["sel"])
    assert np.allclose(qfm.d2h(view.wts, np.float32, (T, K)), r["w"], rtol=2e-6, atol=1e-7)
    y = dy.download(np.float32, (T, hidden))
    rel = max(_rel(y[t], r["y"][t]) for t in range(T))
    _say("  max rel err", rel)
    assert rel <= TOL
    L.destroy()
    st.destroy()
    qfm.init(H, I, E, K, 1, 1)


@pytest.mark.parametrize("hidden,inter,T,fmt", [(2048, 512, 2800, 0), (2560, 640, 1800, 0), (2560, 640, 2500, 1)])
def test_middle_rows_fp32_top16(lib, hidden, inter, T, fmt):
    """The largest fp32 middle calls at top-16, where a bf16 result runs the tiles:
    both forms of one call on the same rows, by the counters; routing the same, y
    apart by the tiles' 8-bit hidden rows and the bf16 result (2^-9 each)."""
    _say("middle rows fp32 top-16 H", hidden, "T", T, "fmt", fmt)
    qfm.init(hidden, inter, E, 16, 1, 1)
    st = qfm.Stream()
    L = qfm.SynthLayer(fmt, 8, 3, stream=st)
    x = orc.fill("gauss_bf16", 8, 62, orc.T_X, 0, T * hidden).reshape(T, hidden)
    dx, dy = qfm.DevBuf.from_array(x), qfm.DevBuf(T * hidden * 4)
    wsb = lib.qfm_workspace_bytes(T)
    ws = qfm.DevBuf(wsb)
    view = qfm.QfmWsView()
    got = []
    for f32 in (False, True):
        fwd = lib.qfm_moe_forward_f32 if f32 else lib.qfm_moe_forward
        qfm.check(fwd(C.byref(L.s.layer), dx.ptr, T, dy.ptr, ws.ptr, wsb, st.h), "forward")
        st.sync()
        lib.qfm_workspace_view(ws.ptr, T, C.byref(view))
        sel = qfm.d2h(view.sel, np.int32, (T, 16))
        counters = qfm.d2h(view.counters, np.int32, 3).tolist()
        assert counters[1:] == _gemm_blocks(sel, T, hidden, inter, fmt, True, not f32)
        got.append((sel, dy.download(np.float32, (T, hidden)) if f32 else orc.bf16_to_f32(dy.download(np.uint16, (T, hidden)))))
    assert np.array_equal(got[0][0], got[1][0])
    err = float(np.linalg.norm(got[0][1] - got[1][1]) / np.linalg.norm(got[1][1]))
    _say("  2-norm difference", err)
    assert err <= 2 * 2.0 ** -9
    L.destroy()
    st.destroy()
    qfm.init(H, I, E, K, 1, 1)


# ------------------------------------------------------------------ fork rows sharing experts
@pytest.mark.parametrize("M,fmt,boost", [(2, 0, 64.0), (8, 0, 64.0), (8, 1, 64.0), (8, 0, 1.5), (5, 1, 1.5)])
def test_fork_rows_sharing_experts(lib, M, fmt, boost):
    """Fork rows (M <= 8) whose experts coincide: a router bias of +boost on
    experts 100..109 sends every row to exactly those ten (boost 64: each
    distinct expert carries all M rows, so the gate/up blocks stage rows past
    the first two of their pair range) or makes them likely without forcing
    them (boost 1.5 against logits of spread ~0.9: a mix of shared and
    private experts). Routing bit-exact,
    every row's y against the grouped fp64 oracle with the same bias."""
    seed, layer, xl = 6, 27, 93
    _say("fork rows sharing experts M", M, "fmt", fmt, "boost", boost)
    qfm.init(H, I, E, K, 1, 1)
    st = qfm.Stream()
    L = qfm.SynthLayer(fmt, seed, layer, with_bias=True, stream=st)
    st.sync()
    forced = boost >= 32
    bias = np.full(E, -64.0, np.float32) if forced else np.zeros(E, np.float32)
    bias[100:110] = boost + np.arange(10, dtype=np.float32) * (0.25 if forced else 0.0)
    qfm.check(lib.qfm_memcpy_h2d(L.s.layer.router_bias, bias.ctypes.data, bias.nbytes), "bias")
    x = orc.fill("gauss_bf16", seed, xl, orc.T_X, 0, M * H).reshape(M, H)
    g = _forward(lib, L.s.layer, x, st)
    r = orc.moe_layer_grouped(H, I, E, K, M, seed, layer, xl, use_bias=1, x=x, fmt=fmt, bias=bias)
    assert np.array_equal(g["sel"], r["sel"])
    if forced:
        assert (np.sort(g["sel"], axis=1) == np.arange(100, 110)).all()
    shared = len(np.unique(g["sel"]))
    assert np.allclose(g["wts"], r["w"], rtol=2e-6, atol=1e-7)
    rel = max(_rel(g["y"][t], r["y"][t]) for t in range(M))
    _say("  distinct experts", shared, "of", M * K, "max rel err", rel)
    assert rel <= TOL
    L.destroy()
    st.destroy()


# ------------------------------------------------------------------ prefill: near ties
def test_prefill_near_ties_exact_order(lib):
    """Router rows built so that token 0's 9th..12th experts have identical bf16
    roundings while their exact logits differ by a few ulps, plus one exact
    duplicate (a true tie, lower index wins). The selection of a middle call (exact
    router) must equal the oracle's exact top-K for every token."""
    T, seed, layer, xl = 33, 3, 12, 88
    _say("prefill near ties")
    qfm.init(H, I, E, K, 1, 1)
    st = qfm.Stream()
    L = qfm.SynthLayer(qfm.QFM_FMT_INT8, seed, layer, with_bias=False, stream=st)
    W = orc.fill("gauss", seed, layer, orc.T_ROUTER, 0, E * H, 0.02).reshape(E, H).copy()
    x = orc.fill("gauss_bf16", seed, xl, orc.T_X, 0, T * H).reshape(T, H)
    lg = orc.router_logits(W, x[:1])[0]
    order = np.argsort(-lg.astype(np.float64), kind="stable")
    base = int(order[8])                              # token 0's 9th expert
    targets = [int(e) for e in order[20:24]]          # rows that become near copies of it
    xf = orc.bf16_to_f32(x[0]).astype(np.float64)
    k_big = int(np.argmax(np.abs(xf)))
    for j, e in enumerate(targets):
        W[e] = W[base]
        if j < 3:
            # nudge one weight by a few fp32 ulps: its bf16 rounding is unchanged
            w = np.float32(W[base, k_big])
            W[e, k_big] = np.nextafter(w, np.float32(np.inf) if (j % 2) == (xf[k_big] > 0) else np.float32(-np.inf))
            for _ in range(j):
                W[e, k_big] = np.nextafter(W[e, k_big], np.float32(np.inf) if (j % 2) == (xf[k_big] > 0) else np.float32(-np.inf))
    bf = lambda a: (a.view(np.uint32) + 0x7FFF + ((a.view(np.uint32) >> 16) & 1)) >> 16
    for e in targets:
        assert np.array_equal(bf(W[e]), bf(W[base])), "bf16 roundings coincide"
    dW = qfm.DevBuf.from_array(W)
    lay = qfm.QfmLayer.from_buffer_copy(L.s.layer)
    lay.router = dW.ptr
    g = _forward(lib, lay, x, st)
    r = orc.moe_layer_grouped(H, I, E, K, T, seed, layer, xl, x=x, router=W)
    lg0 = orc.router_logits(W, x[:1])[0]
    _say("  token 0 logits of the tied rows", [float(lg0[e]) for e in [base] + targets], "sel", g["sel"][0].tolist())
    assert np.array_equal(g["sel"], r["sel"])
    assert np.allclose(g["wts"], r["w"], rtol=2e-6, atol=1e-7)
    assert _rel(g["y"][0], r["y"][0]) <= TOL
    L.destroy()
    st.destroy()


# ------------------------------------------------------------------ E4M3 bytes
ALL_BYTES = np.arange(256)
S2 = 0.01


def _e4m3(b):
    return np.array([orc.load().orc_e4m3(int(v)) for v in np.atleast_1d(b)], np.float64)


class _F4Layer:
    """An NVFP4 layer without a shared expert whose e4m3 scale arrays the test
    overwrites; codes and routing stay those of the generator."""

    def __init__(self, lib, seed, layer, bias):
        self.lib, self.seed, self.layer = lib, seed, layer
        self.st = qfm.Stream()
        self.L = qfm.SynthLayer(qfm.QFM_FMT_NVFP4, seed, layer, with_bias=bias, stream=self.st)
        self.st.sync()             # generated on st; the scales are then overwritten from the host
        lay = qfm.QfmLayer.from_buffer_copy(self.L.s.layer)
        lay.sh_gate, lay.sh_up, lay.sh_down, lay.sh_gate_inp = qfm.Qf8I8Mat(), qfm.Qf8I8Mat(), qfm.Qf8I8Mat(), None
        self.lay = lay
        self.a = self.L.s.arena
        self.cache = {}

    def set_scales(self, gate_up_byte=None, down_rows=None):
        """gate/up: every block of every expert = gate_up_byte; down: row c of
        every expert = down_rows[c] for all its blocks."""
        n_gu = E * I * H // 16
        if gate_up_byte is not None:
            qfm.check(self.lib.qfm_memset(self.a.s_gate, int(gate_up_byte), n_gu), "memset")
            qfm.check(self.lib.qfm_memset(self.a.s_up, int(gate_up_byte), n_gu), "memset")
        if down_rows is not None:
            pat = np.repeat(np.asarray(down_rows, np.uint8)[:, None], I // 16, axis=1)
            big = np.ascontiguousarray(np.tile(pat.ravel(), E))
            qfm.check(self.lib.qfm_memcpy_h2d(self.a.s_down, big.ctypes.data, big.nbytes), "h2d")

    def unit(self, e):
        """Expert e's codes read back from the device, dequantized with unit
        block scales (byte 0x38 = 1.0): Wg, Wu, Wd (times s2) in fp64."""
        if e not in self.cache:
            ones_g = np.full((I, H // 16), 0x38, np.uint8)
            ones_d = np.full((H, I // 16), 0x38, np.uint8)
            GW = I * H // 2
            Fg = qfm.d2h(self.a.w_gate + e * GW, np.uint8, (I, H // 2))
            Fu = qfm.d2h(self.a.w_up + e * GW, np.uint8, (I, H // 2))
            Fd = qfm.d2h(self.a.w_down + e * GW, np.uint8, (H, I // 2))
            self.cache[e] = (orc.nvfp4_dequant(Fg, ones_g, S2, I, H), orc.nvfp4_dequant(Fu, ones_g, S2, I, H),
                             orc.nvfp4_dequant(Fd, ones_d, S2, H, I))
        return self.cache[e]

    def check_arrays(self, gate_up_byte, down_rows, experts):
        """The scale bytes the kernels read are the planted ones."""
        for e in list(experts)[:2]:
            sg = qfm.d2h(self.a.s_gate + e * (I * H // 16), np.uint8, I * H // 16)
            sd = qfm.d2h(self.a.s_down + e * (H * I // 16), np.uint8, (H, I // 16))
            assert (sg == gate_up_byte).all()
            assert np.array_equal(sd[:, 0], np.asarray(down_rows, np.uint8))

    def ref(self, x, sel, wts, sg_scale, sd_row_scale):
        """y[t] = sum_k w_k Wd_k (silu(s Wg_k x) * (s Wu_k x)) with the block
        scales applied as exact factors (the dequantized weight is
        e2m1 * e4m3 * s2, a product exact in fp64)."""
        X = orc.bf16_to_f32(x).astype(np.float64) if x.dtype == np.uint16 else x.astype(np.float64)
        y = np.zeros((X.shape[0], H))
        for t in range(X.shape[0]):
            for k in range(sel.shape[1]):
                Wg, Wu, Wd = self.unit(int(sel[t, k]))
                g = sg_scale * (Wg @ X[t])
                u = sg_scale * (Wu @ X[t])
                with np.errstate(over="ignore", invalid="ignore"):
                    h = g / (1.0 + np.exp(-g)) * u
                    y[t] += float(wts[t, k]) * (sd_row_scale * (Wd @ h))
        return y

    def destroy(self):
        self.L.destroy()
        self.st.destroy()


def _paths(lib, F, x_rows, x_pf, rng):
    """Run every NVFP4 decode path on the current scale bytes. Returns a list of
    (name, y, x, sel, wts)."""
    out = []
    g = _forward(lib, F.lay, x_rows, F.st)                       # fused fork-row kernels (M = 2)
    out.append(("fused M=2", g["y"], x_rows, g["sel"], g["wts"]))
    p = _forward(lib, F.lay, x_pf, F.st)                         # middle rows (T = 9)
    out.append(("middle T=9", p["y"], x_pf, p["sel"], p["wts"]))
    a = F.a
    x1 = orc.bf16_to_f32(x_rows[0]).astype(np.float32)
    sel = rng.choice(E, K, replace=False).astype(np.int32)
    wts = (rng.random(K) + 0.1).astype(np.float32)
    dx, dsel, dw = qfm.DevBuf.from_array(x1), qfm.DevBuf.from_array(sel), qfm.DevBuf.from_array(wts)
    hid, y1 = qfm.DevBuf(K * I * 4), qfm.DevBuf(H * 4)
    qfm.check(lib.qf5_nvfp4_moe_all_ex(a.w_gate, a.s_gate, a.w_up, a.s_up, a.w_down, a.s_down, dx.ptr, hid.ptr, y1.ptr,
                                       a.s2g_dev, a.s2u_dev, a.s2d_dev, dw.ptr, dsel.ptr, dsel.ptr, K, None), "moe_all")
    _sync(lib)
    out.append(("compat M=1", y1.download(np.float32, (1, H)), x1[None, :], sel[None, :], wts[None, :]))
    return out


@pytest.fixture(scope="module")
def f4(lib):
    qfm.init(H, I, E, K, 1, 1)
    F = _F4Layer(lib, 9, 21, bias=True)
    yield F
    F.destroy()


def test_e4m3_every_gate_up_byte(lib, f4):
    """Each of the 255 finite scale bytes (0x7F = +inf would make every output
    NaN) in turn as the gate and up block scale of every expert, down scales 1.0:
    the fused fork-row, middle-row and reference-named M=1 paths against the
    oracle's dequantization. Bytes >= 0x80 are scales up to 2^24 * 1.875."""
    _say("e4m3 gate/up bytes")
    x_rows = orc.fill("gauss_bf16", 9, 501, orc.T_X, 0, 2 * H).reshape(2, H)
    x_pf = orc.fill("gauss_bf16", 9, 502, orc.T_X, 0, 9 * H).reshape(9, H)
    f4.set_scales(down_rows=np.full(H, 0x38, np.uint8))
    bytes_ = [b for b in ALL_BYTES if b != 0x7F]
    runs = {}                                        # path -> (x, sel, wts, [y per byte])
    for b in bytes_:
        f4.set_scales(gate_up_byte=b)
        _sync(lib)
        if b in (0x00, 0x80, 0xFF):
            f4.check_arrays(b, np.full(H, 0x38, np.uint8), [0])
        for name, y, x, sel, wts in _paths(lib, f4, x_rows, x_pf, np.random.default_rng(0)):
            if name not in runs:
                runs[name] = (x, sel, wts, [])
            else:                                    # routing does not depend on the expert weights
                assert np.array_equal(runs[name][1], sel), name
            runs[name][3].append(y)
    scales = _e4m3(np.array(bytes_))
    for name, (x, sel, wts, ys) in runs.items():
        Y = np.stack(ys)                                              # [byte][rows][H]
        R = np.zeros_like(Y, dtype=np.float64)
        X = orc.bf16_to_f32(x).astype(np.float64) if x.dtype == np.uint16 else x.astype(np.float64)
        for t in range(X.shape[0]):
            for k in range(sel.shape[1]):
                Wg, Wu, Wd = f4.unit(int(sel[t, k]))
                g = np.outer(scales, Wg @ X[t])                       # [byte][I]
                u = np.outer(scales, Wu @ X[t])
                with np.errstate(over="ignore", invalid="ignore"):
                    h = g / (1.0 + np.exp(-g)) * u
                R[:, t] += float(wts[t, k]) * (h @ Wd.T)
        worst = 0.0
        for i, b in enumerate(bytes_):
            if scales[i] == 0.0:
                assert not Y[i].any(), (name, b)
                continue
            rel = max(_rel(Y[i, t], R[i, t]) for t in range(X.shape[0]))
            worst = max(worst, rel)
            assert rel <= TOL, (name, hex(b), rel)
        _say("  ", name, "worst rel err over the 255 finite bytes", worst)


def test_e4m3_every_down_byte(lib, f4):
    """Down block scales: row c of every expert takes byte c % 256 (all 256
    bytes, eight rows each; gate/up scales 1.0). Rows with a 0x7F (+inf) scale
    must come out non-finite and leave the other rows finite; every other byte's
    rows are checked against the oracle relative to their own magnitude, and a
    zero scale gives exact zeros."""
    _say("e4m3 down bytes")
    rng = np.random.default_rng(4)
    x_rows = orc.fill("gauss_bf16", 9, 503, orc.T_X, 0, 2 * H).reshape(2, H)
    x_pf = orc.fill("gauss_bf16", 9, 504, orc.T_X, 0, 9 * H).reshape(9, H)
    rows = (np.arange(H) % 256).astype(np.uint8)
    f4.set_scales(gate_up_byte=0x38, down_rows=rows)
    _sync(lib)
    f4.check_arrays(0x38, rows, [0])
    srow = _e4m3(rows)
    finite = np.isfinite(srow)
    paths = _paths(lib, f4, x_rows, x_pf, rng)
    # the reference-named M=8 tier (atomic down into a pre-zeroed y), 8 rows
    a = f4.a
    M = 8
    x8 = orc.fill("gauss_bf16", 9, 505, orc.T_X, 0, M * H).reshape(M, H)
    xf = orc.bf16_to_f32(x8).astype(np.float32)
    sel = np.stack([rng.choice(E, K, replace=False) for _ in range(M)]).astype(np.int32)
    wt = (rng.random((M, K)) + 0.1).astype(np.float32)
    P = M * K
    dsel, dwt, dx = qfm.DevBuf.from_array(sel), qfm.DevBuf.from_array(wt), qfm.DevBuf.from_array(xf)
    d_slot, d_ptr, d_tok, d_pw, d_cnt = (qfm.DevBuf(P * 4), qfm.DevBuf((P + 1) * 4), qfm.DevBuf(P * 4),
                                         qfm.DevBuf(P * 4), qfm.DevBuf(8))
    qfm.check(lib.qf5_m8_build_csr_ex(dsel.ptr, dwt.ptr, M, K, 0, E, 0, d_slot.ptr, d_ptr.ptr, d_tok.ptr, d_pw.ptr,
                                      d_cnt.ptr, None), "csr")
    _sync(lib)
    cnt = d_cnt.download(np.int32, 2)
    rt = qfm.Qf5M8Route(0, int(cnt[1]), M, P, d_cnt.ptr, d_slot.ptr, d_ptr.ptr, d_tok.ptr, d_pw.ptr)
    hid, yp = qfm.DevBuf(P * I * 4), qfm.DevBuf.from_array(np.zeros((M, H), np.float32))
    qfm.check(lib.qf5_m8_gateup_ex(a.w_gate, a.s_gate, a.w_up, a.s_up, a.s2g_dev, a.s2u_dev, dx.ptr, hid.ptr,
                                   C.byref(rt), None), "m8 gateup")
    qfm.check(lib.qf5_m8_downacc_ex(a.w_down, a.s_down, a.s2d_dev, hid.ptr, yp.ptr, C.byref(rt), None), "m8 down")
    _sync(lib)
    paths.append(("compat M=8", yp.download(np.float32, (M, H)), xf, sel, wt))
    for name, y, x, sel_, wts_ in paths:
        r = f4.ref(x, sel_, wts_, 1.0, np.where(finite, srow, 0.0))
        assert np.isfinite(y[:, finite]).all(), name
        assert not np.isfinite(y[:, ~finite]).any(), name           # the 0x7F rows
        worst = 0.0
        for b in range(256):
            if b == 0x7F:
                continue
            cols = np.nonzero(rows == b)[0]
            ref_b, got_b = r[:, cols], y[:, cols]
            if srow[b] == 0.0:
                assert not got_b.any(), (name, b)
                continue
            rel = float(np.abs(got_b - ref_b).max() / np.abs(ref_b).max())
            worst = max(worst, rel)
            assert rel <= TOL, (name, hex(b), rel)
        _say("  ", name, "worst rel err over the 255 finite bytes", worst)


def test_e4m3_bytes_in_tiles(lib, f4):
    """Every finite scale byte as the gate and up block scale of every expert
    through the 128-row tiles (384 rows crowded on ten experts), and every byte as
    a down row's scale: three rows (the first, one in the second tile, the last)
    against the oracle's dequantization, as the paths above."""
    T, rows = 384, [0, 200, 383]
    _say("e4m3 bytes in tiles")
    x = orc.fill("gauss_bf16", 9, 506, orc.T_X, 0, T * H).reshape(T, H)
    bias = np.full(E, -64.0, np.float32)
    bias[100:110] = 64.0
    db = qfm.DevBuf.from_array(bias)
    lay = qfm.QfmLayer.from_buffer_copy(f4.lay)
    lay.router_bias = db.ptr
    f4.set_scales(down_rows=np.full(H, 0x38, np.uint8))
    bytes_ = [b for b in ALL_BYTES if b != 0x7F]
    ys = []
    for b in bytes_:
        f4.set_scales(gate_up_byte=b)
        _sync(lib)
        g = _forward(lib, lay, x, f4.st)
        assert g["counters"].tolist()[1:] == _gemm_blocks(g["sel"], T, H, I, 1, False, True)
        ys.append(g["y"][rows])
    sel, wts, scales = g["sel"], g["wts"], _e4m3(np.array(bytes_))
    X = orc.bf16_to_f32(x).astype(np.float64)
    for q, t in enumerate(rows):
        R = np.zeros((len(bytes_), H))
        for k in range(K):
            Wg, Wu, Wd = f4.unit(int(sel[t, k]))
            gg, uu = np.outer(scales, Wg @ X[t]), np.outer(scales, Wu @ X[t])
            with np.errstate(over="ignore", invalid="ignore"):
                R += float(wts[t, k]) * ((gg / (1.0 + np.exp(-gg)) * uu) @ Wd.T)
        for i, b in enumerate(bytes_):
            if scales[i] == 0.0:
                assert not ys[i][q].any(), hex(b)
            else:
                assert _rel(ys[i][q], R[i]) <= TOL, (hex(b), t)
    bytes_c = (np.arange(H) % 256).astype(np.uint8)
    f4.set_scales(gate_up_byte=0x38, down_rows=bytes_c)
    _sync(lib)
    g = _forward(lib, lay, x, f4.st)
    srow = _e4m3(bytes_c)
    finite = np.isfinite(srow)
    r = f4.ref(x[rows], g["sel"][rows], g["wts"][rows], 1.0, np.where(finite, srow, 0.0))
    y = g["y"][rows]
    assert np.isfinite(y[:, finite]).all() and not np.isfinite(y[:, ~finite]).any()
    for b in bytes_:
        cols = np.nonzero(bytes_c == b)[0]
        if srow[b] == 0.0:
            assert not y[:, cols].any(), hex(b)
        else:
            assert float(np.abs(y[:, cols] - r[:, cols]).max() / np.abs(r[:, cols]).max()) <= TOL, hex(b)


# ------------------------------------------------------------------ decode: zero rows
@pytest.mark.parametrize("M,fmt,bias", [(1, 0, False), (3, 0, False), (1, 1, True), (5, 1, False)])
def test_decode_zero_rows(lib, M, fmt, bias):
    """All-zero x rows through the fused decode paths (at M = 1 the INT8 gate/up
    kernel's own selection): without a bias every logit is 0, the selection is
    experts 0..9 (ties to the lower index) with weights 0.1; with a bias the
    logits are the bias and the selection its top 10. Every expert's output is
    0, so y is 0."""
    _say("decode zero rows M", M, "fmt", fmt, "bias", bias)
    qfm.init(H, I, E, K, 1, 1)
    st = qfm.Stream()
    L = qfm.SynthLayer(fmt, 5, 61, with_bias=bias, stream=st)
    st.sync()
    x = np.zeros((M, H), np.uint16)
    g = _forward(lib, L.s.layer, x, st)
    r = orc.moe_layer_grouped(H, I, E, K, M, 5, 61, 0, use_bias=int(bias), x=x, fmt=fmt)
    assert np.array_equal(g["sel"], r["sel"])
    assert np.allclose(g["wts"], r["w"], rtol=2e-6, atol=1e-7)
    if not bias:
        assert np.array_equal(g["sel"], np.tile(np.arange(K), (M, 1)))
        assert np.allclose(g["wts"], 0.1, rtol=1e-6)
    assert not g["y"].any() and not r["y"].any()
    L.destroy()
    st.destroy()


# ------------------------------------------------------------------ dynamic range of x
@pytest.mark.parametrize("M,fmt,shift", [(1, 0, 24), (1, 0, -24), (4, 1, 24), (4, 0, -24), (40, 0, 24), (40, 1, -24)])
def test_input_dynamic_range(lib, M, fmt, shift):
    """x rows scaled by 2^shift (exact in bf16) through the fused decode and
    middle-row paths: the activations as fp16 scaled per token or per 16 values,
    the hidden vectors' fp16 chunks and rows and the scaled fp16 partials must
    follow the magnitude. At 2^24 the softmax is one-hot, at 2^-24 nearly
    uniform; the routing stays bit-exact and y within the usual bound."""
    _say("dynamic range M", M, "fmt", fmt, "shift", shift)
    qfm.init(H, I, E, K, 1, 1)
    st = qfm.Stream()
    L = qfm.SynthLayer(fmt, 7, 71, with_bias=False, stream=st)
    st.sync()
    x0 = orc.fill("gauss_bf16", 7, 600 + M, orc.T_X, 0, M * H).reshape(M, H)
    xf = orc.bf16_to_f32(x0) * np.float32(2.0 ** shift)
    x = (xf.view(np.uint32) >> 16).astype(np.uint16)
    assert np.array_equal(orc.bf16_to_f32(x), xf)                 # the scaling is exact
    g = _forward(lib, L.s.layer, x, st)
    r = orc.moe_layer_grouped(H, I, E, K, M, 7, 71, 0, x=x, fmt=fmt)
    assert np.array_equal(g["sel"], r["sel"])
    assert np.allclose(g["wts"], r["w"], rtol=2e-6, atol=1e-7)
    assert np.isfinite(g["y"]).all()
    rel = max(_rel(g["y"][t], r["y"][t]) for t in range(M))
    _say("  max rel err", rel)
    assert rel <= TOL
    L.destroy()
    st.destroy()


@pytest.mark.parametrize("T,fmt,shift", [(384, 0, 24), (385, 1, 24), (640, 0, -24), (384, 1, -24)])
def test_input_dynamic_range_in_tiles(lib, T, fmt, shift):
    """The same scaled rows through the 128-row tiles (rows crowded on ten experts
    by a bias far above the logits): x as scaled fp16 (INT8) or bf16 with the row
    sums of the offset corrections, bf16 hidden rows and the scaled fp16 partials."""
    _say("dynamic range in tiles T", T, "fmt", fmt, "shift", shift)
    qfm.init(H, I, E, K, 1, 1)
    st = qfm.Stream()
    L = qfm.SynthLayer(fmt, 7, 72, with_bias=True, stream=st)
    st.sync()
    bias = np.full(E, -2.0 ** 30, np.float32)
    bias[100:110] = 2.0 ** 30
    qfm.check(lib.qfm_memcpy_h2d(L.s.layer.router_bias, bias.ctypes.data, bias.nbytes), "bias")
    xf = orc.bf16_to_f32(orc.fill("gauss_bf16", 7, 640, orc.T_X, 0, T * H).reshape(T, H)) * np.float32(2.0 ** shift)
    x = (xf.view(np.uint32) >> 16).astype(np.uint16)
    g = _forward(lib, L.s.layer, x, st)
    assert g["counters"].tolist()[1:] == _gemm_blocks(g["sel"], T, H, I, fmt, True, True)
    r = orc.moe_layer_grouped(H, I, E, K, T, 7, 72, 0, x=x, fmt=fmt, use_bias=1, bias=bias)
    assert np.array_equal(g["sel"], r["sel"])
    assert np.allclose(g["wts"], r["w"], rtol=2e-6, atol=1e-7)
    assert np.isfinite(g["y"]).all()
    rel = max(_rel(g["y"][t], r["y"][t]) for t in range(T))
    _say("  max rel err", rel)
    assert rel <= TOL
    L.destroy()
    st.destroy()
