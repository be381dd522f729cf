"""GPU routing beyond the exact router's rows (601 and more): the bf16 MFMA
router, its candidates and their exact recomputation (k_pf_router_mfma,
k_pf_select), four waves a token and one, over the K slices of the router GEMM.

Selection bit-exact and weights against the CPU oracle's router and top-K; the
workspace counter says how many tokens had more than 64 candidates.
"""
import ctypes as C
import sys

import numpy as np
import pytest

import _oracle as orc
import qfm

pytestmark = pytest.mark.gpu

E = 512
SHAPES = {2048: 512, 2560: 640}


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def lib():
    L = qfm.load()
    assert qfm.device_info()["arch"].startswith("gfx950")
    yield L
    qfm.init(2048, 512, E, 10, 1, 1)


def _route(lib, H, T, K, bias=None, renorm=1, x=None, router=None, fmt=qfm.QFM_FMT_NVFP4):
    """qfm_moe_forward's routing of T rows and the oracle's: got, ref (sel, wts), counters."""
    seed, layer = 12, 7
    _say("routing H", H, "T", T, "K", K, "bias", bias is not None, "renorm", renorm)
    qfm.init(H, SHAPES[H], E, K, renorm, 1)
    st = qfm.Stream()
    L = qfm.SynthLayer(fmt, seed, layer, stream=st)
    st.sync()                            # generated on st; the router and bias are the test's own
    W = orc.fill("gauss", seed, layer, orc.T_ROUTER, 0, E * H, 0.02).reshape(E, H) if router is None else router
    if x is None:
        x = orc.fill("gauss_bf16", seed, 40, orc.T_X, 0, T * H).reshape(T, H)
    lay = qfm.QfmLayer.from_buffer_copy(L.s.layer)
    dW, dx, dy = qfm.DevBuf.from_array(W), qfm.DevBuf.from_array(x), qfm.DevBuf(T * H * 2)
    db = None if bias is None else qfm.DevBuf.from_array(np.ascontiguousarray(bias, np.float32))
    lay.router, lay.router_bias = dW.ptr, db.ptr if db else None
    wsb = lib.qfm_workspace_bytes(T)
    ws = qfm.DevBuf(wsb)
    qfm.check(lib.qfm_moe_forward(C.byref(lay), dx.ptr, T, dy.ptr, ws.ptr, wsb, st.h), "forward")
    st.sync()
    view = qfm.QfmWsView()
    lib.qfm_workspace_view(ws.ptr, T, C.byref(view))
    got = qfm.d2h(view.sel, np.int32, (T, K)), qfm.d2h(view.wts, np.float32, (T, K))
    counters = qfm.d2h(view.counters, np.int32, 3)
    sel, w, _ = orc.topk(orc.router_logits(W, x, bias), K, renorm)
    for b in (dW, dx, dy, ws) + ((db,) if db else ()):
        b.free()
    L.destroy()
    st.destroy()
    _say("  tokens with more than 64 candidates", int(counters[0]))
    return got, (sel, w), counters


def _check(got, ref):
    assert np.array_equal(got[0], ref[0])
    assert np.allclose(got[1], ref[1], rtol=2e-6, atol=1e-7)


# ------------------------------------------------------------------ candidates
@pytest.mark.parametrize("H,T,K,per", [(2048, 601, 16, 4), (2048, 1200, 16, 4), (2560, 601, 16, 4), (2560, 1500, 10, 3),
                                       (2048, 601, 16, 10), (2560, 1200, 16, 10)])
def test_hot_experts_in_few_lanes(lib, H, T, K, per):
    """A lane of the selecting wave holds the experts that agree modulo 64. A
    bias of +6 on experts 64 j + {0 .. per - 1} puts the hot experts into `per`
    lanes, fewer than top_k. The candidate bound must be the K-th largest lower
    bound all the same, not a cold expert's as the K-th largest lane maximum is:
    no token then has more than 64 candidates. With per = 10 more than 64
    experts (80 hot ones) lie above that lane maximum."""
    bias = np.zeros(E, np.float32)
    for j in range(8):
        bias[64 * j:64 * j + per] = 6.0
    got, ref, counters = _route(lib, H, T, K, bias)
    _check(got, ref)
    assert counters[0] == 0


@pytest.mark.parametrize("H,T,K,finite", [(2048, 601, 10, 212), (2048, 1200, 16, 212), (2560, 1200, 10, 212),
                                          (2048, 601, 10, 10), (2048, 4100, 10, 300), (2560, 601, 10, 6)])
def test_masked_experts(lib, H, T, K, finite):
    """Experts masked by a router bias of -inf are no candidates while top_k
    others are left (their bounds are not NaN), and none is selected. With fewer
    than top_k left every expert is a candidate, and the masked ones follow in
    index order with weight 0."""
    keep = np.random.default_rng(3).permutation(E)[:finite]
    bias = np.full(E, -np.inf, np.float32)
    bias[keep] = 0.0
    got, ref, counters = _route(lib, H, T, K, bias)
    _check(got, ref)
    if finite >= K:
        assert counters[0] == 0 and np.isin(got[0], keep).all()
    else:
        assert counters[0] == T and not got[1][:, finite:].any()


@pytest.mark.parametrize("H,T,bias", [(2048, 601, False), (2048, 1200, True), (2560, 601, True), (2560, 1200, False),
                                      (2560, 2100, True), (2560, 4200, False)])
def test_near_ties_exact_order(lib, H, T, bias):
    """Router rows whose bf16 roundings coincide, so that the MFMA logits of the
    9th..12th experts of token 0 are equal while the exact ones differ by a few
    ulps, with an exact duplicate (the lower index wins): only the exact
    recomputation orders them. Four slices of H and four waves a token, four and
    one, two and one, one and one."""
    rng = np.random.default_rng(T)
    W = orc.fill("gauss", 12, 7, orc.T_ROUTER, 0, E * H, 0.02).reshape(E, H).copy()
    x = orc.fill("gauss_bf16", 12, 40, orc.T_X, 0, T * H).reshape(T, H)
    b = np.zeros(E, np.float32)
    if bias:
        b[:] = rng.choice([0.0, 0.25, 0.5], E)
    order = np.argsort(-orc.router_logits(W, x[:1], b)[0].astype(np.float64), kind="stable")
    base, near = int(order[8]), [int(e) for e in order[20:24]]
    k = int(np.argmax(np.abs(orc.bf16_to_f32(x[0]))))
    for j, e in enumerate(near):
        W[e], b[e] = W[base], b[base]
        for _ in range(j):                                   # near[0]: the duplicate
            W[e, k] = np.nextafter(W[e, k], np.float32(np.inf if j % 2 else -np.inf))
    bits = lambda a: (a.view(np.uint32) + 0x7FFF + ((a.view(np.uint32) >> 16) & 1)) >> 16
    assert all(np.array_equal(bits(W[e]), bits(W[base])) for e in near)
    got, ref, _ = _route(lib, H, T, 10, bias=b if bias else None, x=x, router=W)
    _check(got, ref)


# ------------------------------------------------------------------ counters
@pytest.mark.parametrize("H,T,fmt,renorm,per", [(2048, 40, 0, 1, 16), (2048, 40, 1, 0, 16), (2560, 601, 1, 0, 16),
                                                (2048, 601, 1, 1, 16), (2560, 1200, 0, 1, 16), (2048, 1300, 0, 0, 64),
                                                (2048, 2900, 0, 0, 128), (2560, 1801, 0, 0, 128), (2560, 2501, 1, 1, 256)])
def test_workspace_counters(lib, H, T, fmt, renorm, per):
    """The view's counters: the tokens with more than 64 candidates (here the
    zero rows, whose logits all tie), with and without renormalization, and the
    blocks of work of the two GEMMs, from the selection: items of `per` rows of
    one expert times the weight blocks of each."""
    K, I = 10, SHAPES[H]
    x = orc.fill("gauss_bf16", 12, 41, orc.T_X, 0, T * H).reshape(T, H)
    zero = [0, 7, T - 1]
    x[zero] = 0
    got, ref, counters = _route(lib, H, T, K, x=x, renorm=renorm, fmt=fmt)
    _check(got, ref)
    rows = min(per, 128)                                 # (256: NVFP4 tiles of 128 rows, 256 down columns)
    items = int((-(-np.bincount(got[0].ravel(), minlength=E) // rows)).sum()) - (-T // rows)   # and the shared expert's
    gate_up, down = {16: (I // 64, H // 256), 64: (I // 64, H // 512), 128: (I // 128, H // 128), 256: (I // 128, H // 256)}[per]
    assert counters.tolist() == [len(zero), items * gate_up, items * down]
