"""The pair form of the device-routed MoE layer (a few tokens: no grouping, SwiGLU + down + combine in one launch) against the
oracle's moe_n restatement, bit for bit: 1 to 29 tokens, 1 to 16 choices, every K-quant down projection, K-quant and
32-element gate/up projections, one to four blocks of h, output rows that are not a multiple of a workgroup's, every
reference order, experts chosen more than once and choices that name no expert."""
import numpy as np
import pytest

import es_hip_quant as E
import oracle as O
from test_hip_moe import MODES, Experts, bits

pytestmark = pytest.mark.gpu


@pytest.fixture
def hipo(hip):
    yield hip
    hip.set_order(E.ORDER_X86_CONTRACT)


def layer(hip, orc, types, n, ff, n_exp, sel, w, seed, mode=MODES[0]):
    N, k = sel.shape
    ex = Experts(hip, orc, types, n_exp, n, ff, seed)
    x = orc.quantize_act(types[0], orc.gauss(seed + 1, 1.0, N * n).reshape(N, n))
    ctx = hip.moe_ctx(ex.args(np.zeros(1, np.int32), np.zeros((1, k), np.int32), np.zeros((1, k), np.float32)), N, k)
    ds, dw, dx = hip.upload(sel), hip.upload(w), hip.upload(x)
    dout = hip.upload(np.full((N, n + 3), -5.0, np.float32))
    ctx.run(N, ds, dw, dx, x.strides[0], dout, n + 3)
    out = hip.download(dout, np.zeros((N, n + 3), np.float32))
    ctx.close()
    ok = (sel >= 0) & (sel < n_exp)
    ref = orc.moe_ffn(types, ex.host, n, ff, x, np.where(ok, sel, 0), np.where(ok, w, 0.0).astype(np.float32), order=mode[1], path=mode[2])
    assert np.all(out[:, n:] == -5.0)
    assert np.array_equal(bits(out[:, :n]), bits(ref))


def routing(rng, N, n_exp, k):
    sel = np.stack([rng.permutation(n_exp)[:k] for _ in range(N)]).astype(np.int32)
    return sel, rng.random((N, k)).astype(np.float32)


@pytest.mark.parametrize("types", [(O.Q4_K, O.Q4_K, O.Q6_K), (O.Q2_K, O.Q2_K, O.Q2_K), (O.Q5_K, O.Q5_K, O.Q3_K),
                                   (O.Q6_K, O.Q6_K, O.Q5_K), (O.Q4_0, O.Q4_0, O.Q4_K)], ids=lambda t: "-".join(map(str, t)))
@pytest.mark.parametrize("N,k,ff", [(1, 8, 768), (3, 1, 256), (2, 16, 512), (18, 2, 1024), (29, 4, 256)])
def test_pairs(hipo, orc, types, N, k, ff):
    n = 352 if types[0] == O.Q4_0 else 512
    rng = np.random.default_rng(N * 100 + k)
    sel, w = routing(rng, N, 40, k)
    layer(hipo, orc, types, n, ff, 40, sel, w, 11 + N)


@pytest.mark.parametrize("mode", MODES, ids=["clang", "gcc", "scalar"])
def test_pairs_orders(hipo, orc, mode):
    hipo.set_order(mode[0])
    sel, w = routing(np.random.default_rng(5), 4, 24, 6)
    layer(hipo, orc, (O.Q4_K, O.Q4_K, O.Q6_K), 256, 512, 24, sel, w, 31, mode)


def test_pairs_repeats_and_no_expert(hipo, orc):
    sel, w = routing(np.random.default_rng(6), 5, 12, 4)
    sel[0] = 7                      # one expert four times
    sel[1, 2], sel[3, 0] = -1, 12   # no expert
    layer(hipo, orc, (O.Q4_K, O.Q4_K, O.Q4_K), 256, 256, 12, sel, w, 41)


def test_routing_under_the_outputs(hipo, orc):
    """the routing read from where the outputs go, and the routing outputs of run_logits over its own logits"""
    types, n, ff, n_exp, N, k = (O.Q4_K, O.Q4_K, O.Q6_K), 512, 256, 24, 8, 4
    ex = Experts(hipo, orc, types, n_exp, n, ff, 51)
    x = orc.quantize_act(types[0], orc.gauss(52, 1.0, N * n).reshape(N, n))
    logits = orc.gauss(53, 1.0, N * n_exp).reshape(N, n_exp)
    sel, w, _ = orc.route_softmax(logits, k, True)
    ref = orc.moe_ffn(types, ex.host, n, ff, x, sel, w, order=MODES[0][1], path=MODES[0][2])
    ctx = hipo.moe_ctx(ex.args(np.zeros(1, np.int32), np.zeros((1, k), np.int32), np.zeros((1, k), np.float32)), N, k)
    buf = np.zeros((N, n), np.float32)
    buf[0, :N * k] = np.ascontiguousarray(sel, np.int32).view(np.float32).ravel()
    buf[1, 1:1 + N * k] = w.ravel()
    dx, dout = hipo.upload(x), hipo.upload(buf)
    ctx.run(N, dout, int(dout) + 4 * (n + 1), dx, x.strides[0], dout, n)
    assert np.array_equal(bits(hipo.download(dout, np.zeros((N, n), np.float32))), bits(ref))
    dl, dout = hipo.upload(logits), hipo.upload(np.zeros((N, n), np.float32))
    ctx.run_logits(N, dl, 0, True, dx, x.strides[0], dout, n, int(dl) + 4 * N * k, dl)
    assert np.array_equal(bits(hipo.download(dout, np.zeros((N, n), np.float32))), bits(ref))
    assert np.array_equal(bits(hipo.download(dl, np.zeros((N, k), np.float32))), bits(w))
    assert np.array_equal(hipo.download(dl, np.zeros((N, k), np.int32), offset=4 * N * k), sel)
    ctx.close()
