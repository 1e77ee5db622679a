"""The Q6_K kernel with one wave per superblock (es_hip_m6w.hip) against the oracle, bit for bit, at its edges: superblock
counts around the 8 waves (one round, several, uneven), activations around its 16-wide tiles and from the smallest batch it
takes, rows around its 16-row groups with a row range and a padded odd output stride, several products in one launch, and
blocks at the extremes of codes, scales and activation values (the two int8 planes hold -8064..8001)."""
import numpy as np
import pytest

import es_hip_quant as E
import oracle as O

pytestmark = pytest.mark.gpu
MODES = [(E.ORDER_X86_CONTRACT, O.CONTRACT, O.PATH_X86), (E.ORDER_X86_STRICT, O.STRICT, O.PATH_X86)]


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def run(hip, W, cols, rows, acts, r0, r1, ys):
    na = acts.shape[0]
    dW, dA = hip.upload(W), hip.upload(acts)
    dY = hip.upload(np.full((na, ys), -7.0, np.float32))
    hip.matvec_multi_dev(O.Q6_K, dW, cols, r0, r1, dA, acts.strides[0], na, dY, ys)
    return hip.download(dY, np.zeros((na, ys), np.float32))


@pytest.mark.parametrize("nbk", [1, 3, 7, 8, 9, 17, 32])
@pytest.mark.parametrize("na,rows", [(5, 1), (15, 17), (16, 250), (33, 16), (65, 33), (130, 47)])
def test_edges(hip, orc, nbk, na, rows):
    cols = 256 * nbk
    st = np.array([nbk * 1000 + na], np.uint64)
    W = orc.mtest_blocks(O.Q6_K, st, rows, cols)
    acts = orc.quantize_act(O.Q6_K, orc.mtest_acts(st, na * cols).reshape(na, cols))
    r0, ys = (3 if rows > 20 else 0), rows + 5
    try:
        for mode in MODES:
            hip.set_order(mode[0])
            y = run(hip, W, cols, rows, acts, r0, rows, ys)
            ref = orc.matvec_multi(O.Q6_K, W, cols, rows, acts, mode[1], mode[2])
            assert np.array_equal(bits(y[:, r0:rows]), bits(ref[:, r0:])), mode
            assert np.all(y[:, rows:] == -7.0) and np.all(y[:, :r0] == -7.0)
    finally:
        hip.set_order(E.ORDER_X86_CONTRACT)


@pytest.mark.parametrize("code", [0x00, 0xFF, 0xA5])
@pytest.mark.parametrize("scale", [-128, 127, -1])
def test_extremes(hip, orc, code, scale):
    rows, nbk, na = 20, 2, 18
    W = np.full((rows, nbk, 210), code, np.uint8)
    W[..., 192:208] = np.uint8(scale & 0xFF)
    W[..., 208:210] = np.array([0.5], np.float16).view(np.uint8)
    x = np.ones((na, 256 * nbk), np.float32)
    x[1::3] = -1.0
    x[2::3, ::2] = -1.0
    acts = orc.quantize_act(O.Q6_K, x)   # every value +-127
    y = run(hip, W.reshape(-1), 256 * nbk, rows, acts, 0, rows, rows)
    assert np.array_equal(bits(y), bits(orc.matvec_multi(O.Q6_K, W.reshape(-1), 256 * nbk, rows, acts)))


def test_several_products_in_a_launch(hip, orc):
    specs, want, outs, keep = [], [], [], []
    for j, (rows, nbk, na) in enumerate([(40, 4, 20), (16, 4, 31), (100, 4, 18), (33, 12, 40)]):
        st = np.array([500 + j], np.uint64)
        W = orc.mtest_blocks(O.Q6_K, st, rows, 256 * nbk)
        acts = orc.quantize_act(O.Q6_K, orc.mtest_acts(st, na * 256 * nbk).reshape(na, 256 * nbk))
        want.append(orc.matvec_multi(O.Q6_K, W, 256 * nbk, rows, acts))
        dW, dA, dY = hip.upload(W), hip.upload(acts), hip.alloc(na * rows * 4)
        keep += [dW, dA]
        outs.append(dY)
        specs.append(dict(type=O.Q6_K, rows=rows, cols=256 * nbk, W=dW, act=dA, astride=acts.strides[0], nb=na, y=dY, ystride=rows))
    hip.run_jobs(specs)
    for dY, w in zip(outs, want):
        assert np.array_equal(bits(hip.download(dY, np.zeros_like(w))), bits(w))


@pytest.mark.parametrize("shapes", [
    [(2048, 1, 5 + j % 11) for j in range(40)],                       # several row groups per workgroup, chunks rounded to 8
    [(1000 + 16 * j, 3, 20 + j) for j in range(20)],                  # ... at two tiles of activations
    [(160, 4, 8), (96, 4, 15), (16, 4, 1), (7, 9, 3)],                # a decode launch beside it
    [(16, 4, 5), (300, 4, 2), (250, 2, 4)],                           # few products of 5: all in the decode launch
    [(64, 9, 6), (64, 9, 1)], [(64, 9, 9), (64, 9, 1)],               # rows longer than its waves
    [(40, 2, 9), (40, 2, 33), (40, 2, 2)],                            # every kind
    [(1024, 3, 33 + 5 * j) for j in range(8)],                        # four tiles of activations, three waves
    [(300, 4, 8), (33, 4, 8), (2500, 4, 7), (16, 4, 5)],              # jobs of unequal length as kernel arguments
    [(300, 4, 8), (33, 4, 8), (2500, 4, 7), (16, 4, 5), (50, 4, 8)],  # ... and one more than fit
    [(2100, 8, 6), (512, 8, 6), (500, 8, 6)],                         # a long job over several rows of the grid
    [(2700, 4, 70), (64, 4, 70), (40, 4, 64), (1300, 4, 33)],         # ... with several tiles of activations
], ids=["chunks", "tiles", "beside", "left", "long6", "long9", "mixed", "threes", "four", "five", "rows", "rowtiles"])
def test_batches(hip, orc, shapes):
    specs, want, outs, keep = [], [], [], []
    for j, (rows, nbk, na) in enumerate(shapes):
        st = np.array([900 + j], np.uint64)
        W = orc.mtest_blocks(O.Q6_K, st, rows, 256 * nbk)
        acts = orc.quantize_act(O.Q6_K, orc.mtest_acts(st, na * 256 * nbk).reshape(na, 256 * nbk))
        want.append(orc.matvec_multi(O.Q6_K, W, 256 * nbk, rows, acts))
        dW, dA, dY = hip.upload(W), hip.upload(acts), hip.upload(np.full((na, rows), -7.0, np.float32))
        keep += [dW, dA]
        outs.append(dY)
        specs.append(dict(type=O.Q6_K, rows=rows, cols=256 * nbk, W=dW, act=dA, astride=acts.strides[0], nb=na, y=dY, ystride=rows))
    plan = hip.plan(specs)
    plan.run()
    hip.synchronize()
    plan.close()
    for dY, w in zip(outs, want):
        assert np.array_equal(bits(hip.download(dY, np.zeros_like(w))), bits(w))


@pytest.mark.parametrize("nbk", [1, 2, 3, 4, 8, 9, 17])
@pytest.mark.parametrize("rows", [4096, 8203])
def test_several_tiles_of_activations(hip, orc, nbk, rows):
    """at least 256 row groups, so that a workgroup takes 2 or 4 tiles of 16 activations: rows of fewer superblocks (so fewer
    waves) than tiles, full and ragged tiles, several rounds per row; every output against the vector kernel, the first and last
    activations of the tiles against the oracle"""
    cols = 256 * nbk
    st = np.array([nbk * 100 + rows], np.uint64)
    W = orc.mtest_blocks(O.Q6_K, st, rows, cols)
    every = orc.quantize_act(O.Q6_K, orc.mtest_acts(st, 128 * cols).reshape(128, cols))
    r0, ys = (5 if rows > 4096 else 0), rows + 3
    for na in (17, 31, 32, 33, 48, 49, 64, 65, 128):
        acts = np.ascontiguousarray(every[:na])
        y = run(hip, W, cols, rows, acts, r0, rows, ys)
        prev = hip.set_q6k_mfma_min_batch(0)
        try:
            ref = run(hip, W, cols, rows, acts, r0, rows, ys)
        finally:
            hip.set_q6k_mfma_min_batch(prev)
        assert np.array_equal(bits(y), bits(ref)), na
    pick = [0, 15, 16, 31, 32, 47, 48, 63, 64, 127]
    assert np.array_equal(bits(y[pick, r0:rows]), bits(orc.matvec_multi(O.Q6_K, W, cols, rows, np.ascontiguousarray(every[pick]))[:, r0:]))
