"""The wave-specialised persistent kernel's 64-activation tiles, and its Q5_K form, against the oracle and against the
per-tile launches bit for bit: activations around one and several tiles, rows around the 64-row tiles, 2 to 32 superblocks,
products of different shapes in one launch, a row range with a padded output stride, extreme blocks."""
import numpy as np
import pytest

import es_hip_quant as E
import oracle as O

pytestmark = pytest.mark.gpu
MODES = [(E.ORDER_X86_CONTRACT, O.CONTRACT, O.PATH_X86), (E.ORDER_X86_STRICT, O.STRICT, O.PATH_X86)]


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def inputs(orc, t, rows, cols, na, seed):
    st = np.array([seed], np.uint64)
    return orc.mtest_blocks(t, st, rows, cols), orc.quantize_act(t, orc.mtest_acts(st, na * cols).reshape(na, cols))


@pytest.mark.parametrize("t", [O.Q4_K, O.Q5_K])
@pytest.mark.parametrize("rows,nbk,na", [(1, 2, 64), (65, 4, 33), (64, 32, 63), (130, 8, 65), (200, 2, 129), (300, 6, 200)])
def test_vs_oracle(hip, orc, t, rows, nbk, na):
    W, acts = inputs(orc, t, rows, 256 * nbk, na, rows + na)
    r0, ys = (2 if rows > 100 else 0), rows + 67
    dW, dA = hip.upload(W), hip.upload(acts)
    try:
        for mode in MODES:
            hip.set_order(mode[0])
            dY = hip.upload(np.full((na, ys), -3.0, np.float32))
            hip.matvec_multi_dev(t, dW, 256 * nbk, r0, rows, dA, acts.strides[0], na, dY, ys)
            y = hip.download(dY, np.zeros((na, ys), np.float32))
            ref = orc.matvec_multi(t, W, 256 * nbk, rows, acts, mode[1], mode[2])
            assert np.array_equal(bits(y[:, r0:rows]), bits(ref[:, r0:])), mode
            assert np.all(y[:, rows:] == -3.0) and np.all(y[:, :r0] == -3.0)
    finally:
        hip.set_order(E.ORDER_X86_CONTRACT)


@pytest.mark.parametrize("t", [O.Q4_K, O.Q5_K])
def test_forms_agree(hip, orc, t):
    """several products in one launch (one tile, some tiles and more than one tile of 128 per CU) in every form"""
    shapes = [(2048, 4, 70), (64, 8, 64), (9000, 2, 300)]
    ins = [inputs(orc, t, r, 256 * b, na, 9 + r) for r, b, na in shapes]
    for use in ([0], [0, 1], [0, 1, 2]):
        out = {}
        for on in (0, 1, 2, 3):
            prev = hip.set_direct_persistent(on)
            try:
                keep, specs = [], []
                for i in use:
                    (rows, nbk, na), (W, a) = shapes[i], ins[i]
                    dW, dA, dY = hip.upload(W), hip.upload(a), hip.alloc(na * rows * 4)
                    keep += [dW, dA, dY]
                    specs.append(dict(type=t, rows=rows, cols=256 * nbk, W=dW, act=dA, astride=a.strides[0], nb=na, y=dY, ystride=rows))
                hip.run_jobs(specs)
                out[on] = [hip.download(s["y"], np.zeros((s["nb"], s["rows"]), np.float32)) for s in specs]
            finally:
                hip.set_direct_persistent(prev)
        for on in (1, 2, 3):
            for a, b in zip(out[0], out[on]):
                assert np.array_equal(bits(a), bits(b)), (use, on)


@pytest.mark.parametrize("fill", [0x00, 0xFF])
def test_q5k_extremes(hip, orc, fill):
    rows, nbk, na = 70, 2, 40
    W = np.full((rows, nbk, 176), fill, np.uint8)
    W[..., 0:2] = np.array([0.01], np.float16).view(np.uint8)
    W[..., 2:4] = np.array([0.02], np.float16).view(np.uint8)
    x = np.ones((na, 256 * nbk), np.float32)
    x[1::2] = -1.0
    acts = orc.quantize_act(O.Q5_K, x)
    y = hip.matvec_multi(O.Q5_K, W.reshape(-1), 256 * nbk, rows, acts)
    assert np.array_equal(bits(y), bits(orc.matvec_multi(O.Q5_K, W.reshape(-1), 256 * nbk, rows, acts)))
