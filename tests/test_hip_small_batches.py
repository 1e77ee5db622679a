"""Decode batches whose jobs travel as kernel arguments (up to four per launch, one grid row each) against the oracle: one to
five products, so the last needs a job table; rows from one to several workgroups, so grid rows differ in length and the
shorter jobs' last workgroups have nothing to do; one format or two (two launches); one activation, several, and a mix (which
takes the table). Run from run_jobs and from a kept plan."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("n", [1, 2, 4, 5])
@pytest.mark.parametrize("types,nas", [((O.Q4_K,), (1,)), ((O.Q4_K,), (3,)), ((O.Q4_K,), (1, 2)), ((O.Q6_K, O.Q4_K), (1,)),
                                       ((O.Q6_K, O.Q4_K), (1, 2, 2)), ((O.Q4_0,), (1,)), ((O.Q8_0, O.Q5_0), (1,))])
def test_jobs_as_arguments(hip, orc, n, types, nas):
    rows = [1, 70, 513, 33, 128]
    specs, want, bufs, outs = [], [], [], []
    for j in range(n):
        t, na, cols = types[j % len(types)], nas[j % len(nas)], 512 if j != 2 else 1280
        W = orc.quantize_rows(t, orc.gauss(100 + j, 0.05, rows[j] * cols).reshape(rows[j], cols))
        a = orc.quantize_act(t, orc.gauss(7 + j, 1.0, na * cols).reshape(na, cols))
        want.append(orc.matvec_multi(t, W, cols, rows[j], a))
        dW, dA, dY = hip.upload(W), hip.upload(a), hip.alloc(na * rows[j] * 4)
        bufs += [dW, dA]
        outs.append(dY)
        specs.append(dict(type=t, rows=rows[j], cols=cols, W=dW, act=dA, astride=a.strides[0], nb=na, y=dY, ystride=rows[j]))

    def check(what):
        for j in range(n):
            got = hip.download(outs[j], np.zeros_like(want[j]))
            assert np.array_equal(bits(got), bits(want[j])), (what, j)
            hip.memset(outs[j], 0xFF, got.nbytes)

    for y, w in zip(outs, want):
        hip.memset(y, 0xFF, w.nbytes)
    hip.run_jobs(specs)
    check("run_jobs")
    plan = hip.plan(specs)
    for _ in range(2):
        plan.run()
        hip.synchronize()
        check("plan")
    plan.close()
