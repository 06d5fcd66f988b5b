"""GPU: the FP64 flux z kernel of 1024-point rows, three blocks to a row
(k_zc3): all x kernels that read its lines (the vw share of E on a line of its
own) against the oracle, with tilted walls and an x-row count that leaves each
XCD an odd run of rows."""
import math

import numpy as np
import pytest

import mwf_amd as mw
import oracle

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    num = sum(np.sum((x - y) ** 2) for x, y in zip(a, b))
    return math.sqrt(num / sum(np.sum(y ** 2) for y in b))


# MM = 16 (8 K0 k_xstep blocks: k_xall), 128 (k_xstep); plan 10 = split x kernels
@pytest.mark.parametrize("k0,mm", [(4, 16), (6, 16), (4, 128), (6, 128)])
@pytest.mark.parametrize("choice", [mw.PLAN_FLUX, mw.PLAN_FLUX | mw.PLAN_SPLIT_X])
def test_three_block_rows_match_oracle(k0, mm, choice):
    nn = 1024
    p = mw.make_params(k0, mm, nn, mm * math.pi / 4, nn * math.pi / 4, 200.0, 0.02, thdeg=-25.0)
    mw.autotune(2 + choice)
    try:
        v = mw.Velocity(p)
    finally:
        mw.autotune(0)
    assert v.plan_info() == choice
    o = oracle.Oracle(k0, mm, nn, p.alpha, p.gamma, p.re, p.dt, theta=p.theta)
    re, im = mw.ic_gaussian(p, 7, 0.2, 4.0)
    v.set_state(re, im)
    o.set_state(re, im)
    a, b = v.vel_nonlinear(), o.nonlinear()
    nerr = max(np.abs(a[i] - b[i]).max() for i in range(2)) / max(np.abs(b[0]).max(), np.abs(b[1]).max())
    v.set_state(re, im)
    v.vel_TS(5)
    o.step(5)
    err = rel_l2(v.get_state(), o.get_state())
    print(f"k0={k0} mm={mm} plan {choice}: nonlinear {nerr:.2e}, 5 steps {err:.2e}")
    assert nerr <= 1e-12 and err <= 1e-12
    v.close()
