"""GPU: the kernels of small launches -- the z kernel that takes an x-row in one
batch (zbatch.hpp, rows of up to 256 points) and the fused x kernel that
transforms all lines of a narrow tile at once (xall.hpp) -- at the edges of
their ranges: against the oracle, and against the kernels that a larger launch
of the same size runs."""
import math

import numpy as np
import pytest

import mwf_amd as mw
import oracle

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    num = sum(np.sum((x - y) ** 2) for x, y in zip(a, b))
    return math.sqrt(num / sum(np.sum(y ** 2) for y in b))


def _params(k0, mm, nn, mixed=False, theta=0.0):
    return mw.make_params(k0, mm, nn, mm * math.pi / 4, nn * math.pi / 4, 200.0, 0.01, thdeg=theta,
                          precision=mw.MWF_MIXED if mixed else mw.MWF_FP64)


# smallest and longest rows, both bases; x tiles of 64 to 512 values, of one
# column (MM = 512), of fewer columns than NN allows, and k_xstep's
@pytest.mark.parametrize("k0,mm,nn", [(4, 16, 16), (6, 16, 16), (4, 16, 256), (6, 32, 128), (4, 128, 256), (6, 256, 16),
                                      (4, 512, 16), (4, 512, 64), (6, 128, 128), (4, 512, 128), (6, 256, 128)])
@pytest.mark.parametrize("mixed", [False, True])
def test_small_sizes_match_oracle(k0, mm, nn, mixed):
    p = _params(k0, mm, nn, mixed, theta=20.0)
    v = mw.Velocity(p)
    assert v.plan_info() & mw.PLAN_FLUX
    o = oracle.Oracle(k0, mm, nn, p.alpha, p.gamma, p.re, p.dt, theta=p.theta)
    re, im = mw.ic_gaussian(p, 8, 0.2, 4.0)
    v.set_state(re, im)
    o.set_state(re, im)
    v.vel_TS(10)
    o.step(10)
    err = rel_l2(v.get_state(), o.get_state())
    print(f"k0={k0} mm={mm} nn={nn} mixed={mixed}: 10 steps rel_l2 {err:.2e}")
    assert err <= (1e-5 if mixed else 1e-12)
    v.close()


@pytest.mark.parametrize("k0,mm,nn,mixed", [(4, 64, 64, False), (4, 64, 64, True), (4, 32, 32, False), (6, 128, 128, False),
                                            (4, 128, 32, True), (6, 16, 64, False), (4, 256, 32, False),
                                            (4, 512, 16, True), (6, 256, 128, False), (4, 64, 1024, True)])
def test_members_step_alike_in_small_and_large_launches(k0, mm, nn, mixed):
    """A single model's launches take the all-lines x kernel or half tiles, those
    of enough members of the same size k_xstep's whole tiles: the same bits."""
    p = _params(k0, mm, nn, mixed)
    n = 128 // ((nn // min(nn, 2048 // mm)) * k0) + 1  # more than 128 whole tiles
    ic = mw.ic_gaussian(p, 4, 0.2, 4.0)
    ens, v = mw.Ensemble([p] * n), mw.Velocity(p)
    for i in range(n):
        ens.set_state(i, *ic)
    v.set_state(*ic)
    ens.step(5)
    v.vel_TS(5)
    a, b = ens.get_state(n - 1), v.get_state()
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    ens.close()
    v.close()
