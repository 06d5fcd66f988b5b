"""GPU: the plans of the advective form (forced; the default is the flux form, and
the tuner takes its candidates on trust) against the oracle: each z kernel in both
precisions, and the fused and split x kernels at row counts from the smallest to
the two-wave transforms of MM = 1024."""
import math

import numpy as np
import pytest

import cases
import mwf_amd as mw
import oracle

pytestmark = pytest.mark.gpu

ZB, SPLIT = mw.PLAN_ZB, mw.PLAN_SPLIT_X


def rel_l2(a, b):
    return math.sqrt(sum(((x - y) ** 2).sum() for x, y in zip(a, b)) / sum((y ** 2).sum() for y in b))


def _model(p, choice):
    mw.autotune(2 + choice)
    try:
        v = mw.Velocity(p)
    finally:
        mw.autotune(0)
    assert v.plan_info() == choice
    return v


def _check(k0, mm, nn, choice, mixed):
    p = mw.make_params(k0, mm, nn, mm * math.pi / 4, nn * math.pi / 4, 200.0, 0.02, thdeg=20.0,
                       precision=mw.MWF_MIXED if mixed else mw.MWF_FP64)
    v = _model(p, choice)
    o = oracle.Oracle(k0, mm, nn, p.alpha, p.gamma, p.re, p.dt, theta=p.theta)
    re, im = mw.ic_gaussian(p, 5, 0.2, 4.0)
    v.set_state(re, im)
    o.set_state(re, im)
    nl = rel_l2(v.vel_nonlinear(), o.nonlinear())
    v.set_state(re, im)
    v.vel_TS(10)
    o.step(10)
    err = rel_l2(v.get_state(), o.get_state())
    print(f"plan {choice} k0={k0} mm={mm} nn={nn} mixed={mixed}: nonlinear {nl:.2e}, 10 steps {err:.2e}", flush=True)
    v.close()
    bar = 1e-5 if mixed else 1e-12
    assert nl <= bar and err <= bar


# k_z over its row lengths, k_zb at 256 and 512, and at 1024 where it is the only one
@pytest.mark.parametrize("k0,nn,choice", [(4, 16, 0), (6, 64, 0), (4, 256, 0), (6, 512, 0), (6, 32, SPLIT), (4, 256, ZB),
                                          (6, 512, ZB), (6, 256, ZB | SPLIT), (4, 1024, 0), (6, 1024, 0), (4, 1024, SPLIT)])
@pytest.mark.parametrize("mixed", [False, True])
def test_z_kernels_match_oracle(k0, nn, choice, mixed):
    _check(k0, 32, nn, choice, mixed)


# x-tiles of many, some and two columns; NN below a whole tile's columns at MM = 64
@pytest.mark.parametrize("k0,mm,nn", [(4, 16, 64), (6, 64, 16), (4, 128, 32), (6, 512, 16), (4, 1024, 16), (6, 1024, 32)])
@pytest.mark.parametrize("choice", [0, SPLIT])
@pytest.mark.parametrize("mixed", [False, True])
def test_x_kernels_match_oracle(k0, mm, nn, choice, mixed):
    _check(k0, mm, nn, choice, mixed)


@pytest.mark.parametrize("choice", [0, SPLIT, mw.PLAN_ZB_SPLIT, mw.PLAN_ZB_SPLIT | SPLIT])
def test_m6_2048_advective_plans_match_the_default(choice):
    """M6 2048^2, FP64: the advective plans against the default plan, which is held
    to the oracle at this size elsewhere: nonlinear term and 3 steps."""
    p = cases.params("m6_2048")
    seed, scl, k0ic = cases.ic_of("m6_2048")
    re, im = mw.ic_gaussian(p, seed, scl, k0ic)
    out = []
    for v in (mw.Velocity(p), _model(p, choice)):
        v.set_state(re, im)
        nl = v.vel_nonlinear()
        v.set_state(re, im)
        v.vel_TS(3)
        out.append((nl, v.get_state()))
        v.close()
    nl, err = rel_l2(out[1][0], out[0][0]), rel_l2(out[1][1], out[0][1])
    print(f"plan {choice} M6 2048^2: nonlinear {nl:.2e}, 3 steps {err:.2e}", flush=True)
    assert nl <= 1e-12 and err <= 1e-12
