"""GPU: errors that the mixed form makes alike in every step (rounded twiddles and
multipliers) add up along a run: the state after 50 steps against FP64, a mean over
five initial conditions, is no further off in the default flux form than in the
advective one."""
import math

import numpy as np
import pytest

import mwf_amd as mw

pytestmark = pytest.mark.gpu


def _state(k0, mm, nn, seed, precision, mode):
    p = mw.make_params(k0, mm, nn, mm * math.pi / 4, nn * math.pi / 4, 250.0, 0.01, precision=precision)
    mw.autotune(mode)
    try:
        v = mw.Velocity(p)
    finally:
        mw.autotune(0)
    v.set_state(*mw.ic_gaussian(p, seed, 0.3, 8.0))
    v.vel_TS(50)
    s = np.stack(v.get_state())
    v.close()
    return s


# rows of 64 points (one batch), of 512 (two buffers) and of 1024; x transforms on two waves
@pytest.mark.parametrize("k0,mm,nn", [(6, 64, 64), (4, 64, 512), (6, 64, 1024), (6, 1024, 64)])
def test_state_error_of_the_mixed_form(k0, mm, nn):
    err = {0: [], 2: []}  # modes: the default rules, the advective plan 0
    for seed in range(1, 6):
        want = _state(k0, mm, nn, seed, mw.MWF_FP64, 0)
        for mode in err:
            got = _state(k0, mm, nn, seed, mw.MWF_MIXED, mode)
            err[mode].append(np.linalg.norm(got - want) / np.linalg.norm(want))
    flux, adv = (float(np.mean(err[m])) for m in (0, 2))
    print(f"k0={k0} mm={mm} nn={nn}: 50 steps, flux {flux:.2e} advective {adv:.2e}", flush=True)
    assert flux <= adv
