"""GPU: the nonlinear term of the flux form where the spectrum fills wavenumbers
far above the wall-normal ones (alpha MM = gamma NN = 4096, flat velocity
spectrum), from the split and from the fused x kernels, against the oracle.  The
error is that of the velocity tendency, relative to its norm."""
import math

import numpy as np
import pytest

import mwf_amd as mw
import oracle

pytestmark = pytest.mark.gpu

BETA = math.pi / 2


def _wave(k0, mm, nn, kmax):
    """Squared wall-parallel wavenumbers and, per mpt slot, |velocity|^2 per |slot|^2."""
    m = np.concatenate([np.arange(mm), np.arange(-(mm - 1), 0)]) * (kmax / mm)
    k2 = (np.arange(nn) * (kmax / nn))[:, None] ** 2 + (m ** 2)[None, :]
    k2[0, 0] = 1.0
    ak2 = (np.arange(1, k0) * BETA) ** 2
    return np.concatenate([np.repeat(k2[:, :, None], k0, 2), k2[:, :, None] * (k2[:, :, None] + ak2)], 2)


# the one-batch z kernel and the all-lines x kernel; rows of 256 points in k_zc (M6 FP64) and in the
# one-batch kernel; two-buffer rows of 512; rows of 1024, in FP64 three blocks each; x transforms on two waves
@pytest.mark.parametrize("k0,mm,nn", [(4, 32, 32), (6, 16, 256), (4, 64, 512), (6, 16, 1024), (4, 1024, 16)])
@pytest.mark.parametrize("mixed", [False, True])
def test_nonlinear_term_of_a_fine_box(k0, mm, nn, mixed):
    kmax = 4096.0
    p = mw.make_params(k0, mm, nn, 2 * math.pi * mm / kmax, 2 * math.pi * nn / kmax, 200.0, 1e-9, thdeg=10.0,
                       precision=mw.MWF_MIXED if mixed else mw.MWF_FP64)
    v = mw.Velocity(p)
    assert v.plan_info() & mw.PLAN_FLUX
    o = oracle.Oracle(k0, mm, nn, p.alpha, p.gamma, p.re, p.dt, theta=p.theta)
    w = _wave(k0, mm, nn, kmax)
    rng = np.random.default_rng(3)
    c = (rng.standard_normal(v.mpt_shape) + 1j * rng.standard_normal(v.mpt_shape)) / np.sqrt(w)
    c[0, mm:] = c[0, 1:mm][::-1].conj()
    c[0, 0] = 0
    re, im = np.ascontiguousarray(c.real), np.ascontiguousarray(c.imag)
    o.set_state(re, im)
    s = 0.3 / math.sqrt(o.energy())
    re, im = re * s, im * s
    o.set_state(re, im)
    nl = o.nonlinear()
    want = nl[0] + 1j * nl[1]
    norm = math.sqrt((abs(want) ** 2 / w).sum())
    # some ten roundings of relative size u in the transforms, products and lines (5 u of their
    # root mean square); the oracle's own as well in FP64
    u = 2.0 ** -24 if mixed else 2.0 ** -53
    bar = (10 if mixed else 20) * u
    v.set_state(re, im)
    a = v.vel_nonlinear()
    split = math.sqrt((abs(a[0] + 1j * a[1] - want) ** 2 / w).sum()) / norm
    v.set_state(re, im)
    v.vel_TS(1)
    b = v.get_onl()
    fused = math.sqrt((abs(b[0] + 1j * b[1] - want) ** 2 / w).sum()) / norm
    print(f"k0={k0} mm={mm} nn={nn} mixed={mixed}: split {split:.2e} fused {fused:.2e} bar {bar:.1e}", flush=True)
    v.close()
    assert split <= bar and fused <= bar
