"""GPU: transfers on both sides of the size up to which kernels read and write the
staging memory themselves (1 MB; hostio.hpp): states and histories there and back
with the staging memory used again at once, and the transform module's fields."""
import math

import numpy as np
import pytest

import mwf_amd as mw

pytestmark = pytest.mark.gpu


# planes 54 KB to 1.4 MB, fields 198 KB to 4.9 MB; ragged plane tiles and rows
@pytest.mark.parametrize("k0,mm,nn", [(4, 16, 16), (6, 32, 32), (4, 64, 64), (6, 64, 64), (6, 16, 128)])
@pytest.mark.parametrize("mixed", [False, True])
def test_small_transfers(k0, mm, nn, mixed):
    p = mw.make_params(k0, mm, nn, mm * math.pi / 4, nn * math.pi / 4, 200.0, 0.01,
                       precision=mw.MWF_MIXED if mixed else mw.MWF_FP64)
    v = mw.Velocity(p)
    rng = np.random.default_rng(mm + nn)
    a, b, o = (rng.standard_normal((2,) + v.mpt_shape) for _ in range(3))
    want = o.astype(np.float32).astype(np.float64) if mixed else o
    for c in (a, b):
        v.set_state(*c)
        v.set_onl(*o)
        assert np.array_equal(np.stack(v.get_state()), c)
        assert np.array_equal(np.stack(v.get_onl()[:2]), want)
    s = rng.standard_normal((2,) + v.spec_shape)
    s[:, 0] = 0  # n = 0 is not Hermitian
    f = v.tra_spec2phys(*s)
    r = np.stack(v.tra_phys2spec(f))
    assert np.array_equal(v.tra_spec2phys(*s), f)
    # two transforms of at most 3072 points, unit values: a few roundings per pass
    assert np.abs(r - s).max() <= (1e-5 if mixed else 1e-13)
    assert np.array_equal(np.stack(v.get_state()), b)
    v.close()
