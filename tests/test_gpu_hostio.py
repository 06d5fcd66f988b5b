"""GPU: the host boundary's transposes and staged copies (hostio.hpp) move every
value unchanged: states and histories there and back, at sizes below, at and
above one staging chunk and with slot counts and row lengths that leave ragged
tiles, from several threads at once."""
import math
import threading

import numpy as np
import pytest

import mwf_amd as mw

pytestmark = pytest.mark.gpu


def _round_trip(k0, mm, nn, mixed, seed):
    p = mw.make_params(k0, mm, nn, mm * math.pi / 4, nn * math.pi / 4, 200.0, 0.01,
                       precision=mw.MWF_MIXED if mixed else mw.MWF_FP64)
    v = mw.Velocity(p)
    rng = np.random.default_rng(seed)
    c, o = (rng.standard_normal((2,) + v.mpt_shape) for _ in range(2))
    v.set_state(*c)
    assert np.array_equal(np.stack(v.get_state()), c)
    v.set_onl(*o)
    got = np.stack(v.get_onl()[:2])
    assert np.array_equal(got, o.astype(np.float32).astype(np.float64) if mixed else o)
    assert np.array_equal(np.stack(v.get_state()), c)
    v.close()


# (4, 16, 16): a state of 55 KB; (4, 256, 256): two chunks of 8 MB; (6, 256, 512): more than the four
# chunks of a handle's staging
@pytest.mark.parametrize("k0,mm,nn", [(4, 16, 16), (6, 16, 128), (6, 64, 64), (4, 256, 256), (6, 512, 32), (6, 256, 512)])
@pytest.mark.parametrize("mixed", [False, True])
def test_state_and_history_round_trip(k0, mm, nn, mixed):
    _round_trip(k0, mm, nn, mixed, mm + nn)


def test_concurrent_handles():
    """Handles on several threads share the copy threads."""
    bad = []

    def work(i):
        try:
            for j in range(3):
                _round_trip(4, 128, 128 >> (i % 2), False, 10 * i + j)
        except Exception as e:  # noqa: BLE001
            bad.append((i, repr(e)))

    th = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
