"""CPU: the lines of the flux form and their weights (fluxline.hpp, compiled for
the host).  With a line pair chosen per n no weighted part of a rounded line
cancels, whatever the box: psi and phi from lines in single precision stay within
the rounding of the terms they have in the form without lines."""
import ctypes
import math
import os
import subprocess

import numpy as np
import pytest

import oracle
from test_oracle_nonlinear import BETA, CASES, _from_xz, _gen, _state, _to_xz, _wavenumbers

UW, F, UV, E = range(4)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mwf_amd", "csrc")
    d = tmp_path_factory.mktemp("fluxline")
    src, so = d / "line.cpp", d / "line.so"
    src.write_text("#define __host__\n#define __device__\n"
                   f'#include "{csrc}/fluxline.hpp"\n'
                   'template <typename M> static void put(M m, double* o) { o[0] = m.ak; o[1] = m.e; o[2] = m.f; o[3] = m.h; o[4] = m.far; }\n'
                   'extern "C" void mul(double g, double ak, int single, double* o) {\n'
                   "  if (single) put(dev_mul<float>(g, 1 / g, ak), o);\n"
                   "  else put(dev_mul<double>(g, 1 / g, ak), o);\n}\n"
                   'extern "C" void weights(int li, double a, double g, double ak, double* o) {\n'
                   "  dev_weights(li, a, g, ak, ak == 0 ? -1.0 : 1 / ak, o[0], o[1]);\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-Wno-unknown-pragmas", "-o", str(so), str(src)], check=True)
    L = ctypes.CDLL(str(so))
    dp, cd, ci = ctypes.POINTER(ctypes.c_double), ctypes.c_double, ctypes.c_int
    L.mul.argtypes, L.weights.argtypes = [cd, cd, ci, dp], [ci, cd, cd, cd, dp]
    return L


def _call(fn, n, *args):
    out = np.empty(n)
    fn(*args, out.ctypes.data_as(ctypes.POINTER(ctypes.c_double)))
    return out


def _psi_phi(lib, lines, a, g, ak):
    """psi, phi of an index k >= 1 from its four lines at one (m, n)."""
    psi = phi = 0j
    for li in (UW, F, UV, E):
        cp, cq = _call(lib.weights, 2, li, a, g, ak)
        x = complex(lines[li]) * (1j if li == UV else 1)
        psi, phi = psi + cp * x, phi + cq * x
    return psi, phi


def test_single_precision_lines_keep_the_precision_of_the_terms(lib):
    """Rows of unit size.  Each line is a sum of up to three shares (row times
    multiplier), a share with at most three roundings and a sum with two: 5 u of the
    sum of its shares.  By |g| <= |ak| or |g| > |ak| the weighted shares are at most
    four times a term that psi and phi have without lines, so 20 u of these in all."""
    u = 2.0 ** -24
    rng = np.random.default_rng(5)
    for _ in range(4000):
        a, g = 10.0 ** rng.uniform(-2, 4, 2) * rng.choice([-1, 1], 2)
        k = int(rng.integers(1, 6))
        ak = (-1) ** k * k * BETA
        if rng.random() < 0.1:
            g = ak * rng.choice([-1, 1]) * (1 + rng.choice([0.0, 1e-9, -1e-9]))
        uv, uw, vvuu, vw, vvww = (rng.uniform(-1, 1, 5) + 1j * rng.uniform(-1, 1, 5)).astype(np.complex64)
        akr, e, f, h, far = _call(lib.mul, 5, g, ak, 1)
        assert bool(far) == (abs(g) > abs(ak))
        akr, e, f, h = (np.float32(x) for x in (akr, e, f, h))
        assert np.isfinite([akr, e, f, h]).all()
        x = vvuu - vvww if far else vvuu
        lines = {UW: uw, UV: uv, E: np.complex64(complex(np.float32(akr * x.real + e * vw.imag), np.float32(akr * x.imag - e * vw.real))),
                 F: np.complex64(complex(np.float32(f * vvww.real - h * vw.imag), np.float32(f * vvww.imag + h * vw.real)))}
        psi, phi = _psi_phi(lib, lines, a, g, ak)
        uv, uw, vvuu, vw, vvww = (complex(x) for x in (uv, uw, vvuu, vw, vvww))
        wpsi = (a * a - g * g) * uw + 1j * g * ak * uv + a * g * (vvuu - vvww) - 1j * a * ak * vw
        wphi = (1j * a * (ak * ak - a * a - g * g) * uv - 2 * ak * a * g * uw + a * a * (ak * vvuu - 1j * g * vw)
                + g * (ak * g * vvww + 1j * (ak * ak - g * g) * vw))
        A, G, K = abs(a), abs(g), abs(ak)
        spsi = A * A + G * G + G * K + A * G + A * K
        sphi = A ** 3 + A * G * G + A * K * K + 2 * A * G * K + A * A * K + A * A * G + K * G * G + G * K * K + G ** 3
        for got, want, s in ((psi, wpsi, spsi), (phi, wphi, sphi)):
            assert max(abs((got - want).real), abs((got - want).imag)) <= 20 * u * s, (a, g, k)


@pytest.mark.parametrize("k0,mm,nn,theta,alpha,gamma", CASES)
def test_lines_and_weights_give_the_nonlinear_term(lib, k0, mm, nn, theta, alpha, gamma):
    """In double precision, against the oracle's advective term at every mode."""
    o = oracle.Oracle(k0, mm, nn, alpha, gamma, 200.0, 0.02, theta=theta)
    re, im = _state(o, 29 * k0 + mm + nn)
    o.set_state(re, im)
    want = o.nonlinear()
    sr, si = o.mpt2spec(re, im)
    s = sr + 1j * si
    s[0, 0, 1] += math.cos(theta)
    s[0, 0, 2 * k0] += math.sin(theta)
    p = _to_xz(o, s)
    T = {}
    for name, i, terms in _gen().flux_rows(k0):
        T[name, i] = sum(float(c) * p[:, :, a] * p[:, :, b] for a, b, c in terms)
    kx, kz = _wavenumbers(o)
    got = np.zeros(s.shape[:2] + (o.K,), complex)
    for k in range(k0):
        ak = (-1.0) ** k * k * BETA
        if k == 0:
            uw, wwuu = np.moveaxis(_from_xz(o, np.stack([T["uw", 0], T["ww", 0] - T["uu", 0]], axis=2)), 2, 0)
        else:
            rows = [T["uv", k], T["uw", k], T["vv", k] - T["uu", k], T["vw", k], T["vv", k] - T["ww", k]]
            uv, uw, vvuu, vw, vvww = np.moveaxis(_from_xz(o, np.stack(rows, axis=2)), 2, 0)
        for n in range(o.nn):
            g = float(kz[n, 0, 0])
            _, e, f, h, far = _call(lib.mul, 5, g, ak if k else 1.0, 0)
            for mi in range(o.M):
                a, at = float(kx[0, mi, 0]), (n, mi)
                if k == 0:
                    w = [_call(lib.weights, 2, li, a, g, 0.0)[0] for li in (UW, F)]
                    got[n, mi, 0] = w[0] * uw[at] + w[1] * (g * wwuu[at])
                    continue
                lines = {UW: uw[at], UV: uv[at], E: ak * (vvuu[at] - (vvww[at] if far else 0)) - 1j * e * vw[at],
                         F: f * vvww[at] + 1j * h * vw[at]}
                psi, phi = _psi_phi(lib, lines, a, g, ak)
                if n == 0 and mi == 0:
                    psi, phi = -ak * uv[at], 1j * lines[F] / ak
                got[n, mi, k], got[n, mi, k0 - 1 + k] = psi, phi
    got[0, 0, 0] = 0
    scale = max(np.abs(want[0]).max(), np.abs(want[1]).max())
    assert np.abs(got.real - want[0]).max() <= 1e-13 * scale
    assert np.abs(got.imag - want[1]).max() <= 1e-13 * scale
