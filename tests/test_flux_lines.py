"""CPU pin of the lines that the flux-form z kernel hands to the x kernel
(zflux.hpp, dev_term in kernels.hpp): five real rows and four lines per
wall-normal index k >= 1 (uw, F, uv, E; two for k = 0), of which psi and phi of
the nonlinear term are polynomials in alpha m.  The same algebra in numpy
against var_spec2mpt (program/variables.f90:440-480) of the advective nonlinear
term, at every mode, the mean mode included."""
import ctypes
import math

import numpy as np
import pytest

import oracle
from test_oracle_nonlinear import BETA, CASES, _from_xz, _gen, _state, _to_xz, _wavenumbers


@pytest.mark.parametrize("k0,mm,nn,theta,alpha,gamma", CASES)
def test_lines_give_psi_phi_of_the_nonlinear_term(k0, mm, nn, theta, alpha, gamma):
    o = oracle.Oracle(k0, mm, nn, alpha, gamma, 200.0, 0.02, theta=theta)
    re, im = _state(o, 13 * k0 + mm + 2 * nn)
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
    a, g = kx[:, :, 0], kz[:, :, 0]
    got = np.zeros(s.shape[:2] + (o.K,), complex)
    for k in range(k0):
        ak = (-1) ** k * k * BETA
        zero = np.zeros_like(T["uu", 0])
        uv, vw, vv = (T.get((n, k), zero) for n in ("uv", "vw", "vv"))
        rows = [uv, T["uw", k], vv - T["uu", k], vw, vv - T["ww", k]]
        F = _from_xz(o, np.stack(rows, axis=2))
        UV, UW, VVUU, VW, VVWW = (F[:, :, i] for i in range(5))
        psi = (a ** 2 - g ** 2) * UW
        if k == 0:
            psi = psi + a * (g * (VVUU - VVWW))
        else:
            E = ak * VVUU - 1j * g * VW
            Fk = ak * g * VVWW + 1j * (ak ** 2 - g ** 2) * VW
            psi = psi + 1j * g * ak * UV + (a / ak) * (g * E - Fk)
            phi = a ** 2 * E + g * Fk - 2 * ak * a * g * UW + 1j * a * (ak ** 2 - a ** 2 - g ** 2) * UV
            psi[0, 0], phi[0, 0] = -ak * UV[0, 0], 1j * Fk[0, 0] / ak
            got[:, :, k0 - 1 + k] = phi
        got[:, :, k] = psi
    scale = max(np.abs(want[0]).max(), np.abs(want[1]).max())
    # same bound as the composed term itself: rounding of order-one sums
    assert np.abs(got.real - want[0]).max() <= 1e-13 * scale
    assert np.abs(got.imag - want[1]).max() <= 1e-13 * scale


@pytest.mark.parametrize("k0", [4, 6])
def test_generated_rows_leave_out_only_the_profile_constants(k0, tmp_path):
    """flux_gen.hpp's rows, compiled for the host, at random points: the rows of
    the full field (perturbation plus laminar profile) minus the profile's own
    products."""
    import os
    import subprocess
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mwf_amd", "csrc")
    rows, kk = _gen().dev_rows(k0), 3 * k0 - 1
    src = tmp_path / "rows.cpp"
    src.write_text("#define __host__\n#define __device__\n#define __forceinline__ inline\n"
                   f'#include "{csrc}/flux_gen.hpp"\n'
                   'extern "C" void rows(const double* v, double lu, double lw, double* out) {\n'
                   + "".join(f"  out[{r}] = FluxRows<{k0}>::row<{r}>(v, lu, lw);\n" for r in range(len(rows))) + "}\n")
    lib = tmp_path / "rows.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    fn = ctypes.CDLL(str(lib)).rows
    dp = ctypes.POINTER(ctypes.c_double)
    fn.argtypes = [dp, ctypes.c_double, ctypes.c_double, dp]
    rng = np.random.default_rng(k0)
    for _ in range(20):
        v, lu, lw = rng.standard_normal(kk), *rng.standard_normal(2)
        got = np.empty(len(rows))
        fn(v.ctypes.data_as(dp), lu, lw, got.ctypes.data_as(dp))
        prof = np.zeros(kk)
        prof[1], prof[2 * k0] = lu, lw
        for r, (name, terms) in enumerate(rows):
            want = sum(float(c) * ((v + prof)[a] * (v + prof)[b] - prof[a] * prof[b]) for a, b, c in terms)
            assert abs(got[r] - want) <= 1e-13, name
