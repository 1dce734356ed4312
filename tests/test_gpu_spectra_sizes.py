"""Spectra, mode spectra and density PDF where a workgroup serves one partial run of modes or
cells, rows shorter than a wave, and several runs: against the oracle with the tolerances of
tests/test_gpu_spectra.py.  A spectrum whose components are packed one at a time (no room for
three) sums the same REAL*4 numbers: equal to 1e-12, the order of the FP64 shell sums."""
import os
import sys

import numpy as np
import pytest

from refutil import random_state

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(os.path.dirname(HERE), "oracle"))
import spectra as SP  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision", [(6, 64), (14, 32), (34, 64), (66, 32), (130, 32)])
def test_sizes_against_oracle(monkeypatch, n, precision):
    from isothermal_mhd_amd import VanLeerSolver
    print(f"[gpu] spectra n={n} fp{precision}", flush=True)
    q, bf, _ = random_state(n, n, n, npass=0, seed=31 + n, amp_v=0.6, b0=(0.5, 0.2, 0.1))
    S = VanLeerSolver((n, n, n), npass=0, precision=precision)
    T = VanLeerSolver((n, n, n), npass=0, precision=precision)
    for s in (S, T):
        s.set_state(q, bf, None)
    qs = S.get_state()[0]

    def near(got, want):
        return np.all(np.abs(got - want) <= 2e-5 * np.max(np.abs(want)) + 1e-4 * np.abs(want))

    for which, name in enumerate(["density", "velocity", "bfield", "vpar", "vperp"]):
        k, pk = S.spectrum(name)
        ko, po = SP.spectrum(qs, (n, n, n), which)
        assert np.array_equal(k, ko) and near(pk, po), name
        monkeypatch.setenv("IMHD_TEST_SPEC_SINGLE", "1")
        assert np.allclose(T.spectrum(name)[1], pk, rtol=1e-12, atol=0), name
        monkeypatch.delenv("IMHD_TEST_SPEC_SINGLE")
    k, P = S.mode_spectra()
    ko, Po = SP.mode_spectra(qs, (n, n, n))
    for m in range(8):
        assert near(P[m], Po[m]), m
    for nbins, rmax in ((n, 4.0), (3 * n, 2.0), (5000, 3.0)):
        assert np.array_equal(S.density_pdf(nbins, rmax)[1], SP.density_pdf(qs, (n, n, n), nbins, rmax)[1])
    S.close()
    T.close()
