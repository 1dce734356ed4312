"""A context's spectrum buffers: a vector spectrum takes no more memory than a density spectrum;
once the mode spectra have made their buffers, a vector spectrum packs its three components
together into them and sums the same REAL*4 numbers as one component at a time: equal to 1e-12,
the order of the FP64 shell sums."""
import numpy as np
import pytest

from refutil import random_state

pytestmark = pytest.mark.gpu

VECTORS = ("velocity", "bfield", "vpar", "vperp")


@pytest.mark.parametrize("n,precision", [(6, 64), (34, 64), (66, 32)])
def test_vector_spectra_memory_and_packing(n, precision):
    from isothermal_mhd_amd import VanLeerSolver
    print(f"[gpu] spectrum buffers n={n} fp{precision}", flush=True)
    q, bf, _ = random_state(n, n, n, npass=0, seed=31 + n, amp_v=0.6, b0=(0.5, 0.2, 0.1))
    S = VanLeerSolver((n, n, n), npass=0, precision=precision)
    S.set_state(q, bf, None)
    S.spectrum("density")
    held = S.device_bytes()
    single = {f: S.spectrum(f)[1] for f in VECTORS}
    assert S.device_bytes() == held
    S.mode_spectra()
    modes = S.device_bytes()
    assert modes == held + 2 * n * n * (n // 2 + 1) * 8
    for f in VECTORS:
        assert np.allclose(S.spectrum(f)[1], single[f], rtol=1e-12, atol=0), f
    assert S.device_bytes() == modes
    S.close()
