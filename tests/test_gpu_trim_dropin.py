"""From the native loop to drop-in steps: a drop-in step after trimmed native steps leaves the
state that it leaves after native steps over the reference's ranges (IMHD_TRIM=0), bit for bit
with the ghost cells it updates, before any ghost fill.  FP32 contexts carry compensation terms
of those ghost cells from step to step; eager, replayed and impulsively driven runs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(monkeypatch, trim, dims, riemann, recon, npass, precision, mode):
    from isothermal_mhd_amd import TvdSolver, VanLeerSolver
    monkeypatch.setenv("IMHD_TRIM", trim)
    try:
        if recon == "tvd":
            S = TvdSolver(dims, npass=npass, riemann=riemann, precision=precision)
        else:
            S = VanLeerSolver(dims, npass=npass, riemann=riemann, recon=recon, precision=precision)
    finally:
        monkeypatch.delenv("IMHD_TRIM")
    boxes = [dims] if np.ndim(dims) == 1 else dims
    for b in range(len(boxes)):
        S.init_turbulence(sigma_ln=0.3, b0=(0.4, -0.7, 0.5), kmin=1.0, kmax=2.0, mach=1.5, seed=5 + b, solenoidal=False,
                          passive=npass > 0, box=b)
    S.set_time(t=0.0, dt=1.0e-3)
    if mode == "impulsive":
        S.set_impulsive_forcing(k_max=2, edot=1e-3, dt_turb=2.0e-3)
    out = []
    for n in (5, 1):   # the second drop-in step follows a drop-in step, a ghost fill and one native step
        S.run(n, graph=mode == "graph")
        S.mhd_update(1.0e-3)
        out += [S.get_state(b) for b in range(len(boxes))]
        S.boundary_conditions()
    S.close()
    return out


CASES = [((24, 20, 16), "hlld", "plm", 0, 32, "eager"), ((33, 9, 14), "hlle", "plm", 1, 32, "graph"),
         ((17, 30, 12), "roe", "ppm_prim", 0, 32, "graph"), ((20, 17, 15), "hlld", "ppm_char", 2, 32, "eager"),
         ((16, 18, 20), "hlld", "plm", 0, 32, "impulsive"), ([(8, 33, 14), (31, 6, 22)], "hlld", "plm", 0, 32, "graph"),
         ((20, 17, 15), "hlld", "plm", 1, 64, "eager"), ((18, 24, 13), "roe", "tvd", 1, 32, "eager")]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_dropin_step_after_native_steps(monkeypatch, i):
    print("[gpu] native steps, then a drop-in step", *CASES[i], flush=True)
    ref = run(monkeypatch, "0", *CASES[i])
    got = run(monkeypatch, "1", *CASES[i])
    for a, b in zip(ref, got):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
