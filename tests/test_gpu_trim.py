"""Trimmed native steps: on a periodic box the native loop leaves out the ghost cells that
its ghost fill overwrites.  Held bit for bit, state, time, dt and floor count, to the same
run over the reference's ranges (IMHD_TRIM=0), for every integrator, reconstruction and
solver, with passives and forcing, on the smallest boxes and boxes that tiles do not divide,
as single boxes and ensembles, eager and replayed, and across set_state, whose ghost cells
the first step takes as they come."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(monkeypatch, trim, dims, solver, riemann, recon, npass, precision, ou=False, graph=False, strong=False, raw=False):
    from isothermal_mhd_amd import TvdSolver, VanLeerSolver
    monkeypatch.setenv("IMHD_TRIM", trim)
    try:
        if solver == "tvd":
            S = TvdSolver(dims, npass=npass, riemann=riemann, precision=precision)
        else:
            S = VanLeerSolver(dims, npass=npass, riemann=riemann, recon=recon, precision=precision)
    finally:
        monkeypatch.delenv("IMHD_TRIM")
    boxes = [dims] if np.ndim(dims) == 1 else dims
    for b in range(len(boxes)):
        S.init_turbulence(sigma_ln=0.3, b0=(0.4, -0.7, 0.5), kmin=1.0, kmax=2.0, mach=8.0 if strong else 1.5, seed=5 + b,
                          solenoidal=False, passive=npass > 0, box=b)
    if ou:
        S.set_ou_forcing(seed=11)
    S.set_time(t=0.0, dt=2.0e-2 if strong else 1.0e-3)
    S.run(4, graph=graph)
    if raw:   # a state whose ghost cells are no images: the first step reads them
        rng = np.random.default_rng(1)
        for b in range(len(boxes)):
            q, bf, qp = S.get_state(b)
            inner = np.zeros(q.shape[:3], dtype=bool)
            inner[6:-6, 6:-6, 6:-6] = True
            q[..., 0] *= np.where(inner, 1.0, 1.0 + 0.1 * rng.random(q.shape[:3]))
            S.set_state(q, bf, qp, box=b)
        S.run(3, graph=graph)
    out = [S.get_state(b) for b in range(len(boxes))], S.get_time(), S.floor_count()
    S.close()
    return out


CASES = [
    ((6, 6, 6), "vl", "hlld", "plm", 0, 64, {}), ((9, 7, 17), "vl", "roe", "plm", 2, 64, {"graph": True}),
    ((33, 18, 12), "vl", "hlle", "ppm_prim", 1, 64, {}), ((20, 41, 15), "vl", "hlld", "ppm_char", 1, 64, {"raw": True}),
    ((28, 30, 62), "vl", "hlld", "plm", 1, 64, {"ou": True}), ((64, 27, 33), "vl", "hlld", "plm", 1, 32, {"graph": True}),
    ((17, 60, 9), "vl", "roe", "ppm_char", 0, 32, {"raw": True}), ((40, 12, 35), "vl", "hlle", "ppm_prim", 2, 32, {"ou": True}),
    ((24, 24, 24), "vl", "hlld", "plm", 0, 64, {"strong": True}), ((24, 20, 28), "vl", "hlld", "plm", 0, 32, {"strong": True}),
    ([(8, 33, 14), (31, 6, 22), (45, 29, 30)], "vl", "hlle", "plm", 0, 32, {"graph": True, "raw": True}),
    ([(8, 33, 14), (31, 6, 22)], "vl", "hlld", "ppm_char", 1, 64, {"raw": True}),
    ((6, 6, 6), "tvd", "roe", "plm", 0, 64, {}), ((33, 70, 13), "tvd", "roe", "plm", 2, 64, {"graph": True, "raw": True}),
    ((65, 15, 40), "tvd", "roe", "plm", 1, 32, {"ou": True}), ((14, 9, 61), "tvd", "hlle", "plm", 1, 64, {"raw": True}),
    ((24, 24, 24), "tvd", "roe", "plm", 0, 64, {"strong": True}), ((18, 24, 33), "tvd", "hlle", "plm", 0, 32, {"strong": True}),
    ([(8, 33, 14), (31, 6, 22)], "tvd", "roe", "plm", 0, 32, {}),
]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_trimmed_step_bitwise(monkeypatch, i):
    *args, kw = CASES[i]
    print("[gpu] trimmed native step", *args, kw, flush=True)
    ref = run(monkeypatch, "0", *args, **kw)
    got = run(monkeypatch, "1", *args, **kw)
    for a, b in zip(ref[0], got[0]):
        for x, y in zip(a, b):
            assert np.array_equal(x, y, equal_nan=True)
    assert np.array_equal(ref[1][0], got[1][0]) and np.array_equal(ref[1][1], got[1][1])
    assert ref[2] == got[2]
