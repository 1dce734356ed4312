"""The fused FP32 characteristic PPM corrector: a cell's edge values are formed once, whatever
tile or z-segment its faces belong to, so tile shapes and segments give the same bits; they
agree with the three-kernel path (IMHD_VPPM=0), whose faces form their own edge values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(monkeypatch, env, dims, riemann, bc, npass, compensated, steps=4, seed=3):
    from isothermal_mhd_amd import VanLeerSolver
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    try:
        S = VanLeerSolver(dims, npass=npass, riemann=riemann, recon="ppm_char", bc=bc, precision=32, compensated=compensated)
    finally:
        for k in env:
            monkeypatch.delenv(k)
    S.init_turbulence(sigma_ln=0.3, b0=(0.4, -0.7, 0.5), kmin=1.0, kmax=1.0, mach=1.5, seed=seed, solenoidal=False,
                      passive=npass > 0)
    S.set_time(t=0.0, dt=1.0e-3)
    S.run(steps, graph=False)
    out = S.get_state(), S.get_time()
    S.close()
    return out


# 14 (30) columns per tile; the corrector reaches four cells beyond the box
EDGES = [(6, 6, 6), (9, 7, 6), (10, 24, 8), (11, 10, 9), (25, 38, 7), (14, 16, 15), (28, 9, 33), (64, 23, 40)]
# four steps of six faces with some eighty roundings each
TOL = 4 * 6 * 80 * 2.0 ** -24


@pytest.mark.parametrize("dims", EDGES)
def test_char_corrector_fp32(monkeypatch, dims):
    i = EDGES.index(dims)
    riemann, bc, npass, comp = ("hlld", "hlle", "roe")[i % 3], ("periodic", "open")[i % 2], i % 3, i % 4 != 1
    print("[gpu] FP32 char corrector", dims, riemann, bc, npass, comp, flush=True)
    ref = run(monkeypatch, {"IMHD_VPPM": "0"}, dims, riemann, bc, npass, comp)
    first = run(monkeypatch, {"IMHD_VSHAPE_C": "0"}, dims, riemann, bc, npass, comp)
    for x, y in zip(ref[0], first[0]):
        assert np.abs(x - y).max() <= TOL * np.abs(x).max() if x.size else True
    # shape 2 has no tiles of its own here and runs on shape 1's
    for env in ({"IMHD_VSHAPE_C": "1"}, {"IMHD_VSHAPE": "2"}, {"IMHD_VSHAPE_C": "0", "IMHD_VSEG": "1"},
                {"IMHD_VSHAPE_C": "1", "IMHD_VSEG": "7"}, {}):
        got = run(monkeypatch, env, dims, riemann, bc, npass, comp)
        for x, y in zip(first[0], got[0]):
            assert np.array_equal(x, y), env
        assert np.array_equal(first[1][0], got[1][0]) and np.array_equal(first[1][1], got[1][1]), env
