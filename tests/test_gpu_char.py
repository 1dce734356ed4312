"""The fused FP64 characteristic PPM corrector (k_vl_char): every edge value is formed once
per cell and shared by its faces, with the cells below a tile formed apart.  It is held bit
for bit to the three-kernel path (IMHD_VPPM=0), whose faces form their own edge values,
where tiles and z-segments begin and end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(monkeypatch, env, dims, riemann, bc, npass, steps=4, seed=3):
    from isothermal_mhd_amd import VanLeerSolver
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    try:
        S = VanLeerSolver(dims, npass=npass, riemann=riemann, recon="ppm_char", bc=bc, precision=64)
    finally:
        for k in env:
            monkeypatch.delenv(k)
    boxes = [dims] if np.ndim(dims) == 1 else dims
    for b in range(len(boxes)):
        S.init_turbulence(sigma_ln=0.3, b0=(0.4, -0.7, 0.5), kmin=1.0, kmax=1.0, mach=1.5, seed=seed + b, solenoidal=False,
                          passive=npass > 0, box=b)
    S.set_time(t=0.0, dt=1.0e-3)
    S.run(steps, graph=False)
    out = [S.get_state(b) for b in range(len(boxes))], S.get_time()
    S.close()
    return out


# 14 (30) columns per tile; the corrector reaches four cells beyond the box.  Boxes of fewer
# cells than ghost layers are left out: their periodic images are ghost cells themselves
EDGES = [(6, 6, 6), (9, 7, 6), (10, 24, 8), (11, 10, 9), (25, 38, 7), (14, 16, 15), (28, 9, 33), (64, 23, 40)]


@pytest.mark.parametrize("dims", EDGES)
@pytest.mark.parametrize("shape", ["0", "1"])
def test_char_corrector_fp64_bitwise(monkeypatch, dims, shape):
    i = EDGES.index(dims)
    riemann, bc, npass = ("hlld", "hlle", "roe")[i % 3], ("periodic", "open")[i % 2], i % 3
    print("[gpu] char corrector", dims, shape, riemann, bc, npass, flush=True)
    ref = run(monkeypatch, {"IMHD_VPPM": "0"}, dims, riemann, bc, npass)
    for env in ({}, {"IMHD_VSEG": "1"}, {"IMHD_VSEG": "7"}):
        got = run(monkeypatch, {"IMHD_VSHAPE": shape, **env}, dims, riemann, bc, npass)
        for x, y in zip(ref[0][0], got[0][0]):
            assert np.array_equal(x, y), env
        assert np.array_equal(ref[1][0], got[1][0]) and np.array_equal(ref[1][1], got[1][1])


def test_char_corrector_fp64_ensemble_bitwise(monkeypatch):
    dims = [(12, 17, 9), (31, 8, 22), (6, 40, 14)]
    print("[gpu] char corrector ensemble", flush=True)
    ref = run(monkeypatch, {"IMHD_VPPM": "0"}, dims, "hlld", "periodic", 1)
    got = run(monkeypatch, {}, dims, "hlld", "periodic", 1)
    for a, b in zip(ref[0], got[0]):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
