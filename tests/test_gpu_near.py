"""The fused FP64 predictor and PLM corrector (k_vl_near): velocities, primitives and slopes
formed once per cell and shared by its faces, bit for bit the three-kernel path (IMHD_VSTAGE=0),
whose faces form their own, where tiles and z-segments begin and end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(monkeypatch, env, dims, riemann, bc, npass):
    from isothermal_mhd_amd import VanLeerSolver
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    try:
        S = VanLeerSolver(dims, npass=npass, riemann=riemann, recon="plm", bc=bc, precision=64)
    finally:
        for k in env:
            monkeypatch.delenv(k)
    boxes = [dims] if np.ndim(dims) == 1 else dims
    for b in range(len(boxes)):
        S.init_turbulence(sigma_ln=0.3, b0=(0.4, -0.7, 0.5), kmin=1.0, kmax=1.0, mach=1.5, seed=3 + b, solenoidal=False,
                          passive=npass > 0, box=b)
    S.set_time(t=0.0, dt=1.0e-3)
    S.run(4, graph=False)
    out = [x for b in range(len(boxes)) for x in S.get_state(b)] + [np.asarray(v) for v in S.get_time()]
    S.close()
    return out


# 14 (30) columns per tile; boxes of fewer cells than ghost layers have images in ghost cells
EDGES = [(6, 6, 6), (9, 7, 6), (10, 24, 8), (11, 10, 9), (25, 38, 7), (14, 16, 15), (28, 9, 33), (64, 23, 40),
         [(12, 17, 9), (31, 8, 22), (6, 40, 14)]]


@pytest.mark.parametrize("i", range(len(EDGES)))
@pytest.mark.parametrize("shape", ["0", "1"])
@pytest.mark.parametrize("riemann", ["hlld", "hlle", "roe"])
def test_near_stages_fp64_bitwise(monkeypatch, i, shape, riemann):
    dims, bc, npass = EDGES[i], ("periodic", "open")[i % 2], i % 3
    print("[gpu] near stages", dims, shape, riemann, bc, npass, flush=True)
    ref = run(monkeypatch, {"IMHD_VSTAGE": "0"}, dims, riemann, bc, npass)
    for env in ({}, {"IMHD_VSEG": "1"}, {"IMHD_VSEG": "7"}):
        got = run(monkeypatch, {"IMHD_VSHAPE": shape, **env}, dims, riemann, bc, npass)
        for x, y in zip(ref, got):
            assert np.array_equal(x, y), env
