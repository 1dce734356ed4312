"""The fused Roe-TVD x sweep over the flat list of rows (waves of 62 + 2 entries) and the
y / z sweeps in segments of any length: FP64 bit for bit the two-kernel sweeps
(IMHD_TVDFUSE=0), on rows shorter than a wave, of just under and over one wave and two, and
columns that no segment divides; single boxes, an ensemble, drop-in and native steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(monkeypatch, fuse, dims, native):
    from isothermal_mhd_amd import TvdSolver
    monkeypatch.setenv("IMHD_TVDFUSE", fuse)
    try:
        S = TvdSolver(dims, precision=64)
    finally:
        monkeypatch.delenv("IMHD_TVDFUSE")
    boxes = [dims] if np.ndim(dims) == 1 else dims
    for b in range(len(boxes)):
        S.init_turbulence(sigma_ln=0.3, b0=(0.4, -0.7, 0.5), kmin=1.0, kmax=2.0, mach=1.5, seed=5 + b, solenoidal=False, box=b)
    if native:
        S.set_time(t=0.0, dt=1.0e-3)
        S.run(3, graph=False)
    else:
        for _ in range(2):
            S.tvd_solve_3d(1.0e-3)
            S.boundary_conditions()
    out = [S.get_state(b)[:2] for b in range(len(boxes))]
    S.close()
    return out


@pytest.mark.parametrize("dims", [(6, 6, 6), (7, 19, 11), (58, 6, 9), (59, 7, 8), (60, 9, 6), (61, 8, 7), (62, 6, 8), (63, 9, 9),
                                  (119, 7, 6), (122, 6, 7), (125, 8, 6), (13, 131, 8), (9, 12, 97),
                                  [(6, 13, 7), (61, 9, 8), (130, 6, 6)]])
def test_fused_sweeps_bitwise(monkeypatch, dims):
    for native in (False, True):
        print("[gpu] fused TVD sweeps", dims, native, flush=True)
        ref = run(monkeypatch, "0", dims, native)
        got = run(monkeypatch, "1", dims, native)
        for a, b in zip(ref, got):
            for x, y in zip(a, b):
                assert np.array_equal(x, y)
