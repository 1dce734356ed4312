"""The Roe-TVD sweeps where their work is cut.  A row or column of n cells has n + 9 faces in a
predictor and n + 5 in a corrector, four fewer of each in a trimmed native step.

FP32: the x sweep's flat list (two entries more than faces per row, waves of 62 + 2), the y / z
sweeps' segments.  FP64: the x sweep's flat list of cells (three more than faces per row, waves
of 61 + 3), the y / z sweeps' flat list of columns (two more than faces per column, workgroups
of 30 + 2 entries, 8 x-neighbours).  Hence rows of 63, 64 and 65 entries in either list and
stage and of several waves, columns of 31, 32 and 33 entries and of several workgroups, columns
that no segment divides, and widths that are no multiple of 8.

Against the two-kernel sweeps (IMHD_TVDFUSE=0), which form the same fluxes face by face: FP64
bit for bit; FP32 within two stages of six faces per cell and step, some hundred roundings per
face, relative to the field's maximum.  A face left out, taken twice or given a wrong neighbour
changes a cell by about dt / dx times the flux, 1e-2 of the maximum.

And FP32 bit for bit: a box alone, whose segments are cut to fill the chip, and the same box as
part of an ensemble, whose boxes have segments of 32 or 8 faces."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STEPS = 2
TOL = STEPS * 2 * 6 * 100 * 2.0 ** -24


def run(monkeypatch, fuse, dims, native, precision=32):
    from isothermal_mhd_amd import TvdSolver
    monkeypatch.setenv("IMHD_TVDFUSE", fuse)
    try:
        S = TvdSolver(dims, precision=precision)
    finally:
        monkeypatch.delenv("IMHD_TVDFUSE")
    boxes = [dims] if np.ndim(dims) == 1 else dims
    for b in range(len(boxes)):
        S.init_turbulence(sigma_ln=0.3, b0=(0.4, -0.7, 0.5), kmin=1.0, kmax=2.0, mach=1.5, seed=5 + b, solenoidal=False, box=b)
    if native:
        S.set_time(t=0.0, dt=1.0e-3)
        S.run(STEPS, graph=False)
    else:
        for _ in range(STEPS):
            S.tvd_solve_3d(1.0e-3)
            S.boundary_conditions()
    out = [S.get_state(b)[:2] for b in range(len(boxes))]
    S.close()
    return out


DIMS = [(6, 6, 6), (7, 19, 11), (52, 6, 8), (53, 8, 7), (54, 7, 9), (55, 6, 7), (56, 7, 6), (57, 8, 6), (58, 6, 9), (59, 7, 8), (60, 9, 6), (61, 8, 7), (62, 6, 8),
        (63, 9, 9), (119, 7, 6), (122, 6, 7), (125, 8, 6), (150, 6, 9), (13, 131, 8), (9, 12, 97), (6, 8, 203)]


ROWS64 = [(n, 6 + n % 4, 6 + n % 3) for n in (51, 52, 53, 55, 56, 57, 59, 60, 61, 110, 171)]
COLUMNS64 = [(6 + n % 9, n, 6) for n in (20, 21, 22, 24, 25, 26, 28, 29, 30, 79)] + \
            [(6 + n % 7, 7, n) for n in (20, 21, 22, 24, 25, 26, 28, 29, 30, 111)]


@pytest.mark.parametrize("dims", ROWS64 + COLUMNS64 + [[(9, 25, 7), (53, 8, 6), (11, 6, 29)]])
def test_fused_sweeps_fp64(monkeypatch, dims):
    for native in (False, True):
        print("[gpu] fused FP64 TVD sweeps", dims, native, flush=True)
        ref = run(monkeypatch, "0", dims, native, 64)
        got = run(monkeypatch, "1", dims, native, 64)
        for a, b in zip(ref, got):
            for x, y in zip(a, b):
                assert np.array_equal(x, y)


@pytest.mark.parametrize("dims", DIMS + [[(6, 13, 7), (61, 9, 8), (130, 6, 6), (9, 140, 7)]])
def test_fused_sweeps_fp32(monkeypatch, dims):
    for native in (False, True):
        print("[gpu] fused FP32 TVD sweeps", dims, native, flush=True)
        ref = run(monkeypatch, "0", dims, native)
        got = run(monkeypatch, "1", dims, native)
        for a, b in zip(ref, got):
            for x, y in zip(a, b):
                for f in range(x.shape[-1]):
                    assert np.abs(x[..., f] - y[..., f]).max() <= TOL * np.abs(x).max(), f


@pytest.mark.parametrize("dims", [(61, 9, 8), (9, 131, 10), (12, 10, 143), (40, 33, 35)])
def test_single_box_and_ensemble_bitwise(monkeypatch, dims):
    for native in (False, True):
        print("[gpu] FP32 TVD sweeps, alone and in an ensemble", dims, native, flush=True)
        one = run(monkeypatch, "1", dims, native)[0]
        # the first box of an ensemble has the same seed
        both = run(monkeypatch, "1", [dims, (7, 11, 6)], native)[0]
        for x, y in zip(one, both):
            assert np.array_equal(x, y)
