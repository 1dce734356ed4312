"""The FP32 characteristic PPM corrector forms an edge value once per cell with the roundings
that the form with one evaluation per face and side had: a rounding moved there turns up as a
different limiter branch in single cells.  Pinned bit for bit by that form's own outputs on
MI355X (tests/golden/char32.npz, written by write() with the library of commit 2a24fcd, which
still had it): start and interior after four steps, for each solver, with compensated sums
and a passive scalar."""
import os

import numpy as np
import pytest

from refutil import random_state

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "char32.npz")
# 14 columns per tile: two tiles along x, along y, and segments along z
CASES = {"hlld": (17, 10, 8), "hlle": (9, 18, 7), "roe": (16, 8, 15)}
NB = 6


def inner(dims, ghosts):
    return tuple(slice(ghosts, ghosts + n) for n in dims)


def advance(riemann, q, bf, qp):
    """Interior arrays q (7 fields), bf (3), qp (1) four steps on."""
    from isothermal_mhd_amd import VanLeerSolver
    dims = CASES[riemann]
    S = VanLeerSolver(dims, nb=NB, npass=1, riemann=riemann, recon="ppm_char", precision=32, compensated=True)
    sh, shp = S.shapes()
    full = [np.ones(sh + (7,), order="F"), np.zeros(sh + (3,), order="F"), np.zeros(shp[:3] + (1,), order="F")]
    for a, x, ghosts in zip(full, (q, bf, qp), (NB, NB, NB - 2)):
        a[inner(dims, ghosts)] = x
    S.set_state(*full)
    S.boundary_conditions()
    S.set_time(t=0.0, dt=1.0e-3)
    S.run(4, graph=False)
    out = S.get_state(), S.get_time()
    S.close()
    q, bf, qp = (a[inner(dims, ghosts)] for a, ghosts in zip(out[0], (NB, NB, NB - 2)))
    return q.astype(np.float32), bf, qp.astype(np.float32), np.array([out[1][0][0], out[1][1][0]])


def write(path):
    out = {}
    for i, (riemann, dims) in enumerate(CASES.items()):
        start = random_state(*dims, npass=1, seed=70 + i, amp_v=1.2, amp_rho=0.6, amp_b=0.6)
        start = [a[inner(dims, ghosts)].astype(np.float32) for a, ghosts in zip(start, (NB, NB, NB - 2))]
        for name, x in zip(("q0", "b0", "p0"), start):
            out[f"{riemann}_{name}"] = x
        for name, x in zip(("q", "b", "p", "t"), advance(riemann, *start)):
            out[f"{riemann}_{name}"] = x
    np.savez_compressed(path, **out)


@pytest.mark.parametrize("riemann", list(CASES))
def test_same_bits_as_the_per_face_form(riemann):
    print("[gpu] FP32 char corrector, pinned bits", riemann, flush=True)
    gold = np.load(GOLD)
    got = advance(riemann, *(gold[f"{riemann}_{n}"] for n in ("q0", "b0", "p0")))
    for name, x in zip(("q", "b", "p", "t"), got):
        assert np.array_equal(x, gold[f"{riemann}_{name}"]), name
