"""Decoding of a launch's items into cells (32-bit, from the workgroup's first item) against
the y-strip order (IMHD_STRIP=1), which decodes every item on its own in 64 bits: the same
bits from every per-cell kernel, on rows shorter than, of and just over a wave and a
workgroup, planes of few and of many rows, single boxes and an ensemble; and the ghost fill,
with passives, against numpy's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SPEED = {"vl": "vanleer", "tvd": "tvd"}
SIZES = [(6, 6, 6), (7, 61, 6), (51, 6, 7), (52, 9, 6), (53, 6, 52), (115, 7, 6), (243, 6, 6), (245, 7, 6), (6, 244, 6),
         (6, 7, 130), [(6, 13, 7), (53, 9, 8), (130, 6, 6)]]


def make(monkeypatch, scheme, dims, strip):
    from isothermal_mhd_amd import TvdSolver, VanLeerSolver
    monkeypatch.setenv("IMHD_STRIP", strip)
    monkeypatch.setenv("IMHD_VSTAGE", "0")
    monkeypatch.setenv("IMHD_ZSEG", "0")
    try:
        S = (TvdSolver if scheme == "tvd" else VanLeerSolver)(dims, precision=64, npass=2)
    finally:
        for v in ("IMHD_STRIP", "IMHD_VSTAGE", "IMHD_ZSEG"):
            monkeypatch.delenv(v)
    boxes = [dims] if np.ndim(dims) == 1 else dims
    for b in range(len(boxes)):
        S.init_turbulence(sigma_ln=0.3, b0=(0.4, -0.7, 0.5), kmin=1.0, kmax=2.0, mach=1.5, seed=5 + b, solenoidal=False, box=b)
    return S, len(boxes)


@pytest.mark.parametrize("scheme", ["vl", "tvd"])
@pytest.mark.parametrize("dims", SIZES)
def test_item_order_bitwise(monkeypatch, scheme, dims):
    print("[gpu] items", scheme, dims, flush=True)
    out = []
    for strip in ("1", "0"):
        S, n = make(monkeypatch, scheme, dims, strip)
        S.set_time(t=0.0, dt=1.0e-3)
        S.run(2, graph=False)
        out.append([x for b in range(n) for x in S.get_state(b)[:2]] + [np.asarray(getattr(S, f"get_max_speed_{SPEED[scheme]}")())])
        S.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("bc", ["periodic", "open"])
@pytest.mark.parametrize("dims", [(6, 6, 6), (7, 61, 9), (53, 6, 8), (130, 7, 6), [(6, 13, 7), (65, 9, 8)]])
def test_ghost_fill(bc, dims):
    from isothermal_mhd_amd import VanLeerSolver
    nb, npass = 6, 3
    S = VanLeerSolver(dims, precision=64, npass=npass, bc=bc)
    boxes = [dims] if np.ndim(dims) == 1 else dims
    rng = np.random.default_rng(3)
    states = []
    for b, d in enumerate(boxes):
        q, bf, qp = (rng.random(tuple(n + 2 * w for n in d) + (f,)) for w, f in ((nb, 7), (nb, 3), (nb - 2, npass)))
        S.set_state(q, bf, qp, box=b)
        states.append((q, bf, qp))
    print("[gpu] ghost fill", bc, dims, flush=True)
    S.boundary_conditions()
    mode = "wrap" if bc == "periodic" else "edge"
    for b, (q, bf, qp) in enumerate(states):
        for got, ref, w, depth in zip(S.get_state(b), (q, bf, qp), (nb, nb, nb - 2), (nb, nb, 3)):
            want = ref.copy()
            n = boxes[b]
            inner = ref[w:w + n[0], w:w + n[1], w:w + n[2]]
            o = w - depth
            want[o:o + n[0] + 2 * depth, o:o + n[1] + 2 * depth, o:o + n[2] + 2 * depth] = \
                np.pad(inner, [(depth, depth)] * 3 + [(0, 0)], mode=mode)
            assert np.array_equal(got, want)
    S.close()
