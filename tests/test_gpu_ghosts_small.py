"""The periodic ghost fill of boxes with fewer cells than ghost layers along an axis: the
reference fills the layers one after the other from layers that are filled already, so every
ghost cell holds the interior cell a whole number of box lengths away."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def images(n, ghosts):
    return [np.mod(np.arange(-ghosts, k + ghosts), k) + ghosts for k in n]


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("dims,nb", [((4, 4, 4), 6), ((5, 9, 4), 6), ((4, 5, 11), 9), ((6, 4, 7), 6), ((6, 6, 6), 6)])
def test_every_ghost_cell_is_an_image(dims, nb, precision):
    from isothermal_mhd_amd import VanLeerSolver
    print("[gpu] ghost fill", dims, nb, precision, flush=True)
    S = VanLeerSolver(dims, nb=nb, npass=2, bc="periodic", precision=precision)
    rng = np.random.default_rng(7)
    sh, shp = S.shapes()
    q, b, qp = (rng.integers(1, 1000, size=s).astype(float) for s in (sh + (7,), sh + (3,), shp[:3] + (2,)))
    S.set_state(q, b, qp)
    S.boundary_conditions()
    got = S.get_state()
    # the passive scalars have two ghost layers less, and three are filled
    for start, x, ghosts, filled in ((q, got[0], nb, nb), (b, got[1], nb, nb), (qp, got[2], nb - 2, 3)):
        want = start[np.ix_(*images(dims, ghosts))]
        cut = tuple(slice(ghosts - filled, ghosts + n + filled) for n in dims)
        assert np.array_equal(x[cut], want[cut])
        outside = np.ones(x.shape[:3], dtype=bool)
        outside[cut] = False
        assert np.array_equal(x[outside], start[outside])
    S.close()
