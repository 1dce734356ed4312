"""The next time step is formed by one wavefront per box: an ensemble of more boxes than a
wavefront has lanes takes, box by box, the steps that each box takes alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", ["vl", "tvd"])
@pytest.mark.parametrize("nbox", [1, 5, 70])
def test_ensemble_time_steps(solver, nbox):
    from isothermal_mhd_amd import TvdSolver, VanLeerSolver
    cls, kw = (TvdSolver, {}) if solver == "tvd" else (VanLeerSolver, {"riemann": "hlld"})
    dims = [(6 + b % 3, 6 + b % 4, 7 + b % 2) for b in range(nbox)]

    def run(boxes):
        print("[gpu] new dt", solver, nbox, len(boxes), flush=True)
        S = cls([dims[b] for b in boxes], bc="periodic", precision=64, **kw)
        for n, b in enumerate(boxes):
            S.init_turbulence(sigma_ln=0.2, b0=(0.3, 0.1 + 0.01 * b, 0.2), kmin=1.0, kmax=1.0, mach=0.5 + 0.02 * b,
                              seed=100 + b, solenoidal=True, passive=False, box=n)
        S.set_time(t=0.0, dt=1.0e-3)
        S.run(3, graph=False)
        t, dt = S.get_time()
        S.close()
        return np.atleast_1d(t), np.atleast_1d(dt)

    t, dt = run(list(range(nbox)))
    assert len(np.unique(dt)) == nbox
    for b in sorted({0, nbox // 2, nbox - 1}):
        t1, dt1 = run([b])
        assert t1[0] == t[b] and dt1[0] == dt[b]
