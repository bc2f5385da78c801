"""V-cycles whose small levels run as one-workgroup legs: every level's iterate
and right-hand side have the bits of the per-level launches (which a launch
shape tuned for the levels selects)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def vcycle(mg, phi, rhs, per_level):
    from warpflow import autotune
    f64 = mg.levels[0].dtype == np.float64
    autotune.reset()
    try:
        for lev in mg.levels if per_level else ():
            autotune.set_shape(autotune.SWEEP_PAIRS_F64 if f64 else autotune.SWEEP_PAIRS_F32,
                               lev.n3, 1)
        for lev in mg.levels:
            lev.phi.zero_()
            lev.rhs.zero_()
        mg.levels[0].phi.assign(phi)
        mg.levels[0].rhs.assign(rhs)
        mg._vcycle()
        mg._refill(mg.levels[0])
        return [a.numpy() for lev in mg.levels for a in (lev.phi, lev.rhs)]
    finally:
        autotune.reset()


# legs from the first, second and third level; whole and part segments and columns
# (RI = 4, 8, 24, 32), thin levels, the most columns and planes a shape takes
@pytest.mark.parametrize("prec", [np.float64, np.float32])
@pytest.mark.parametrize("n3,levels", [
    ((24, 24, 24), 3), ((4, 4, 4), 2), ((16, 16, 16), 3), ((12, 20, 16), 2), ((20, 24, 28), 3),
    ((32, 32, 32), 3), ((32, 8, 8), 2), ((8, 32, 32), 2), ((6, 2, 18), 2), ((2, 16, 14), 2),
    ((48, 40, 64), 4), ((88, 60, 52), 3), ((64, 56, 60), 3), ((10, 34, 30), 2), ((72, 16, 48), 4),
    ((112, 96, 104), 2),
])
@pytest.mark.parametrize("sweeps", [(6, 6), (1, 3)])
def test_legs_equal_levels(n3, levels, prec, sweeps):
    from types import SimpleNamespace as NS
    from warpflow.multigrid import SIDES, Multigrid
    cfg = NS(boundaries=NS(**{s: "wall" for s in SIDES}), numerics=NS(mg_levels=levels))
    topo = NS(neighbors={a: (-1, -1) for a in "xyz"}, local_ncells=n3)
    mg = Multigrid(cfg, topo, None, 1.0 / n3[0], 1.2 / n3[1], 0.9 / n3[2], prec)
    mg.n_pre, mg.n_post = sweeps
    rng = np.random.default_rng(7)
    shape = mg.levels[0].shape
    phi = np.zeros(shape, prec)
    phi[1:-1, 1:-1, 1:-1] = rng.standard_normal(n3)
    rhs = np.zeros(shape, prec)
    rhs[1:-1, 1:-1, 1:-1] = rng.standard_normal(n3)
    got = vcycle(mg, phi, rhs, False)
    want = vcycle(mg, phi, rhs, True)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)
