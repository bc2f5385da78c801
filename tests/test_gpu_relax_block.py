"""Relaxation by overlapping blocks (several sweeps per launch): the same bits
as one-sweep launches, which the sweep tests tie to the oracle's half-sweeps."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def relax(lev, phi, n, one_sweep):
    from warpflow import _hip, autotune
    f64 = lev.dtype == np.float64
    autotune.reset()
    try:
        if one_sweep:
            autotune.set_shape(autotune.SWEEP_PAIRS_F64 if f64 else autotune.SWEEP_PAIRS_F32,
                               lev.n3, 1)
        lev.phi.assign(phi)
        d = lev.desc()
        _hip.call("wf_mg_relax", C.byref(d), n, None)
        return lev.phi.numpy()
    finally:
        autotune.reset()


# one block (of 8, 12 and 16 planes, whole and part), a few blocks per axis, last
# blocks that overlap the one before, thin and odd levels, and (FP32) the
# 32 x 32 columns of the largest levels
@pytest.mark.parametrize("prec", [np.float64, np.float32])
@pytest.mark.parametrize("n3", [(1, 2, 2), (3, 5, 4), (8, 8, 8), (9, 12, 16), (12, 12, 12),
                                (13, 16, 7), (16, 16, 16), (17, 16, 15), (7, 33, 18),
                                (24, 24, 24), (33, 2, 40), (37, 42, 70), (96, 81, 100)])
def test_blocks_equal_one_sweep_launches(gpu, prec, n3):
    from warpflow.multigrid import _Level
    lev = _Level(n3, tuple(1.0 / n for n in n3), None, prec)
    rng = np.random.default_rng(5)
    lev.rhs.assign(rng.standard_normal(lev.shape))
    phi = np.zeros(lev.shape)
    phi[1:-1, 1:-1, 1:-1] = rng.standard_normal(n3)
    for n in (2, 3, 6, 7):
        want = relax(lev, phi, n, True)
        assert np.array_equal(relax(lev, phi, n, False), want), n


# members whose levels are one block each (all sweeps in one launch), a few
# blocks, and blocks of fewer planes than the kernel's
@pytest.mark.parametrize("sizes,levels", [([(16, 12, 8), (12, 8, 16)], 2),
                                          ([(20, 36, 24), (28, 12, 16), (36, 20, 44)], 2),
                                          ([(56, 40, 24), (24, 72, 56)], 4)])
def test_batched_blocks_equal_single_solvers(gpu, sizes, levels):
    from warpflow import FlowSolver, build_topology
    from warpflow.ensemble import Ensemble, MemberSpec, member_config
    specs = [MemberSpec(n3, 200.0 + 100.0 * m, m + 1) for m, n3 in enumerate(sizes)]
    ens = Ensemble(specs, 5e-4, mg_levels=levels)
    for _ in range(2):
        ens.step()
    for m, sp in enumerate(specs):
        cfg = member_config(sp, 5e-4, mg_levels=levels)
        sol = FlowSolver(cfg, build_topology(cfg), "hip:0")
        for _ in range(2):
            sol.step()
        for name in ("u", "v", "w", "p"):
            assert np.array_equal(ens.field(name, m).numpy(), sol.f[name].numpy()), (m, name)
    ens.close()
