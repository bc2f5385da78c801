"""FP64 coarse operators above 4096 cells, by the level's reflections, against the
sweeps they stand for.  A row sums N products, so N 2^-53 on either side of the
largest value (N = 16384: 4e-12 in all), and the sweeps add 600 half-sweeps of 8
roundings (5e-13): 1e-11."""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def level(n3, h, prec=np.float64):
    from warpflow.multigrid import _Level
    lev = _Level(n3, h, None, prec)
    lev.rhs.assign(np.random.default_rng(9).standard_normal(lev.shape))
    return lev


# the smallest and the largest, flat and long ones, unequal spacings, few sweeps
# and none (phi = 0)
@pytest.mark.parametrize("n3", [(18, 16, 16), (16, 32, 32), (64, 8, 16), (2, 64, 48), (32, 128, 2)])
@pytest.mark.parametrize("h", [(1.0, 1.0, 1.0), (1.0, 0.1, 0.02), (0.01, 0.5, 1.0)])
@pytest.mark.parametrize("nsweeps", [0, 1, 300])
def test_reflections_equal_sweeps(gpu, n3, h, nsweeps):
    from warpflow import _hip
    a, b = level(n3, h), level(n3, h)
    assert a.build_coarse_operator(nsweeps)
    a.phi.fill_(0.0)
    b.phi.fill_(0.0)
    da, db = a.desc(), b.desc()
    _hip.call("wf_mg_coarse_op_apply", C.byref(da), None)
    _hip.call("wf_mg_relax", C.byref(db), nsweeps, None)
    if nsweeps == 0:
        assert not a.phi.numpy().any()
    else:
        assert rel_err(a.phi.numpy(), b.phi.numpy()) < 1e-11


# phi = M rhs whatever phi held, its ring included
@pytest.mark.parametrize("n3,prec", [((20, 20, 20), np.float64), ((12, 12, 12), np.float64),
                                     ((20, 20, 20), np.float32), ((19, 20, 20), np.float64)])
def test_old_iterate_is_not_read(gpu, n3, prec):
    from warpflow import _hip
    lev = level(n3, tuple(1.0 / n for n in n3), prec)
    assert lev.build_coarse_operator(30)
    d = lev.desc()
    got = []
    for old in (0.0, np.nan):
        lev.phi.assign(np.full(lev.shape, old))
        _hip.call("wf_mg_coarse_op_apply", C.byref(d), None)
        got.append(lev.phi.numpy())
    inner = np.zeros(lev.shape, bool)
    for a in range(3):  # real cells and face ring
        s = [slice(1, -1)] * 3
        s[a] = slice(None)
        inner[tuple(s)] = True
    assert np.array_equal(got[0][inner], got[1][inner])
