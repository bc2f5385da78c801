"""Relaxation of levels of few planes and many columns, of more blocks than the CUs
take at once, and by blocks of 20 planes: the bits of one-sweep launches, the
ring included."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PRECS = [np.float64, np.float32]


def one_sweep(lev, on):
    from warpflow import autotune
    knob = autotune.SWEEP_PAIRS_F64 if lev.dtype == np.float64 else autotune.SWEEP_PAIRS_F32
    autotune.set_shape(knob, lev.n3, 1 if on else 0)


def plan(lev, n):
    from warpflow import _hip
    out = (C.c_int32 * 4)()
    d = lev.desc()
    _hip.call("wf_mg_relax_plan", C.byref(d), n, out)
    return tuple(out)


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("n3", [(8, 80, 80), (8, 96, 64), (8, 31, 256), (12, 96, 96), (7, 90, 90),
                                (15, 90, 90), (2, 200, 130), (128, 128, 128)])
def test_flat_levels_equal_one_sweep_launches(gpu, prec, n3):
    from warpflow import _hip, autotune
    from warpflow.multigrid import _Level
    lev = _Level(n3, tuple(1.0 / n for n in n3), None, prec)
    rng = np.random.default_rng(11)
    lev.rhs.assign(rng.standard_normal(lev.shape))
    phi = np.zeros(lev.shape)
    phi[1:-1, 1:-1, 1:-1] = rng.standard_normal(n3)
    d = lev.desc()
    autotune.reset()
    try:
        if n3[0] == 128 and prec == np.float32:
            assert plan(lev, 6)[2] == 20
        for n in (2, 6, 7):
            got = []
            for one in (True, False):
                one_sweep(lev, one)
                lev.phi.assign(phi)
                _hip.call("wf_mg_relax", C.byref(d), n, None)
                got.append(lev.phi.numpy())
            assert np.array_equal(got[0], got[1]), n
    finally:
        autotune.reset()


# through the V-cycle: a level may relax by another kernel before the coarse
# correction than after it, where blocks also add the interpolation
@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("n3", [(16, 160, 160), (16, 62, 512), (8, 1024, 1024), (4, 48, 40),
                                (2, 20, 40), (40, 16, 24)])
def test_flat_hierarchy_equals_one_sweep_launches(gpu, prec, n3):
    from warpflow import _hip, autotune
    from warpflow.multigrid import _Level
    levs = [_Level(tuple(n >> l for n in n3), tuple(2.0 ** l / n for n in n3), None, prec)
            for l in range(2)]
    rng = np.random.default_rng(12)
    levs[0].rhs.assign(rng.standard_normal(levs[0].shape))
    descs = (_hip.WfMgLevel * 2)(*[lev.desc() for lev in levs])
    autotune.reset()
    try:
        got = []
        for one in (True, False):
            for lev in levs:
                one_sweep(lev, one)
                lev.phi.fill_(0.0)
            _hip.call("wf_mg_vcycle", descs, 2, 6, 5, 20, None)
            got.append([lev.phi.numpy() for lev in levs])
        for a, b in zip(*got):
            assert np.array_equal(a, b)
    finally:
        autotune.reset()


# planes of 121 MB: one-sweep launches, where two-sweep ones would be refused
def test_wide_planes_relax(gpu):
    from warpflow import _hip
    from warpflow.device import zeros
    n3 = (10, 5500, 5500)
    phi, rhs, tmp = [zeros(tuple(n + 2 for n in n3), np.float32) for _ in range(3)]
    d = _hip.WfMgLevel(phi.ptr, rhs.ptr, *n3, 4, *(1.0 / n for n in n3), tmp.ptr, None, 0, 0)
    _hip.call("wf_mg_relax", C.byref(d), 2, None)
    _hip.call("wf_synchronize")
