"""The smoother chosen for a level (wf_mg_relax_plan): host logic only, the level's
array addresses are never followed."""
import ctypes as C

import pytest

BLOCKS, LDS, SWEEP2, SWEEP, HALF = 1, 2, 3, 4, 5
N = (1, 2, 3, 7, 8, 9, 12, 13, 16, 17, 20, 31, 32, 33, 40, 64, 80, 90, 96, 128, 160, 256, 400)


def plan(n3, prec, nsweeps, tmp=True):
    from warpflow import _hip
    lev = _hip.WfMgLevel(64, 64, *n3, prec, *(1.0 / n for n in n3), 64 if tmp else None, None,
                         0, 0)
    out = (C.c_int32 * 4)()
    _hip.call("wf_mg_relax_plan", C.byref(lev), nsweeps, out)
    return tuple(out)


# a block kernel whose planes must all exist never runs on a level of fewer, nor
# one for levels of few planes on a level of more
@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("tmp", [True, False])
def test_block_planes_fit_the_level(prec, tmp):
    blocks = 0
    for n0 in list(range(1, 41)) + [64, 80, 96]:
        for n1 in N:
            for n2 in N:
                for n in (1, 2, 3, 6, 7):
                    kind, launches, planes, part = plan((n0, n1, n2), prec, n, tmp)
                    assert launches >= 1
                    if kind == BLOCKS:
                        blocks += 1
                        assert (n0 <= planes) if part else (n0 >= planes), (n0, n1, n2, n)
    assert blocks


# small levels with an extent above 16 (one LDS launch takes every sweep) and
# levels of a few planes with many columns (blocks would be mostly halo) keep
# the launches that are faster there; blocks elsewhere
@pytest.mark.parametrize("n3,prec,nsweeps,kind", [
    ((4, 8, 64), 8, 300, LDS), ((2, 8, 24), 4, 300, LDS), ((20, 20, 20), 4, 300, LDS),
    ((24, 12, 32), 4, 300, BLOCKS), ((27, 27, 27), 8, 300, BLOCKS),
    ((2, 20, 6), 4, 6, LDS), ((1, 10, 20), 8, 6, LDS), ((24, 24, 24), 4, 6, BLOCKS),
    ((1, 1024, 1024), 4, 6, SWEEP), ((2, 512, 512), 8, 6, SWEEP), ((4, 512, 512), 4, 6, SWEEP),
    ((4, 512, 512), 8, 6, SWEEP), ((4, 256, 256), 4, 6, BLOCKS), ((8, 256, 256), 8, 6, BLOCKS),
    ((16, 256, 256), 4, 6, BLOCKS), ((512, 2, 512), 4, 6, BLOCKS), ((512, 512, 2), 8, 6, BLOCKS),
    ((12, 12, 12), 8, 300, BLOCKS), ((16, 16, 16), 4, 6, BLOCKS), ((32, 32, 32), 4, 300, BLOCKS),
    ((128, 128, 128), 4, 6, BLOCKS), ((80, 80, 80), 8, 6, BLOCKS)])
def test_faster_smoother_is_taken(n3, prec, nsweeps, kind):
    assert plan(n3, prec, nsweeps)[0] == kind


# planes whose offsets in a two-sweep chunk pass 2^30 bytes take one-sweep launches
@pytest.mark.parametrize("n3,prec,kind", [
    ((16, 5500, 5500), 4, SWEEP), ((16, 8000, 8000), 4, SWEEP), ((16, 5400, 5400), 4, SWEEP2),
    ((16, 3900, 3900), 8, SWEEP), ((16, 3800, 3800), 8, SWEEP2)])
def test_wide_planes_are_not_refused(n3, prec, kind):
    assert plan(n3, prec, 6)[0] == kind


# large levels of few planes or rows: a two-sweep chunk would be mostly the
# planes and rows around it
@pytest.mark.parametrize("n3,prec,kind", [
    ((4, 1056, 1056), 4, SWEEP), ((8, 744, 744), 4, SWEEP), ((12, 608, 608), 4, SWEEP2),
    ((1224, 8, 1224), 4, SWEEP), ((608, 12, 608), 4, SWEEP2), ((608, 608, 12), 4, SWEEP2),
    ((1496, 1496, 2), 4, SWEEP2), ((2, 1048, 1048), 8, SWEEP), ((8, 520, 520), 8, SWEEP),
    ((8, 1224, 1224), 8, SWEEP2), ((10, 464, 464), 8, SWEEP2), ((256, 256, 256), 4, SWEEP2),
    ((128, 128, 128), 8, SWEEP2)])
def test_large_flat_levels(n3, prec, kind):
    assert plan(n3, prec, 6)[0] == kind
