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
