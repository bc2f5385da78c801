"""Batched relaxation and V-cycle of members with small and flat levels: the bits of
the single-domain V-cycle, whichever launches the batch takes."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# one level (ncoarse sweeps, odd counts too) or more: members by the hundred, whose
# small levels relax in LDS, elongated and flat levels, members of unlike sizes
@pytest.mark.parametrize("shapes,nmem,nlev,sweeps", [
    ([(2, 16, 128)], 300, 1, (0, 0, 3)), ([(2, 16, 128)], 300, 1, (0, 0, 6)),
    ([(4, 8, 64)], 270, 1, (0, 0, 5)), ([(4, 8, 64)], 3, 1, (0, 0, 41)),
    ([(2, 24, 48), (6, 24, 24)], 130, 1, (0, 0, 7)), ([(24, 12, 12)], 5, 1, (0, 0, 6)),
    ([(4, 32, 256)], 40, 2, (3, 3, 5)), ([(4, 32, 256)], 3, 2, (6, 6, 8)),
    ([(16, 48, 32), (8, 16, 48)], 6, 3, (6, 4, 21)), ([(2, 256, 256)], 40, 1, (0, 0, 6))])
def test_batched_relaxation_equals_single(gpu, shapes, nmem, nlev, sweeps):
    from warpflow import _hip
    from warpflow.ensemble import Ensemble, MemberSpec
    from warpflow.multigrid import _Level
    specs = [MemberSpec(shapes[m % len(shapes)], 100.0, m + 1) for m in range(nmem)]
    ens = Ensemble(specs, 1e-4, mg_levels=nlev, sgs=False, graph=False)
    su = np.random.default_rng(4).standard_normal(ens.pool["su"].shape)
    ens.pool["su"].assign(su)
    npre, npost, nco = sweeps

    def solve(pre, post, coarse):
        return _hip.lib.wf_batch_mg_solve_mixed(
            ens.handle, ens._lptr["phi"], ens._lptr["rhs"], ens._lptr["tmp"], None,
            ens.pool["su"].ptr, ens.pool["pp"].ptr, 1, pre, post, coarse, 0, None, None)

    if nlev > 1 and npre % 2:  # odd counts are refused above 4096 cells a member
        assert solve(npre, npost, nco) == _hip.WF_EINVAL
        npre = npost = 6
    _hip.check(solve(npre, npost, nco), "wf_batch_mg_solve_mixed")
    _hip.call("wf_synchronize")
    phi = ens.lpool["phi"][0].numpy()
    for m in sorted({0, 1 % nmem, nmem - 1}):
        n3 = specs[m].n3
        levs = [_Level(tuple(n >> l for n in n3), tuple(2.0 ** l / n for n in n3), None,
                       np.float32) for l in range(nlev)]
        rhs = np.zeros(levs[0].shape)
        rhs[1:-1, 1:-1, 1:-1] = su[ens.field_off[m]:][:np.prod(ens.member_shape(m))].reshape(
            ens.member_shape(m))[3:-3, 3:-3, 3:-3]
        levs[0].rhs.assign(rhs)
        descs = (_hip.WfMgLevel * nlev)(*[lev.desc() for lev in levs])
        _hip.call("wf_mg_vcycle", descs, nlev, npre, npost, nco, None)
        want = levs[0].phi.numpy()
        off = ens.level_off[0][m]
        got = phi[off:off + want.size].reshape(want.shape)
        assert np.array_equal(got, want), m
    ens.close()
