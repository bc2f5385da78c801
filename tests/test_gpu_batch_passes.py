"""The ensemble's fused passes against the passes they replace, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# ragged tiles, one-tile members, more than one chunk, many members
SIZES = [
    ([(8, 8, 8)], 1),
    ([(24, 40, 56), (32, 8, 16), (48, 24, 40)], 3),
    ([(96, 20, 36), (4, 68, 100)], 2),
    ([(16, 8 * (1 + m % 5), 8 * (1 + m % 9)) for m in range(40)], 2),
]


def _ensemble(sizes, levels, seed=3):
    from warpflow.ensemble import Ensemble, MemberSpec
    ens = Ensemble([MemberSpec(n, 200.0 + 50.0 * m, m + 1, 0.02) for m, n in enumerate(sizes)],
                   dt=1e-3, mg_levels=levels, graph=False)
    rng = np.random.default_rng(seed)
    for name, pool in ens.pool.items():
        pool.assign(rng.standard_normal(pool.shape) * (0.1 if name != "vis" else 1e-3))
    return ens


@pytest.mark.parametrize("sizes,levels", SIZES)
def test_wale_checkdt_is_the_two_passes(sizes, levels):
    ens = _ensemble(sizes, levels)
    P, s = ens.pool, ens.stream
    vis = np.abs(P["vis"].numpy()) + 1e-3
    P["vis"].assign(vis)
    vel = (P["u"].ptr, P["v"].ptr, P["w"].ptr, P["vis"].ptr)
    ens._call("wf_batch_checkdt", *vel, ens.out4.ptr, s)
    ens._call("wf_batch_wale", *vel, s)
    ens.synchronize()
    want = P["vis"].numpy(), ens.out4.numpy()
    P["vis"].assign(vis)
    ens.out4.fill_(-1.0)
    ens._call("wf_batch_wale_checkdt", *vel, ens.out4.ptr, s)
    ens.synchronize()
    assert np.array_equal(P["vis"].numpy(), want[0])
    assert np.array_equal(ens.out4.numpy(), want[1])
