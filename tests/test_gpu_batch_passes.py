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


def _state(ens, names):
    ens.synchronize()
    out = {n: ens.pool[n].numpy() for n in names}
    out.update((n, getattr(ens, n).numpy()) for n in ("rmax", "active", "iters", "status"))
    return out


def _same(a, b):
    for n in a:
        assert np.array_equal(a[n], b[n], equal_nan=True), n


# a first test (every member takes part, whatever `active` held), a later one with
# members out of the loop, members that leave converged, diverged and as NaN
@pytest.mark.parametrize("sizes,levels", SIZES)
@pytest.mark.parametrize("it", [1, 2])
def test_project_test_is_projection_and_mask(sizes, levels, it):
    ens = _ensemble(sizes, levels)
    P, s, n = ens.pool, ens.stream, ens.nmem
    for m in range(n):  # rmax from below eps to above 10
        for c in ("ustar", "vstar", "wstar", "p"):
            f = ens.field(c, m)
            f.assign(f.numpy() * [1e-12, 1e-4, 1e3, 1.0][m % 4])
    if n > 3:
        f = ens.field("ustar", 3)
        a = f.numpy()
        a[5, 5, 5] = np.nan
        f.assign(a)
    start = {k: P[k].numpy() for k in ("u", "v", "w", "su")}
    live = np.array([m % 3 != 1 for m in range(n)], np.int32)
    names = ("u", "v", "w", "su")
    ptrs = [P[k].ptr for k in ("ustar", "vstar", "wstar", "p", "u", "v", "w", "su")]

    def begin(active):
        for k, v in start.items():
            P[k].assign(v)
        ens.rmax.fill_(0.5)
        ens.active.assign(active)
        ens.iters.assign(np.full(n, it - 1, np.int32))
        ens.status.assign(np.zeros(n, np.int32))
        ens.lpool["rhs"][0].fill_(-7.0)

    from warpflow import _hip
    begin(np.ones(n, np.int32) if it == 1 else live)
    ens._call("wf_batch_calvel3_calmas", *ptrs, ens.rmax.ptr, 1.0, ens.active.ptr, s)
    _hip.call("wf_batch_project_mask", ens.handle, ens.rmax.ptr, 1e-6, it, ens.active.ptr,
              ens.iters.ptr, ens.status.ptr, s)
    want = _state(ens, names)
    begin(live)
    ens._call("wf_batch_project_test", *ptrs, ens.lpool["rhs"][0].ptr, ens.rmax.ptr, 1.0, 1e-6,
              it, ens.active.ptr, ens.iters.ptr, ens.status.ptr, s)
    _same(want, _state(ens, names))
    rhs = ens.lpool["rhs"][0].numpy()
    for m in range(n):
        n3 = ens.specs[m].n3
        o = ens.level_off[0][m]
        r = rhs[o:o + int(np.prod([x + 2 for x in n3]))].reshape([x + 2 for x in n3])
        r = r[1:-1, 1:-1, 1:-1]
        if it == 1 or live[m]:
            su = ens.field("su", m).numpy()[3:-3, 3:-3, 3:-3]
            assert np.array_equal(r, su.astype(np.float32), equal_nan=True)
        else:
            assert np.all(r == -7.0)


@pytest.mark.parametrize("sizes,levels", SIZES)
@pytest.mark.parametrize("ncycles,flags", [(0, 2), (1, 2), (1, 0), (2, 2), (3, 2), (2, 0)])
def test_correct_is_solve_and_add(sizes, levels, ncycles, flags):
    ens = _ensemble(sizes, levels)
    P, s, n = ens.pool, ens.stream, ens.nmem
    live = np.array([m % 3 != 1 for m in range(n)], np.int32)
    ens.active.assign(live)
    p0, pp0 = P["p"].numpy(), np.zeros(P["pp"].shape)
    args = (ncycles, 2, 2, 8, flags, ens.active.ptr, s)
    lv = (ens._lptr["phi"], ens._lptr["rhs"], ens._lptr["tmp"], None)

    def rhs():  # (float)su on the real cells, as the projection leaves it
        r = ens.lpool["rhs"][0].numpy()
        for m in range(n):
            n3 = [x + 2 for x in ens.specs[m].n3]
            o = ens.level_off[0][m]
            v = r[o:o + int(np.prod(n3))].reshape(n3)
            v[1:-1, 1:-1, 1:-1] = ens.field("su", m).numpy()[3:-3, 3:-3, 3:-3]
        ens.lpool["rhs"][0].assign(r)

    P["pp"].assign(pp0)
    ens._call("wf_batch_mg_solve_mixed", *lv, P["su"].ptr, P["pp"].ptr, *args)
    ens._call("wf_batch_add_ring", P["p"].ptr, P["pp"].ptr, ens.active.ptr, s)
    want = _state(ens, ("p", "pp"))
    P["p"].assign(p0)
    for m in range(n):  # real cells, faces, edges and corners are all written
        a = np.zeros(ens.member_shape(m))
        a[2:-2, 2:-2, 2:-2] = 5.0
        ens.field("pp", m).assign(a)
    rhs()
    ens._call("wf_batch_mg_correct", *lv, P["su"].ptr, P["pp"].ptr, P["p"].ptr, *args)
    _same(want, _state(ens, ("p", "pp")))
