"""conv4th_u/v/w (tiles streamed along i) against extended-precision sums at tile
edges and remainders."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N = 3


def interp(f, ax):
    def at(s):
        return np.roll(f, -s, ax)
    return (-at(1) + 9 * at(0) + 9 * at(-1) - at(-2)) / 16


def advect(f, c, h):
    total = 0
    for ax in range(3):
        p, q = interp(f[c], ax), interp(f[ax], c)

        def s(m):
            if ax == c:
                return np.roll(p, -(m + 1), ax) ** 2
            return np.roll(p, -(m + 1), ax) * np.roll(np.roll(q, -1, c), -m, ax)
        total = total + (-s(1) + 27 * s(0) - 27 * s(-1) + s(-2)) / (24 * h[ax])
    return total


@pytest.mark.parametrize("n3", [(2, 2, 2), (3, 8, 32), (17, 9, 33), (33, 7, 31), (40, 24, 65)])
@pytest.mark.parametrize("c", [0, 1, 2])
def test_conv4th_tiles(n3, c):
    from warpflow import kernels as K
    from warpflow.device import array
    rng = np.random.default_rng(11)
    shape = tuple(n + 2 * N for n in n3)
    f = [rng.uniform(-1, 1, shape) for _ in range(3)]
    coo = rng.uniform(-1, 1, shape)
    h = tuple(a / n for a, n in zip((1.0, 1.1, 0.9), n3))
    star = array(np.full(shape, 7.0))
    dim = tuple(n - (a == c) for a, n in enumerate(n3))
    (K.conv4th_u, K.conv4th_v, K.conv4th_w)[c](dim, *map(array, f), array(coo), star, *h, 1e-3,
                                               1.0, N)
    want = coo - 1e-3 * advect([a.astype(np.longdouble) for a in f], c,
                               [np.longdouble(x) for x in h])
    box = tuple(slice(N, N + d) for d in dim)
    got = star.numpy()
    # an interpolant is at most 20/16, its product 1.57 with 10 roundings, a bracket
    # 56 of those with 4 more: 14 eps of 56 * 1.57 / (24 h) per axis, plus the sums
    eps = np.finfo(float).eps
    tol = 1e-3 * 16 * eps * sum(56 * 1.57 / (24 * x) for x in h) + 2 * eps
    assert np.max(np.abs(got[box] - want[box])) <= tol
    got[box] = 7.0
    assert np.all(got == 7.0)
