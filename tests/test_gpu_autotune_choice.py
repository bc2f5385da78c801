"""The tuner leaves a level to the built-in smoother exactly where that timed no
slower per sweep than the best launch shape: times are planted, the launches and
the checks of their results run."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class PlantedTimes:
    """us() of the tuner's timer: 10 us a sweep for every tuned shape."""

    def __init__(self, builtin_per_sweep):
        self.times = {"relax": 20.0, "relax4": 40.0, "relax12": 12.0 * builtin_per_sweep}

    def us(self, fn, reps):
        fn()
        return self.times.get(fn.__name__, 0.0)  # copies: nothing


@pytest.mark.parametrize("prec", [np.float64, np.float32])
@pytest.mark.parametrize("per_sweep,left", [(9.0, True), (10.0, True), (11.0, False)])
def test_level_is_left_to_the_builtin_smoother(gpu, prec, per_sweep, left):
    from warpflow import autotune
    from warpflow.multigrid import _Level
    n3 = (20, 24, 36)
    lev = _Level(n3, tuple(1.0 / n for n in n3), None, prec)
    rng = np.random.default_rng(3)
    lev.rhs.assign(rng.standard_normal(lev.shape))
    out = {"entries": [], "timings_us": {}}
    autotune.reset()
    try:
        autotune._tune_level(lev, PlantedTimes(per_sweep), 1, out)
        f64 = prec == np.float64
        knobs = [getattr(autotune, k + ("F64" if f64 else "F32"))
                 for k in ("SWEEP_TILE_", "SWEEP_ICH_", "SWEEP_PAIRS_", "SWEEP2_TILE_",
                           "SWEEP2_ICH_")]
        values = [autotune.get_shape(k, n3) for k in knobs]
        if left:
            assert not out["entries"] and not any(values)
        else:  # a tile (never 0) and the kind of launch are set
            assert out["entries"] and values[0] and values[2]
            assert all(autotune.get_shape(k, n) == v for k, n, v in out["entries"])
    finally:
        autotune.reset()
