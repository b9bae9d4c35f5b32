"""Fields and indices that the device holds in 4 bytes cross the bus in 4: single
copies and parts of 1 MB, across their edges, with every kind of value."""
import numpy as np
import pytest

from conftest import grasph as M

pytestmark = pytest.mark.gpu

PART = (1 << 20) // 4  # elements of a part


@pytest.mark.parametrize("n", [1, 5000, PART, PART + 1, 2 * PART, 2 * PART + 1, 3 * PART + 1])
def test_words_round_trip(n):
    rng = np.random.default_rng(n)
    ps = M.FluidParticleSystem("a", n, 2, 1.0, 1.0)
    sc = M.Session(2, "f32").scene
    want = {}
    for f in ("p", "drhodt", "dvdt", "rho"):
        a = getattr(ps, f)
        a[:] = rng.standard_normal(a.shape) * 10.0 ** rng.integers(-45, 39, a.shape)
        a.flat[: 4] = [np.inf, -0.0, np.nan, 1e300][: a.size]
        want[f] = a.copy()
    ps.id[:] = rng.permutation(n) + 1
    ids = ps.id.copy()
    sc.upload(ps)
    for f in want:
        getattr(ps, f)[:] = 0
    ps.id[:] = 0
    sc.download(ps)
    assert np.array_equal(ps.id, ids)
    with np.errstate(over="ignore"):
        for f, a in want.items():
            b = a if f == "rho" else a.astype(np.float32).astype(np.float64)
            assert np.array_equal(getattr(ps, f), b, equal_nan=True), f
            assert np.array_equal(np.signbit(getattr(ps, f)), np.signbit(b)), f
