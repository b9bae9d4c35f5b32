"""Uploads and downloads in parts of 1 MB: what goes in comes out, across the
parts' edges, in both precisions."""
import numpy as np
import pytest

from conftest import grasph as M

pytestmark = pytest.mark.gpu

PART = (1 << 20) // 8  # elements of a part


@pytest.mark.parametrize("prec", ["f64", "f32"])
# one element; one, two and three parts of a scalar field and their edges; a
# part's edge within a vector field of 3 components
@pytest.mark.parametrize("n", [1, PART // 3, PART // 3 + 1, PART, PART + 1, 2 * PART + 1,
                               3 * PART - 1])
def test_fields_round_trip(n, prec):
    rng = np.random.default_rng(n)
    ps = M.ElastoPlasticParticleSystem("a", n, 3, 6, 1.0, 1.0)
    sc = M.Session(3, prec).scene
    want = {}
    for f in ps.field_names():
        a = getattr(ps, f)
        a[:] = rng.standard_normal(a.shape)
        want[f] = a.copy()
    ps.id[:] = rng.permutation(n) + 1
    want["id"] = ps.id.copy()
    sc.upload(ps)
    for f in want:
        getattr(ps, f)[:] = 0
    sc.download(ps)
    # held in FP32 by an FP32 session
    half = ("dvdt", "drhodt", "p", "strain_rate", "vorticity") if prec == "f32" else ()
    for f, a in want.items():
        b = a.astype(np.float32).astype(np.float64) if f in half else a
        assert np.array_equal(getattr(ps, f), b), f
