"""Targets whose neighbour list overflows, in launches with four lanes per
target: the quad walks the cells itself.  The partners and the order of every
sum are the list's, and so is every bit of the state."""
import numpy as np
import pytest

from conftest import grasph as M
from test_gpu_split import CASES, _disturb

pytestmark = pytest.mark.gpu


def _run(builder, kw, prec, maxnb):
    cfg = builder(**kw)
    _disturb(cfg)
    s = M.Session(cfg["integrator"].ndims, prec)
    s.backend.tune_set(M._abi.GR_TUNE_MAXNB, maxnb)
    h = s.scene.integrator(cfg["integrator"])
    s.scene.upload_all(cfg["integrator"])
    s.backend.integrator_set_dt(h, s.backend.integrator_dt(h, cfg["cfl"]))
    s.backend.step_many([h], 4)
    s.backend.set_timing(2)
    s.backend.step_many([h], 1)  # the counting kernels
    pairs = s.backend.get_pair_count(h)
    s.scene.download_all(cfg["integrator"])
    out = {(k, f): getattr(ps, f).copy() for k, ps in enumerate(cfg["integrator"].systems)
           for f in ps.field_names() + ["id"]}
    s.close()
    return out, pairs


@pytest.mark.parametrize("prec", ["f32", "f64"])
# every list overflows but those of a few entries / the lists of targets with
# several sources
@pytest.mark.parametrize("maxnb", [4, 9])
@pytest.mark.parametrize("name,builder,kw", [c[:3] for c in CASES], ids=[c[0] for c in CASES])
def test_walk_gives_the_lists_bits(name, builder, kw, maxnb, prec):
    listed, pairs = _run(builder, kw, prec, 0)
    walked, pairs_w = _run(builder, kw, prec, maxnb)
    assert pairs == pairs_w and pairs > 0
    for k, v in listed.items():
        assert np.array_equal(walked[k], v, equal_nan=True), k


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("D", [2, 3])
def test_dense_cells(D, prec):
    """Cells of more candidates than any list holds (the default one overflows),
    against the same cloud with lists that hold them."""
    got = []
    for maxnb in (0, 512):
        n = 3000
        x = np.random.default_rng(7).uniform(0.0, 0.3, (n, D))
        ps = M.FluidParticleSystem("a", n, D, 1e-3, 10.0, state_updater=M.TaitEOSUpdater(1000.0))
        ps.x[:] = x
        ps.v[:] = np.random.default_rng(8).uniform(-0.1, 0.1, x.shape)
        ps.rho[:] = 1000.0
        kern = M.WenlandC2Kernel(0.1, ndims=D)
        lf = M.LeapFrogTimeIntegrator([ps], [M.SystemInteraction(kern, M.FluidPfn(0.1, 0.0, 0.1), ps)])
        s = M.Session(D, prec)
        s.backend.tune_set(M._abi.GR_TUNE_MAXNB, maxnb)
        h = s.scene.integrator(lf)
        s.scene.upload_all(lf)
        s.backend.integrator_set_dt(h, 1e-6)
        s.backend.step_many([h], 2)
        s.scene.download_all(lf)
        got.append({f: getattr(ps, f).copy() for f in ps.field_names() + ["id"]})
        s.close()
    for f in got[0]:
        assert np.all(np.isfinite(got[0][f])), f
        assert np.array_equal(got[0][f], got[1][f]), f
