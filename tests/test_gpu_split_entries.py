"""The sweeps with four lanes per target stage 24 list entries of a target and
the entry counts of 8 sources; beyond either the entries are loaded as they come
up.  Against the same scene stepped with a companion large enough for one lane
per target: every bit is the same."""
import numpy as np
import pytest

from conftest import grasph as M

pytestmark = pytest.mark.gpu


def _fluid(name, x, h, nwalls=0):
    D = x.shape[1]
    ps = M.FluidParticleSystem(name, len(x), D, 1000.0 * h ** D, 10.0,
                               state_updater=M.TaitEOSUpdater(1000.0))
    ps.x[:] = x
    ps.rho[:] = 1000.0
    ps.v[:] = np.random.default_rng(8).uniform(-0.1, 0.1, x.shape)
    kern, pfn = M.WenlandC2Kernel(h, ndims=D), M.FluidPfn(0.1, 0.0, h)
    ints, walls = [M.SystemInteraction(kern, pfn, ps)], []
    for k in range(nwalls):
        w = M.FluidParticleSystem(f"{name}w{k}", 40, D, 1000.0 * h ** D, 10.0)
        w.x[:] = np.random.default_rng(20 + k).uniform(0.0, 0.3, (40, D))
        w.rho[:] = 1000.0
        nrm = np.zeros(D)
        nrm[-1] = 1.0
        walls.append(w)
        ints.append(M.SystemInteraction(kern, pfn, ps,
                                        M.DynamicBoundarySystem(w, nrm, np.zeros(D) - 1.0, 2.5)))
    return ps, M.LeapFrogTimeIntegrator([ps] + walls, ints)


def _scene(name, D):
    rng = np.random.default_rng(4)
    if name == "entries":  # up to 9 strips (3 in 2D) of 3 cells of 70 (600) particles
        return _fluid("a", rng.uniform(0.0, 0.8, (4480 if D == 3 else 9600, D)), 0.1)
    return _fluid("a", rng.uniform(0.0, 0.3, (500, D)), 0.03 if D == 3 else 0.015,
                  {"sources8": 7, "sources9": 8, "sources11": 10}[name])


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("name", ["entries", "sources8", "sources9", "sources11"])
def test_beyond_what_is_staged(name, D, prec):
    got = []
    for companion in (False, True):  # uploaded in both: the quantum of positions is shared
        ps, lf = _scene(name, D)
        n = 160000
        y = np.random.default_rng(3).uniform(0.0, 0.02 * n ** (1.0 / D), (n, D))
        lfs = [lf, _fluid("b", y, 0.02)[1]]
        s = M.Session(D, prec)
        hs = [s.scene.integrator(f) for f in lfs]
        for h, f in zip(hs, lfs):
            s.scene.upload_all(f)
            s.backend.integrator_set_dt(h, 1e-7)
        s.backend.step_many(hs if companion else hs[:1], 2)
        s.scene.download_all(lf)
        got.append({f: getattr(ps, f).copy() for f in ps.field_names() + ["id"]})
        s.close()
    for f in got[0]:
        assert np.all(np.isfinite(got[0][f])), f
        assert np.array_equal(got[0][f], got[1][f]), f
