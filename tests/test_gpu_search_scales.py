"""The neighbour search in any unit of length: lengths whose squares are beyond
or below single precision's range give the oracle's partner counts, with one
and with four lanes per target."""
import numpy as np
import pytest

from conftest import grasph as M, oracle_scene

pytestmark = pytest.mark.gpu


def _cloud(x, h, name):
    D = x.shape[1]
    ps = M.FluidParticleSystem(name, len(x), D, 1e-3, 10.0, state_updater=M.TaitEOSUpdater(1000.0))
    ps.x[:] = x
    ps.rho[:] = 1000.0
    kern = M.WenlandC2Kernel(h, ndims=D)
    return ps, M.LeapFrogTimeIntegrator([ps], [M.SystemInteraction(kern, M.NeighborCounterPfn(), ps)])


def _points(D):
    """A cluster, and one so far off that a wavefront holds targets of both."""
    rng = np.random.default_rng(2)
    x = rng.uniform(0.0, 1.0, (900, D)) * (12.0 if D == 2 else 5.0)
    return np.concatenate([x, x[:30] + 40.0])


@pytest.mark.parametrize("prec", ["f64", "f32"])
# alone, or with a companion that takes the launch to each larger kernel (four
# lanes per target strip by strip, one lane)
@pytest.mark.parametrize("companion", [0, 1, 2])
@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("unit", [1e-40, 1e-22, 1e-19, 1e-17, 1e-14, 1e14, 1e17, 1e19, 1e22, 1e40])
def test_partner_counts(unit, D, companion, prec):
    got = []
    for sc in (M.Session(D, prec).scene, oracle_scene(D)):
        ps, lf = _cloud(_points(D) * unit, 0.5 * unit, "a")
        lfs = [lf]
        if companion and not got:
            n = (70000 if D == 2 else 60000) if companion == 1 else 140000
            y = np.random.default_rng(3).uniform(0.0, 0.4 * n ** (1.0 / D), (n, D))
            lfs.append(_cloud(y * unit, 0.5 * unit, "b")[1])
        hs = [sc.integrator(f) for f in lfs]
        for f in lfs:
            sc.upload_all(f)
        if not got:
            for k in hs:
                sc.be.integrator_set_dt(k, 1e-100)
            sc.be.step_many(hs, 1)
        else:
            sc.be.step(hs[0], 1, 1e-100)
        sc.download_all(lf)
        got.append(ps.drhodt[np.argsort(ps.id)])
    assert np.any(got[1])
    assert np.array_equal(*got)
