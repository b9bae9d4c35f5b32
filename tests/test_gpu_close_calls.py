"""Which candidates are neighbours is decided in FP32 but for the closest calls:
partner counts equal the oracle's where distances lie within a few units in
the last place of the cutoff, at large coordinates, and where one wavefront's
targets are far apart; with one and with four lanes per target."""
import numpy as np
import pytest

from conftest import grasph as M, oracle_scene

pytestmark = pytest.mark.gpu


def _lattice(D, base):
    dx, side = 0.01, 40 if D == 2 else 13
    g = np.stack(np.meshgrid(*[np.arange(side)] * D, indexing="ij"), -1).reshape(-1, D)
    rng = np.random.default_rng(2)
    x = base + 0.37 * dx + g * dx  # partners at 3 dx: the cutoff; none on a cell's edge
    return x + rng.integers(-3, 4, x.shape) * np.spacing(np.abs(x) + dx), dx


def _clusters(D):
    x, dx = _lattice(D, 0.0)
    # a wavefront's 16 or 64 consecutive sorted targets hold several
    far = 40.0 if D == 2 else 2.0
    return np.concatenate([x[:: 3], x[:7] + far, x[:50:9] - 0.1 * far]), dx


SCENES = {
    "origin": lambda D: _lattice(D, 0.0),
    "offset": lambda D: _lattice(D, 1234.5),
    "clusters": _clusters,
}


def _cloud(x, h, name):
    ps = M.FluidParticleSystem(name, len(x), x.shape[1], 1e-3, 10.0,
                               state_updater=M.TaitEOSUpdater(1000.0))
    ps.x[:] = x
    ps.rho[:] = 1000.0
    kern = M.WenlandC2Kernel(h, ndims=x.shape[1])
    return ps, M.LeapFrogTimeIntegrator([ps], [M.SystemInteraction(kern, M.NeighborCounterPfn(), ps)])


@pytest.mark.parametrize("prec", ["f32", "f64"])
# alone, or with a companion that takes the launch to each larger kernel (four
# lanes per target strip by strip, one lane)
@pytest.mark.parametrize("companion", [0, 1, 2])
@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("name", list(SCENES))
def test_partner_counts(name, D, companion, prec):
    x, dx = SCENES[name](D)
    h = 1.5 * dx
    got = []
    for sc in (M.Session(D, prec).scene, oracle_scene(D)):
        ps, lf = _cloud(x, h, "a")
        lfs = [lf]
        if companion and not got:
            n = (70000 if D == 2 else 60000) if companion == 1 else 140000
            y = np.random.default_rng(3).uniform(0.0, dx * n ** (1.0 / D), (n, D))
            lfs.append(_cloud(y, h, "b")[1])
        hs = [sc.integrator(f) for f in lfs]
        for f in lfs:
            sc.upload_all(f)
        if not got:
            for k in hs:
                sc.be.integrator_set_dt(k, 1e-30)
            sc.be.step_many(hs, 1)
        else:
            sc.be.step(hs[0], 1, 1e-30)
        sc.download_all(lf)
        got.append(ps.drhodt[np.argsort(ps.id)])
    assert np.array_equal(*got)
