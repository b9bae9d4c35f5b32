"""The partner records of a stage: written by its updaters, and for ghosts
together with their kinematics and copies, where nothing comes in between."""
import numpy as np
import pytest

from conftest import grasph as M, oracle_scene

pytestmark = pytest.mark.gpu

# rates of one step against the oracle, of the largest: FP64 sums of ~30 terms;
# FP32 pair terms (a few roundings of 6e-8 each, cancelling by up to 1/100)
TOL = {"f64": 1e-11, "f32": 2e-5}


def _scene(kind, D):
    rng = np.random.default_rng(5)
    n, dx = (500, 0.02) if D == 2 else (1000, 0.05)
    h = 1.3 * dx
    side = int(round(n ** (1.0 / D)))
    g = np.stack(np.meshgrid(*[(np.arange(side) + 0.5) * dx] * D, indexing="ij"), -1)
    x = g.reshape(-1, D) + rng.uniform(-0.2, 0.2, (side ** D, D)) * dx
    pfns, copier = (M.FluidPfn(0.1, 0.05, h),), (M.GhostCopier("p"),)
    stress = kind in ("ep", "vpmc")
    if stress:
        ns = 4 if D == 2 else 6
        upd = {"ep": M.ElastoPlasticStressUpdater(1e6, 0.3, 0.5, 0.0, 10.0),
               "vpmc": M.ViscoPlasticMCStressUpdater(M.TaitEOSUpdater(1000.0), 0.5, 0.0)}[kind]
        ps = M.ElastoPlasticParticleSystem(
            "a", len(x), D, ns, 0.4, 20.0,
            state_updater=(M.ZeroFieldUpdater("strain_rate", "vorticity"), upd))
        ps.stress[:] = rng.uniform(-500.0, 500.0, ps.stress.shape)
        pfns = (M.StrainRateVorticityPfn(), M.CauchyFluidPfn(0.1, 0.0, h))
        copier = (None, M.GhostCopier(("stress", M.HouseholderReflect())))
    else:
        ps = M.FluidParticleSystem("a", len(x), D, 0.4, 20.0,
                                   state_updater=(M.TaitEOSUpdater(1000.0),))
        ps.p[:] = rng.uniform(-500.0, 500.0, ps.n)
    ps.x[:] = x
    ps.v[:] = rng.uniform(-0.3, 0.3, x.shape)
    ps.rho[:] = 1000.0 * (1.0 + rng.uniform(-0.01, 0.01, ps.n))
    ghost = M.GhostParticleSystem(ps, *copier)
    e = np.eye(D)
    entry = M.GhostEntry(ghost, 3 * h, (e[-1], np.zeros(D)), (e[0], np.zeros(D)))
    kern = M.WenlandC2Kernel(h, ndims=D)
    ints = [M.SystemInteraction(kern, pfns, ps), M.SystemInteraction(kern, pfns, ps, ghost)]
    if kind == "counter":
        ints.append(M.SystemInteraction(kern, M.NeighborCounterPfn(), ps, ghost))
    return ps, M.LeapFrogTimeIntegrator([ps], ints, ghosts=(entry,))


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind,D", [("eos", 2), ("eos", 3), ("counter", 2), ("counter", 3),
                                    ("ep", 2), ("vpmc", 2), ("vpmc", 3)])
def test_rates_of_a_step(kind, D, prec):
    got = []
    for scene in (M.Session(D, prec).scene, oracle_scene(D)):
        ps, lf = _scene(kind, D)
        h = scene.integrator(lf)
        scene.upload_all(lf)
        scene.be.step(h, 2, 1e-6)
        scene.download_all(lf)
        order = np.argsort(ps.id)
        got.append({f: getattr(ps, f)[order].copy()
                    for f in ("dvdt", "drhodt", "p", "stress") if hasattr(ps, f)})
    for f, ref in got[1].items():
        scale = max(np.max(np.abs(ref)), 1e-300)
        assert np.max(np.abs(got[0][f] - ref)) <= TOL[prec] * scale, f
