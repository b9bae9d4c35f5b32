"""Strain rate and vorticity of one target from several sources: a source whose
functor gives no vorticity adds none, whatever the source before it gave."""
import numpy as np
import pytest

from conftest import grasph as M, oracle_scene

pytestmark = pytest.mark.gpu

# of the largest: FP64 sums of ~30 terms; FP32 pair terms (a few roundings of
# 6e-8 each, cancelling by up to 1/100)
TOL = {"f64": 1e-11, "f32": 2e-5}
SRV, SR = M.StrainRateVorticityPfn, M.StrainRatePfn


def _body(name, x, h):
    D = x.shape[1]
    ps = M.ElastoPlasticParticleSystem(name, len(x), D, 4 if D == 2 else 6, 1000.0 * h ** D, 20.0,
                                       state_updater=M.ZeroFieldUpdater("strain_rate", "vorticity"))
    ps.x[:] = x
    ps.v[:] = np.random.default_rng(6).uniform(-0.3, 0.3, x.shape)
    ps.rho[:] = 1000.0
    return ps


def _scene(D, pfns, name="a"):
    """A body, a wall below it (mirrored velocities) and a second body on its
    side, each with a functor of its own."""
    rng = np.random.default_rng(5)
    dx = 0.02 if D == 2 else 0.05
    h = 1.3 * dx

    def block(shape, origin):
        g = np.stack(np.meshgrid(*[np.arange(k) + 0.5 for k in shape], indexing="ij"), -1)
        return (g.reshape(-1, D) + origin + rng.uniform(-0.2, 0.2, (np.prod(shape), D))) * dx

    side = 23 if D == 2 else 9
    a = _body(name, block((side,) * D, np.zeros(D)), h)
    below, beside = np.zeros(D), np.zeros(D)
    below[-1], beside[0] = -3.0, side
    w = M.BasicParticleSystem(name + "w", 3 * side ** (D - 1), D, 1000.0 * h ** D, 20.0)
    w.x[:] = block((side,) * (D - 1) + (3,), below)
    w.rho[:] = 1000.0
    b = _body(name + "b", block((4,) + (side,) * (D - 1), beside), h)
    up = np.zeros(D)
    up[-1] = 1.0
    kern = M.WenlandC2Kernel(h, ndims=D)
    wall = M.DynamicBoundarySystem(w, up, np.zeros(D), 2.5)
    ints = [M.SystemInteraction(kern, p(), *o)
            for p, o in zip(pfns, [(a,), (a, wall), (a, b)])]
    return a, M.LeapFrogTimeIntegrator([a, w, b], ints), h


ORDERS = [(SRV, SR, SR), (SR, SRV, SR), (SRV, SR, SRV), (SR, SR, SRV)]


def _ids(o):
    return "-".join("srv" if p is SRV else "sr" for p in o)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("order", ORDERS, ids=_ids)
def test_rates_equal_oracle(order, D, prec):
    got = []
    for scene in (M.Session(D, prec).scene, oracle_scene(D)):
        a, lf, _ = _scene(D, order)
        h = scene.integrator(lf)
        scene.upload_all(lf)
        scene.be.step(h, 2, 1e-7)
        scene.download_all(lf)
        o = np.argsort(a.id)
        got.append({f: getattr(a, f)[o].copy() for f in ("strain_rate", "vorticity")})
    for f, ref in got[1].items():
        assert np.any(ref), f
        assert np.max(np.abs(got[0][f] - ref)) <= TOL[prec] * np.max(np.abs(ref)), f


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("order", ORDERS[:2], ids=_ids)
def test_rates_equal_beside_a_large_companion(order, D, prec):
    """Four lanes per target alone, one beside a companion of 160000."""
    got = []
    for companion in (False, True):  # uploaded in both: the quantum of positions is shared
        a, lf, h = _scene(D, order)
        n = 160000
        big = _body("c", np.random.default_rng(3).uniform(0.0, 0.8 * h * n ** (1.0 / D), (n, D)), h)
        kern = M.WenlandC2Kernel(h, ndims=D)
        lfs = [lf, M.LeapFrogTimeIntegrator([big], [M.SystemInteraction(kern, SRV(), big)])]
        s = M.Session(D, prec)
        hs = [s.scene.integrator(f) for f in lfs]
        for k, f in zip(hs, lfs):
            s.scene.upload_all(f)
            s.backend.integrator_set_dt(k, 1e-7)
        s.backend.step_many(hs if companion else hs[:1], 2)
        s.scene.download_all(lf)
        got.append({f: getattr(a, f).copy() for f in ("strain_rate", "vorticity", "id")})
        s.close()
    for f in got[0]:
        assert np.array_equal(got[0][f], got[1][f]), f
