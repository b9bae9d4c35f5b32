"""The cell sort of a step where a body has outgrown the table entries that its
plan gave it: within a call, before the plan is made anew, several cells share an
entry.  The order is the oracle's, bit for bit, the other bodies' too."""
import numpy as np
import pytest

from conftest import grasph as M, oracle_scene
from test_gpu_step_sort_dense import H

pytestmark = pytest.mark.gpu


def _body(name, x, v):
    ps = M.FluidParticleSystem(name, len(x), x.shape[1], 1e-3, 10.0,
                               state_updater=M.TaitEOSUpdater(1000.0))
    ps.x[:], ps.v[:] = x, v
    ps.rho[:] = 1000.0
    return ps


def _scene(D, n, speed, ghost):
    """A body that flies apart between two that do not, none moved by a functor."""
    rng = np.random.default_rng(4)

    def cloud(m):
        return rng.uniform(0.0, 1.0, (m, D))

    width = 0.2 * (n / 60.0) ** (1.0 / D)  # cells of some 60
    flying = rng.uniform(-1.0, 1.0, (n, D)) * speed * rng.uniform(0.0, 1.0, (n, 1)) ** 3
    ps = [_body("calm", cloud(1500), rng.uniform(-2.0, 2.0, (1500, D))),
          _body("flying", width * cloud(n), flying),
          _body("late", cloud(700), rng.uniform(-2.0, 2.0, (700, D))),
          _body("wall", -3.0 - 0.1 * cloud(5), 0.0)]
    ints = [M.SystemInteraction(M.WenlandC2Kernel(H, ndims=D), M.NeighborCounterPfn(), ps[-1])]
    e, entries = np.eye(D), ()
    if ghost:
        g = [M.GhostParticleSystem(q, M.GhostCopier("p")) for q in ps[:3]]
        entries = tuple(M.GhostEntry(q, 10 * H, (e[-1], np.zeros(D)), (e[0], np.zeros(D)))
                        for q in g)
    return ps, M.LeapFrogTimeIntegrator(ps, ints, ghosts=entries)


@pytest.mark.parametrize("steps", [3, 16, 35])  # within a chunk of steps, and over chunks
@pytest.mark.parametrize("ghost", [False, True], ids=["real", "ghost"])
@pytest.mark.parametrize("speed", [30.0, 400.0])  # entries of a few cells, of thousands
@pytest.mark.parametrize("D", [2, 3])
def test_order_in_flight(D, speed, ghost, steps):
    got = []
    for scene in (M.Session(D, "f64").scene, oracle_scene(D)):
        ps, lf = _scene(D, 2500, speed, ghost)
        h = scene.integrator(lf)
        scene.upload_all(lf)
        scene.be.step(h, 1, 1e-12)  # the plan
        scene.be.step(h, steps, 0.01)
        scene.download_all(lf)
        got.append([q.id.copy() for q in ps] + [q.x.copy() for q in ps] +
                   [g.ghost.idx_original.copy() for g in lf.ghosts])
    for u, v in zip(*got):
        assert len(v) and np.array_equal(u, v)


# 1024 workgroups of 256 particles find the next step's bounds at a step's end
@pytest.mark.parametrize("n", [2500, 265000])
@pytest.mark.parametrize("D", [2, 3])
def test_order_after_a_wide_upload(D, n):
    """A plan made for a compact body, and positions far wider uploaded into it."""
    got = []
    for scene in (M.Session(D, "f64").scene, oracle_scene(D)):
        ps, lf = _scene(D, n, 1.0, False)
        h = scene.integrator(lf)
        scene.upload_all(lf)
        scene.be.step(h, 1, 1e-9)
        scene.download_all(lf)
        out = []
        x = ps[1].x[np.argsort(ps[1].id)]
        for wider in (5.0, 0.6):
            ps[1].x[:] = np.random.default_rng(6).permutation(wider * x)[ps[1].id - 1]
            scene.upload(ps[1], ["x"])
            scene.be.step(h, 2, 1e-9)
            scene.download_all(lf)
            out += [q.id.copy() for q in ps]
        got.append(out)
    for u, v in zip(*got):
        assert np.array_equal(u, v)
