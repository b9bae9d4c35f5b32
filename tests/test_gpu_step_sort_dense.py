"""The cell sort of a step where cells hold many particles (their order is taken
from the runs of former neighbours): the oracle's order, bit for bit."""
import numpy as np
import pytest

from conftest import grasph as M, oracle_scene

pytestmark = pytest.mark.gpu

H = 0.1  # cells of side 0.2


def _scene(x, ghost=False):
    """A body that no functor moves, beside a wall far off."""
    n, D = x.shape
    a = M.FluidParticleSystem("a", n, D, 1e-3, 10.0, state_updater=M.TaitEOSUpdater(1000.0))
    w = M.FluidParticleSystem("w", 5, D, 1e-3, 10.0, state_updater=M.TaitEOSUpdater(1000.0))
    a.x[:] = x
    w.x[:] = -3.0 - 0.1 * np.random.default_rng(1).uniform(0.0, 1.0, (5, D))
    a.rho[:] = w.rho[:] = 1000.0
    kern = M.WenlandC2Kernel(H, ndims=D)
    ints = [M.SystemInteraction(kern, M.NeighborCounterPfn(), w)]
    if not ghost:
        return a, M.LeapFrogTimeIntegrator([a, w], ints)
    e = np.eye(D)
    g = M.GhostParticleSystem(a, M.GhostCopier("p"))
    entry = M.GhostEntry(g, 3 * H, (e[-1], np.zeros(D)), (e[0], np.zeros(D)))
    return a, M.LeapFrogTimeIntegrator([a, w], ints, ghosts=(entry,))


def _cell(D, n, rng, at=0):
    return 0.2 * (np.arange(D) == 0) * at + 0.005 + 0.19 * rng.uniform(0.0, 1.0, (n, D))


def _cells(D, counts):
    """Cells of these counts in a row, and a sparse cloud around them."""
    rng = np.random.default_rng(3)
    return np.concatenate([_cell(D, k, rng, at) for at, k in enumerate(counts)] +
                          [rng.uniform(0.0, 4.0, (300, D))])


CASES = {
    # the largest cell compared particle by particle, and the next
    "edge": [240, 250, 255, 256, 257, 270],
    "one": [3000],
    # runs of several wavefronts and workgroups of former neighbours
    "long": [9000, 1, 700, 64, 0, 2000],
}


@pytest.mark.parametrize("ghost", [False, True], ids=["real", "ghost"])
@pytest.mark.parametrize("shuffle", [False, True], ids=["ordered", "shuffled"])
@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("name", list(CASES))
def test_order_equals_oracle(name, D, shuffle, ghost):
    x = _cells(D, CASES[name])
    if shuffle:
        x = np.random.default_rng(5).permutation(x)
    # a few leave their cells from step to step
    move = np.random.default_rng(9).uniform(-0.3, 0.3, x.shape)
    move[np.random.default_rng(8).uniform(size=len(x)) > 0.05] = 0.0
    got = []
    for scene in (M.Session(D, "f64").scene, oracle_scene(D)):
        a, lf = _scene(x, ghost)
        h = scene.integrator(lf)
        scene.upload_all(lf)
        out = []
        for _ in range(3):
            scene.be.step(h, 1, 1e-12)
            scene.download_all(lf)
            out.append([a.id.copy()] + [e.ghost.idx_original.copy() for e in lf.ghosts])
            a.x[:] = np.abs(a.x + move[a.id - 1])
            scene.upload(a, ["x"])
        got.append(out)
    for p, q in zip(*got):
        for u, v in zip(p, q):
            assert len(v) and np.array_equal(u, v)
