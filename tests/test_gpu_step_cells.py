"""The cell arrays a step builds (cleared by its sort, empty runs filled a tile
of 1024 cells at a time) equal the oracle's, entry for entry, step after step."""
import numpy as np
import pytest

from conftest import grasph as M, oracle_scene

pytestmark = pytest.mark.gpu

H = 0.1  # cells of side 0.2


def _random(D, n, extent, seed=3):
    return np.random.default_rng(seed).uniform(0.0, 1.0, (n, D)) * extent


def _lattice(D):
    # on the cells' edges, where rounding puts neighbours of a sort cell in
    # either of two grid cells
    g = np.stack(np.meshgrid(*[0.1 * np.arange(24 if D == 2 else 11)] * D, indexing="ij"), -1)
    return np.random.default_rng(4).permutation(g.reshape(-1, D))


CASES = {
    "one": lambda D: _random(D, 1, 1.0),
    "cloud": lambda D: _random(D, 5000, 3.0),
    "lattice": _lattice,
    # an empty run of about one tile, and one of more than 256 tiles
    "gap_tile": lambda D: np.concatenate([_random(D, 60, 0.4),
                                          _random(D, 60, 0.4) + (6.3 if D == 2 else 1.8)]),
    "gap_long": lambda D: np.concatenate([_random(D, 60, 0.4),
                                          _random(D, 60, 0.4) + (140.0 if D == 2 else 14.0)]),
}


@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("name", list(CASES))
def test_step_cells_equal_oracle(name, D):
    x = CASES[name](D)
    wall = _random(D, 300, 1.0, 7) - 0.5
    moves = np.random.default_rng(9).uniform(-0.08, 0.08, x.shape)
    got = []
    for scene in (M.Session(D, "f64").scene, oracle_scene(D)):
        ps = M.FluidParticleSystem("a", len(x), D, 1e-3, 10.0,
                                   state_updater=M.TaitEOSUpdater(1000.0))
        st = M.BasicParticleSystem("b", len(wall), D, 1e-3, 10.0)
        ps.x[:], st.x[:] = x, wall
        ps.rho[:] = 1000.0
        kern = M.WenlandC2Kernel(H, ndims=D)
        ints = [M.SystemInteraction(kern, M.NeighborCounterPfn(), ps),
                M.SystemInteraction(kern, M.NeighborCounterPfn(), ps, st)]
        lf = M.LeapFrogTimeIntegrator([ps, st], ints)
        h = scene.integrator(lf)
        scene.upload_all(lf)
        out = []
        for _ in range(3):
            scene.be.step(h, 1, 1e-12)
            scene.download_all(lf)
            for si in ints:
                hi = scene.interaction(si)
                ming, ng, ncells = scene.be.get_grid(hi, D)
                out.append([ming, ng, scene.be.get_cell_start(hi, 0, ncells + 1)])
            ps.x[:] += moves[ps.id - 1]
            scene.upload(ps, ["x"])
        got.append(out)
    for a, b in zip(*got):
        for u, v in zip(a, b):
            assert np.array_equal(u, v)


# one workgroup per 256 particles: 1024 of them take the next step's bounds as
# they advance the positions, more leave them to a pass of their own
@pytest.mark.parametrize("scheme", ["LeapFrogTimeIntegrator", "RK4TimeIntegrator"])
@pytest.mark.parametrize("n", [1, 257, 262144, 262145])
def test_bounds_follow_the_particles(n, scheme):
    """The box of a cloud that closes in on its centre, over steps of one call:
    the last step's cells and order are the oracle's."""
    x = _random(2, n, max(1.0, 0.02 * n ** 0.5))
    got = []
    for scene in (M.Session(2, "f64").scene, oracle_scene(2)):
        ps = M.FluidParticleSystem("a", n, 2, 1e-3, 10.0, state_updater=M.TaitEOSUpdater(1000.0))
        ps.x[:] = x
        ps.v[:] = 0.4 * (x.mean(axis=0) - x)
        ps.rho[:] = 1000.0
        si = M.SystemInteraction(M.WenlandC2Kernel(0.01, ndims=2), M.NeighborCounterPfn(), ps)
        lf = getattr(M, scheme)([ps], [si])
        h = scene.integrator(lf)
        scene.upload_all(lf)
        scene.be.step(h, 3, 0.25)
        scene.download_all(lf)
        hi = scene.interaction(si)
        ming, ng, ncells = scene.be.get_grid(hi, 2)
        got.append([ps.id.copy(), ps.x.copy(), ming, ng,
                    scene.be.get_cell_start(hi, 0, ncells + 1)])
    for u, v in zip(*got):
        assert np.array_equal(u, v)
