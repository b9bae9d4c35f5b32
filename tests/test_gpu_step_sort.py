"""The cell sort of a step: counting by cell with the cells ordered by former
place, the radix sort's kernels where the key range has no table or the cells
hold more than 256 particles on average.  Both must give the oracle's order bit
for bit."""
import numpy as np
import pytest

from conftest import grasph as M, oracle_scene

pytestmark = pytest.mark.gpu


def _cloud(x, h, v=None):
    n, D = x.shape
    ps = M.FluidParticleSystem("cloud", n, D, 1e-3, 10.0, state_updater=M.TaitEOSUpdater(1000.0))
    ps.x[:] = x
    ps.rho[:] = 1000.0
    if v is not None:
        ps.v[:] = v
    kern = M.WenlandC2Kernel(h, ndims=D)
    return ps, M.LeapFrogTimeIntegrator([ps], [M.SystemInteraction(kern, M.FluidPfn(0.1, 0.0, h), ps)])


def _random(D, n, extent, seed=3):
    return np.random.default_rng(seed).uniform(0.0, 1.0, (n, D)) * extent


def _dense(D):
    x = _random(D, 3000, 4.0)
    x[::2] = 0.05 + 0.01 * x[::2]  # half of them in one cell of side 0.2
    return x


CASES = {
    "one": lambda D: _random(D, 1, 1.0),
    "block_edge": lambda D: _random(D, 257, 1.5),
    "shuffled": lambda D: _random(D, 20011, 6.0 if D == 2 else 3.0),
    # one cell of side 0.2 at the mean that takes the radix sort's kernels
    "one_cell": lambda D: 0.01 + 0.1 * _random(D, 256, 1.0),
    "one_cell_over": lambda D: 0.01 + 0.1 * _random(D, 257, 1.0),
    "dense": _dense,
    # keys of a table's tile edge and beyond: a row of 1023 / 1024 / 5000 cells
    "tile_row": lambda D: np.concatenate([0.2 * np.array([[1022.5] + [0.5] * (D - 1)]),
                                          _random(D, 400, 0.2)]),
    "tile_row1": lambda D: np.concatenate([0.2 * np.array([[1023.5] + [0.5] * (D - 1)]),
                                           _random(D, 400, 0.2)]),
    # two clusters far apart: more cells than a table is kept for
    "far": lambda D: np.concatenate([_random(D, 300, 1.0),
                                     _random(D, 300, 1.0) + (700.0 if D == 2 else 50.0)]),
}


@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("name", list(CASES))
def test_step_order_equals_oracle(name, D):
    x = CASES[name](D)
    # out of their cells from step to step
    v = np.random.default_rng(9).uniform(-1.0, 1.0, x.shape)
    got = []
    for scene in (M.Session(D, "f64").scene, oracle_scene(D)):
        ps, lf = _cloud(x, 0.1, v)
        h = scene.integrator(lf)
        scene.upload_all(lf)
        orders = []
        for _ in range(3):
            scene.be.step(h, 1, 1e-12)  # the forces move nothing, the velocities little
            scene.download_all(lf)
            orders.append(ps.id.copy())
            ps.x[:] += 0.07 * v[ps.id - 1]
            scene.upload(ps, ["x"])
        got.append(orders)
    for a, b in zip(*got):
        assert np.array_equal(a, b)


def test_many_systems_share_a_sort():
    """More systems than a workgroup finds the key bases for: an ensemble of 80
    columns in one call against each alone (whose bases are found inline)."""
    cfgs = [M.configs.ep_column_2d(dx=0.02, width=0.1 + 0.003 * k, height=0.08 + 0.002 * (k % 7),
                                   name=f"c{k}") for k in range(80)]
    alone = [M.configs.ep_column_2d(dx=0.02, width=0.1 + 0.003 * k, height=0.08 + 0.002 * (k % 7),
                                    name=f"a{k}") for k in range(0, 80, 13)]
    s = M.Session(2, "f64")
    hs = []
    for c in cfgs:
        c["fluid"].x[:] = c["fluid"].x[::-1]
        h = s.scene.integrator(c["integrator"])
        s.scene.upload_all(c["integrator"])
        s.backend.integrator_set_dt(h, s.backend.integrator_dt(h, c["cfl"]))
        hs.append(h)
    s.backend.step_many(hs, 5)
    for c in cfgs:
        s.scene.download_all(c["integrator"])
    for k, a in zip(range(0, 80, 13), alone):
        a["fluid"].x[:] = a["fluid"].x[::-1]
        s1 = M.Session(2, "f64")
        h = s1.scene.integrator(a["integrator"])
        s1.scene.upload_all(a["integrator"])
        s1.backend.integrator_set_dt(h, s1.backend.integrator_dt(h, a["cfl"]))
        s1.backend.step_many([h], 5)
        s1.scene.download_all(a["integrator"])
        for f in a["fluid"].field_names() + ["id"]:
            assert np.array_equal(getattr(a["fluid"], f), getattr(cfgs[k]["fluid"], f)), (k, f)


@pytest.mark.parametrize("dx", [0.02, 0.005, 0.0025])  # fluid / ghost keys: below a tile to five
def test_particles_and_ghosts_share_a_table(dx):
    """A scene whose ghosts' keys take another number of tiles than its
    particles': both sorts of a step use one table."""
    rng = np.random.default_rng(11)
    got = []
    cfgs = [M.configs.ep_column_2d(dx=dx, width=0.4, height=0.2, name=f"t{k}") for k in range(2)]
    n = cfgs[0]["fluid"].n
    moves = [rng.uniform(-0.2 * dx, 0.2 * dx, (n, 2)) for _ in range(3)]
    for scene, c in zip((M.Session(2, "f64").scene, oracle_scene(2)), cfgs):
        ps, lf = c["fluid"], c["integrator"]
        ps.x[:] = ps.x[::-1]
        h = scene.integrator(lf)
        scene.upload_all(lf)
        orders = []
        for m in moves:
            scene.be.step(h, 1, 1e-9)
            scene.download_all(lf)
            orders.append([ps.id.copy()] + [e.ghost.idx_original.copy() for e in lf.ghosts])
            ps.x[:] += m[ps.id - 1]
            scene.upload(ps, ["x"])
        got.append(orders)
    for a, b in zip(*got):
        for u, v in zip(a, b):
            assert np.array_equal(u, v)
