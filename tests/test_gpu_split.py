"""Small launches run the neighbour search and the pair sweeps with four lanes
per target, large ones with one.  The choice goes by the size of the launch, so
a scene stepped alone takes the one and the same scene stepped with a large
companion the other: the lists and the order of every sum are the same, and so
must be every bit of the state."""
import numpy as np
import pytest

from conftest import grasph as M

pytestmark = pytest.mark.gpu

# (name, builder, size, companion's size): sizes that leave remainders in
# blocks of 64, 16 and 4 targets, and one of a single block
CASES = [
    ("dambreak2d", M.configs.dambreak_2d, dict(dx=0.037), dict(dx=0.004)),
    ("dambreak2d_block", M.configs.dambreak_2d, dict(dx=0.2), dict(dx=0.004)),
    ("dambreak3d", M.configs.dambreak_3d, dict(dx=0.041), dict(dx=0.0095)),
    ("ep_column2d", M.configs.ep_column_2d, dict(dx=0.005, width=0.115, height=0.075),
     dict(dx=0.002, width=0.8, height=0.7)),
    ("granular3d", M.configs.granular_column_3d,
     dict(dx=0.02, width=0.15, depth=0.07, height=0.09),
     dict(dx=0.005, width=0.4, depth=0.25, height=0.4)),
    ("bubble2d", M.configs.bubble_2d, dict(dx=0.17, variant="bubble3"),
     dict(dx=0.02, variant="bubble3")),
]


def _disturb(cfg):
    """Off the lattice, in motion: partner counts differ between targets."""
    rng = np.random.default_rng(11)
    for ps in cfg["integrator"].systems:
        if ps.source_v.any():
            dx = (ps.mass / ps.rho[0]) ** (1.0 / ps.ndims)
            ps.x += rng.uniform(-0.1, 0.1, ps.x.shape) * dx
            ps.v += rng.uniform(-0.1, 0.1, ps.v.shape)


def _run(builder, kw, prec, companion=None):
    cfg = builder(**kw)
    _disturb(cfg)
    cfgs = [cfg] + ([builder(**companion)] if companion else [])
    s = M.Session(cfg["integrator"].ndims, prec)
    hs = []
    for c in cfgs:
        h = s.scene.integrator(c["integrator"])
        s.scene.upload_all(c["integrator"])
        s.backend.integrator_set_dt(h, s.backend.integrator_dt(h, c["cfl"]))
        hs.append(h)
    s.backend.step_many(hs, 4)
    s.backend.set_timing(2)
    s.backend.step_many(hs[:1], 1)  # the counting kernels, alone in both runs
    pairs = s.backend.get_pair_count(hs[0])
    s.scene.download_all(cfg["integrator"])
    out = {(k, f): getattr(ps, f).copy() for k, ps in enumerate(cfg["integrator"].systems)
           for f in ps.field_names() + ["id"]}
    s.close()
    return out, pairs


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("name,builder,kw,big", CASES, ids=[c[0] for c in CASES])
def test_small_and_large_launches_give_the_same_bits(name, builder, kw, big, prec):
    alone, pairs = _run(builder, kw, prec)
    batch, pairs_b = _run(builder, kw, prec, big)
    assert pairs == pairs_b and pairs > 0
    for k, v in alone.items():
        assert np.array_equal(batch[k], v, equal_nan=True), k
