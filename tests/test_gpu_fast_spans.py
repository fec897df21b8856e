"""The two launches of the fast-mode cast (span search, span walk) against the oracle, bit for bit: lists that outgrow
their first 1,024 spans per workgroup, more spans than one sort holds, one ray per wave, workgroups with no span."""
import numpy as np
import pytest

from parity import both, pair, same_map

pytestmark = pytest.mark.gpu

PROBS = dict(prob_hit=0.9, prob_miss=0.4, prob_thres_min=0.12, prob_thres_max=0.6)


def combs(n_walls, gap, half):
    """Parallel walls across x, one voxel thick and `gap` metres apart: a ray along x meets a span per wall."""
    y, z = np.meshgrid(np.arange(-half, half, 0.45), np.arange(-half, half, 0.45), indexing="ij")
    one = np.stack([np.zeros(y.size), y.ravel(), z.ravel()], 1)
    return np.concatenate([one + [gap * (k + 1) + 0.25, 0, 0] for k in range(n_walls)]).astype(np.float32)


@pytest.mark.parametrize("n", [1, 63, 64, 300, 4097, 40000])
@pytest.mark.parametrize("n_walls", [3, 12])
def test_spans_per_workgroup(n, n_walls):
    R = 16.0 * n_walls
    g, o = pair(0.5, R, fast_mode=True, **PROBS)
    both(g, o, "add_points_to_grid", combs(n_walls, 12.0, 6.0))
    both(g, o, "integrate")  # the topology the casts look in
    rng = np.random.default_rng(n)
    for k in range(3):
        p = np.stack([rng.uniform(0.2, 1.2 * R, n), rng.uniform(-5, 5, n), rng.uniform(-5, 5, n)], 1)
        p[:: 11] *= [-1, 1, 1]  # away from the walls: no span
        p[5:: 13] = np.nan
        both(g, o, "insert", "test", p.astype(np.float32), [0.1, 0.2 * k, -0.3])
    same_map(g, o)


def test_accumulated_between_growths():
    """A cast that ran again with longer lists counts each ray once."""
    g, o = pair(0.5, 200.0, fast_mode=True, **PROBS)
    both(g, o, "add_points_to_grid", combs(14, 12.0, 6.0))
    both(g, o, "integrate")
    rng = np.random.default_rng(3)
    for k, n in enumerate([200, 30000, 500]):
        p = np.stack([np.full(n, 190.0), rng.uniform(-5, 5, n), rng.uniform(-5, 5, n)], 1).astype(np.float32)
        both(g, o, "accumulate", "test", p, [0.1, 0.2 * k, -0.3])
    both(g, o, "integrate")
    same_map(g, o)
    assert g.stats()["rays"] == 30700
