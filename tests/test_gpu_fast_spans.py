"""The two launches of the fast-mode cast (span search, span walk) against the oracle, bit for bit: lists that outgrow
their first 1,024 spans per workgroup, more spans than one sort holds, one ray per wave, workgroups with no span.
(test_spans_per_workgroup stays within the lists' first length: its largest scan has 64 rays a workgroup.)"""
import numpy as np
import pytest

import vdb_mapping_amd as V
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


SPANS = 1024  # of a workgroup's list to start with, and of one sort of the walk
SPAN_BYTES = 24


def groups(n, num_cu=256):
    """(workgroups, rays of each) of a cast of n rays: up to 64 lanes a ray while the chip has room for them."""
    k = 0
    while k < 6 and n << (k + 1) <= num_cu * 1024:
        k += 1
    return min(num_cu * 16, ((n << k) + 255) // 256), 256 >> k


def through(n, R, seed, away=False):
    """n rays along the combs that end beyond the range, so that they fill none of the gaps."""
    rng = np.random.default_rng(seed)
    p = np.stack([np.full(n, 1.5 * R), rng.uniform(-4, 4, n), rng.uniform(-4, 4, n)], 1)
    return (p * [-1.0 if away else 1.0, 1, 1]).astype(np.float32)


@pytest.mark.parametrize("n,n_walls", [(140000, 6), (40000, 20), (140000, 17)])
def test_lists_that_outgrow(n, n_walls):
    """More than 1,024 spans a workgroup: the lists grow (a cast runs again), and a walk sorts them in several parts."""
    n_groups, rays = groups(n)
    assert rays * n_walls > SPANS
    factor = 4 if rays * n_walls <= 4 * SPANS else 16
    R = 12.0 * (n_walls + 2)
    g, o = pair(0.5, R, fast_mode=True, **PROBS)
    both(g, o, "add_points_to_grid", combs(n_walls, 12.0, 6.0))
    both(g, o, "integrate")
    both(g, o, "insert", "test", through(n, R, 1, away=True), [0.1, 0.2, -0.3])  # no span
    before = g.stats()["scratch_bytes"]
    both(g, o, "insert", "test", through(n, R, 2), [0.1, 0.2, -0.3])
    grown = g.stats()["scratch_bytes"] - before - n_groups * (factor - 1) * SPANS * SPAN_BYTES
    assert 0 <= grown < 1 << 20
    same_map(g, o)
    assert V.lib().vdbgpu_release_scratch(g.h) == V.OK
    both(g, o, "insert", "test", through(n, R, 3, away=True), [0.1, 0.2, -0.3])
    assert g.stats()["scratch_bytes"] <= before + (1 << 20)  # the lists start over


def test_accumulated_between_growths():
    """A cast that ran again with longer lists counts each ray once."""
    R, counts = 12.0 * 16, [200, 150000, 500]
    assert groups(counts[0])[1] * 14 <= SPANS < groups(counts[1])[1] * 14
    g, o = pair(0.5, R, fast_mode=True, **PROBS)
    both(g, o, "add_points_to_grid", combs(14, 12.0, 6.0))
    both(g, o, "integrate")
    for k, n in enumerate(counts):
        both(g, o, "accumulate", "test", through(n, R, k), [0.1, 0.2 * k, -0.3])
    both(g, o, "integrate")
    same_map(g, o)
    assert g.stats()["rays"] == sum(counts)
