"""The active-point export (leaves listed and ordered on the device) against the oracle, bytes and order: leaf counts
around the 256 leaves of a workgroup's list tile, nodes and root children of both signs, tiles, inactive leaves."""
import ctypes

import numpy as np
import pytest

import vdb_mapping_amd as V
from parity import both, pair

pytestmark = pytest.mark.gpu

PROBS = dict(prob_hit=0.9, prob_miss=0.4, prob_thres_min=0.12, prob_thres_max=0.6)


def same_points(g, o):
    a, b = g.export_active_points(), o.export_active_points()
    assert a.shape == b.shape
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    return len(a)


def in_leaves(n_leaves, seed, spread):
    """A few points in each of n distinct leaves of a map with resolution 1."""
    rng = np.random.default_rng(seed)
    cells = rng.integers(-spread, spread, (4 * n_leaves + 64, 3))
    cells = np.unique(cells, axis=0)
    cells = cells[rng.permutation(len(cells))][:n_leaves]
    assert len(cells) == n_leaves
    return (cells[:, None, :] * 8 + rng.integers(0, 8, (n_leaves, 3, 3)) + 0.5).reshape(-1, 3).astype(np.float32)


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 511, 513, 5000, 20001])
@pytest.mark.parametrize("spread", [24, 900])  # inside the root children around the origin, and over many of them
def test_leaf_counts(n, spread):
    g, o = pair(1.0, 10.0, **PROBS)
    p = in_leaves(n, n + spread, spread)
    both(g, o, "add_points_to_grid", p)
    assert g.leaf_count() == n
    assert same_points(g, o) > 0
    both(g, o, "remove_points_from_grid", p[: 2 * (len(p) // 3)])  # two thirds of the leaves hold nothing active
    same_points(g, o)
    both(g, o, "add_points_to_grid", in_leaves(n, n + spread + 1, spread))  # appended leaves fall between the others
    same_points(g, o)


def test_tiles_and_an_empty_map():
    g, o = pair(1.0, 10.0, **PROBS)
    assert same_points(g, o) == 0
    b = np.stack(np.meshgrid(*[np.arange(-40, 40)] * 3, indexing="ij"), -1).reshape(-1, 3)
    pts = (np.concatenate([b, in_leaves(300, 3, 8) - 0.5]) + 0.5).astype(np.float32)
    both(g, o, "create_map_from_points", pts, True, False)
    assert len(g.export_tiles()[0]) >= 1000  # active ones inside the block, inactive ones around it
    assert same_points(g, o) > 1000
    both(g, o, "remove_points_from_grid", pts[:1000])  # some tiles become leaves again
    same_points(g, o)


@pytest.mark.parametrize("short", [1, 0])
def test_capacity(short):
    g, o = pair(1.0, 10.0, **PROBS)
    both(g, o, "add_points_to_grid", in_leaves(400, 9, 50))
    want = o.export_active_points()
    out = np.full((len(want) + 1, 3), -7.0, np.float32)
    got = V.lib().vdbgpu_export_active_points(g.h, out.ctypes.data_as(ctypes.c_void_p), len(want) - short)
    assert got == (-len(want) if short else len(want))
    assert np.all(out[-1] == -7.0) and (short or np.array_equal(out[:-1], want))


def test_more_leaves_than_are_ordered_on_the_device():
    """Above 2^19 leaves the host sorts: the same points in the same order."""
    n = (1 << 19) + 300
    g, o = pair(1.0, 10.0, **PROBS)
    i = np.random.default_rng(1).permutation(n)
    p = (np.stack([i % 83 - 40, i // 83 % 81 - 40, i // (83 * 81) - 35], 1) * 8 + 3.5).astype(np.float32)
    both(g, o, "add_points_to_grid", p)
    assert g.leaf_count() == n
    assert same_points(g, o) == n
    both(g, o, "remove_points_from_grid", p[:400])  # back below the line
    assert same_points(g, o) == n - 400
