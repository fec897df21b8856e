"""The topology snapshot behind raytrace and fast mode (a bit per leaf under a hash of 128^3 nodes, extended by the
leaves appended since the last build): queries and fast-mode scans against the oracle after every way the snapshot
can change -- leaves in old and new nodes, more nodes than its first allocation, a reset, rays along node faces."""
import numpy as np
import pytest

import vdb_mapping_amd as V
from parity import both, pair, same_map

pytestmark = pytest.mark.gpu

PROBS = dict(prob_hit=0.9, prob_miss=0.4, prob_thres_min=0.12, prob_thres_max=0.6)


def fast_pair(res=0.5, R=60.0):
    return pair(res, R, fast_mode=True, **PROBS)


def same_queries(g, o, n, seed, half=40.0, length=50.0):
    rng = np.random.default_rng(seed)
    org = rng.uniform(-half, half, (n, 3))
    d = rng.normal(size=(n, 3))
    d[: n // 4, 0] = 0.0  # rays inside a plane of constant x,
    org[: n // 8, 0] = 64 * 0.5 * rng.integers(-1, 2, n // 8)  # half of them on a node face
    d[n // 4: n // 3, :2] = 0.0
    ln = rng.uniform(0.1, length, n)
    a, b = g.raytrace(org, d, ln), o.raytrace(org, d, ln)
    assert a[0] == b[0]
    assert np.array_equal(a[1].astype(bool), np.asarray(b[1]).astype(bool))
    assert np.array_equal(a[2].view(np.uint64), np.asarray(b[2], np.float64).view(np.uint64))
    return int(a[1].sum())


def scan(n, seed, reach):
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(n, 3))
    return (d / np.linalg.norm(d, axis=1, keepdims=True) * rng.uniform(0.2, reach, (n, 1))).astype(np.float32)


@pytest.mark.parametrize("leaves_per_scan", [30, 3000])
def test_snapshot_extends(leaves_per_scan):
    g, o = fast_pair()
    hits = 0
    for k, reach in enumerate([5.0, 20.0, 20.0, 55.0]):
        p = scan(leaves_per_scan, k, reach)
        for _ in range(2):
            both(g, o, "insert", "test", p, [0.1, 0.2 * k, -0.3])
        hits += same_queries(g, o, 800, 10 + k)
    same_map(g, o)
    assert hits > 0


def test_more_nodes_than_first_allocation():
    g, o = fast_pair(0.1, 400.0)
    rng = np.random.default_rng(5)
    for k, n in enumerate([40, 900]):  # one leaf per 128^3 node mostly: past the first 256 nodes
        p = rng.uniform(-150, 150, (n, 3)).astype(np.float32)
        both(g, o, "insert", "test", p, [3.1, 2.2, -4.3])
        same_queries(g, o, 500, 20 + k, half=100.0, length=200.0)
    assert g.leaf_count() > 600


def test_reset_and_rebuild():
    g, o = fast_pair()
    for k in range(2):
        p = scan(2000, 40 + k, 30.0)
        for _ in range(3):
            both(g, o, "insert", "test", p, [3.1, 2.2, -4.3])
        same_queries(g, o, 500, 50 + k)
        g.reset(), o.reset()
        same_queries(g, o, 100, 60 + k)  # the snapshot outlives the reset, the live map is empty
    q = scan(500, 70, 10.0)
    both(g, o, "insert", "test", q, [3.1, 2.2, -4.3])
    same_queries(g, o, 500, 71)


def test_edits_after_the_snapshot():
    """Voxels switched on after the build are seen in the leaves it knows, leaves created after it are not."""
    g, o = fast_pair()
    p = scan(3000, 80, 20.0)
    for _ in range(2):
        both(g, o, "insert", "test", p, [3.1, 2.2, -4.3])
    both(g, o, "add_points_to_grid", scan(300, 81, 35.0))
    both(g, o, "remove_points_from_grid", p[::2])
    same_queries(g, o, 1000, 82)
    both(g, o, "integrate")
    same_queries(g, o, 1000, 83)
    assert g.set_config(V.make_config(max_range=60.0, fast_mode=True, **PROBS)) == V.OK
