"""Accumulated updates through the brick path (a cloud's update leaves merged into its source's set) and the hash
traversal, and their integration (several sources as one group pass) against the oracle, bit for bit: merges into empty,
partly filled and growing sets, other paths in between, more sources than one group pass holds. At 80 voxels of range
all clouds take the hash traversal, at 350 those of up to 4,900 and from 16,000 rays the brick path."""
import numpy as np
import pytest

import vdb_mapping_amd as V
from parity import both, pair, same_map, same_update

pytestmark = pytest.mark.gpu

PROBS = dict(prob_hit=0.7, prob_miss=0.4, prob_thres_min=0.12, prob_thres_max=0.97)


ranges = pytest.mark.parametrize("R", [8.0, 35.0])


def cloud(n, seed, reach=6.0):
    rng = np.random.default_rng(seed)
    return rng.uniform(-reach, reach, (n, 3)).astype(np.float32)


@ranges
@pytest.mark.parametrize("sizes", [[1, 300, 7000], [7000, 1, 300], [40, 40, 40], [20000, 20000, 20000]])
def test_merges(sizes, R):
    """A set that starts small and grows, and one that has room: every cloud OR-ed in, then the set used again."""
    g, o = pair(0.1, R, **PROBS)
    for rep in range(2):
        for k, n in enumerate(sizes):
            both(g, o, "accumulate", "test", cloud(n, 10 * rep + k), [0.1 * k, 0.3, -0.2])
            if k != 1:
                same_update(g, o, "test")
        both(g, o, "integrate")
        same_map(g, o)
    assert g.stats()["rays"] == 2 * sum(sizes)


@ranges
@pytest.mark.parametrize("n_sources", [2, 3, 8, 9, 17])
def test_sources_in_one_pass(n_sources, R):
    """Overlapping sets of several sources, each an update of its own in id order; some empty."""
    names = ["s%02d" % (n_sources - i) for i in range(n_sources)]
    g, o = pair(0.1, R, sources=names, **PROBS)
    for rep in range(3):
        for i, s in enumerate(names):
            if (i + rep) % 4 == 3:
                continue
            for k in range(1 + i % 2):
                both(g, o, "accumulate", s, cloud(900 + 37 * i, 100 * rep + 10 * i + k), [0.05 * i, 0.1 * rep, 0.0])
        both(g, o, "integrate")
        same_map(g, o)


@ranges
def test_other_paths_in_between(R):
    """Hash-traversal accumulates into the same set, inserts of another source, edits, resets and re-added sources."""
    g, o = pair(0.1, R, sources=("a", "b"), **PROBS)
    both(g, o, "accumulate", "a", cloud(4000, 1), [0, 0, 0.05])
    assert g.set_tuning(traversal=1) == V.OK
    both(g, o, "accumulate", "a", cloud(3000, 2), [0.2, 0, 0.05])
    same_update(g, o, "a")
    assert g.set_tuning(traversal=0) == V.OK
    both(g, o, "accumulate", "a", cloud(2500, 3), [0.4, 0, 0.05])
    same_update(g, o, "a")
    both(g, o, "insert", "b", cloud(1500, 4), [0.1, 0.1, 0.05])  # integrates both
    same_map(g, o)
    both(g, o, "accumulate", "b", cloud(500, 5), [0, 0, 0])
    both(g, o, "add_points_to_grid", cloud(50, 6))
    both(g, o, "integrate")
    same_map(g, o)
    both(g, o, "accumulate", "a", cloud(700, 7), [0, 0, 0])
    g.reset(), o.reset()
    both(g, o, "integrate")
    same_map(g, o)
    both(g, o, "accumulate", "a", cloud(700, 8), [0, 0, 0])
    assert g.add_input_source("a", R) == o.add_input_source("a", R)  # an empty set again
    both(g, o, "accumulate", "b", cloud(600, 9), [0, 0, 0])
    both(g, o, "integrate")
    same_map(g, o)


@ranges
def test_artificial_areas_and_noop_probabilities(R):
    """Probabilities of 0.5 create no leaf (no group is opened for one); walls are activated once after the sources."""
    g, o = pair(0.1, R, sources=("a", "b"), prob_hit=0.7, prob_miss=0.5, prob_thres_min=0.12, prob_thres_max=0.97)
    both(g, o, "add_artificial_areas", [[[-2, -2, 0], [2, -2, 0], [2, 2, 0]]], -0.2, 0.3)
    for rep in range(2):
        for k, s in enumerate("ab"):
            both(g, o, "accumulate", s, cloud(800, 20 + 2 * rep + k), [0.1 * k, 0, 0.05])
        both(g, o, "integrate")
        same_map(g, o)


def test_rejected_cloud_leaves_the_set():
    g, o = pair(0.1, 1e9, **PROBS)
    both(g, o, "accumulate", "test", cloud(500, 30), [0, 0, 0])
    far = np.array([[9e5, 0, 0]], np.float32)
    assert g.accumulate("test", far, [0, 0, 0]) == V.OUT_OF_RANGE
    same_update(g, o, "test")


def test_record_sets_stay_two():
    """A map that only accumulates takes two record sets, not the ring of deferred scans."""
    g, _ = pair(0.1, 35.0, **PROBS)
    bytes_at = []
    for k in range(6):
        assert g.accumulate("test", cloud(20000, k), [0, 0, 0]) == V.OK
        bytes_at.append(g.stats()["scratch_bytes"])
    leaves = len(g.export_update("test")[0])
    assert bytes_at[1] - bytes_at[0] <= 2 * 140 * leaves and bytes_at[5] - bytes_at[1] <= 2 * 140 * leaves


@pytest.mark.parametrize("vox,n,brick", [(100, 60000, False), (150, 63999, False), (150, 64000, True), (174, 2000, False),
                                         (175, 2450, True), (175, 2451, False), (250, 23039, False), (250, 23040, True),
                                         (400, 5600, True), (401, 5000, False), (400, 15999, False), (400, 16000, True),
                                         (1000, 16000, True), (1010, 16000, False), (2000, 64000, True)])
def test_path_of_a_cloud(vox, n, brick):
    """Which path a cloud takes by its rays and range (timed walks tell), both sides of the lines."""
    g, _ = pair(1.0, float(vox), **PROBS)
    g.set_profiling(True)
    assert g.accumulate("test", cloud(n, 1, 20.0), [0.5, 0.5, 0.5]) == V.OK
    g.synchronize()
    assert (g.stats()["n_walk"] > 0) == brick


@pytest.mark.parametrize("R,n", [(600.0, 17000), (390.0, 16000), (380.0, 5000)])
def test_many_bricks(R, n):
    """Clouds of more than 4,096 work items (their records lie in 16 regions of a set): overlapping ones into one
    source, then two sources integrated as one group."""
    g, o = pair(1.0, R, sources=("a", "b"), **PROBS)
    g.set_profiling(True)
    rng = np.random.default_rng(n)
    d = rng.normal(size=(3, n, 3))
    p = (d / np.linalg.norm(d, axis=2, keepdims=True) * rng.uniform(0.5 * R, 1.2 * R, (3, n, 1))).astype(np.float32)
    for k in range(2):
        both(g, o, "accumulate", "a", p[k], [0.5, 3.5 * k, -0.5])
    same_update(g, o, "a")
    both(g, o, "accumulate", "b", p[2], [0.5, 3.5, -0.5])
    both(g, o, "integrate")
    same_map(g, o)
    assert g.stats()["n_walk"] >= 3
