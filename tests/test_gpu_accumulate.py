"""Accumulated updates through the brick path (a cloud's update leaves merged into its source's set) and their
integration (several sources as one group pass) against the oracle, bit for bit: merges into empty, partly filled and
growing sets, other paths in between, more sources than one group pass holds."""
import numpy as np
import pytest

import vdb_mapping_amd as V
from parity import both, pair, same_map, same_update

pytestmark = pytest.mark.gpu

PROBS = dict(prob_hit=0.7, prob_miss=0.4, prob_thres_min=0.12, prob_thres_max=0.97)


def cloud(n, seed, reach=6.0):
    rng = np.random.default_rng(seed)
    return rng.uniform(-reach, reach, (n, 3)).astype(np.float32)


@pytest.mark.parametrize("sizes", [[1, 300, 7000], [7000, 1, 300], [40, 40, 40], [20000, 20000, 20000]])
def test_merges(sizes):
    """A set that starts small and grows, and one that has room: every cloud OR-ed in, then the set used again."""
    g, o = pair(0.1, 8.0, **PROBS)
    for rep in range(2):
        for k, n in enumerate(sizes):
            both(g, o, "accumulate", "test", cloud(n, 10 * rep + k), [0.1 * k, 0.3, -0.2])
            if k != 1:
                same_update(g, o, "test")
        both(g, o, "integrate")
        same_map(g, o)
    assert g.stats()["rays"] == 2 * sum(sizes)


@pytest.mark.parametrize("n_sources", [2, 3, 8, 9, 17])
def test_sources_in_one_pass(n_sources):
    """Overlapping sets of several sources, each an update of its own in id order; some empty."""
    names = ["s%02d" % (n_sources - i) for i in range(n_sources)]
    g, o = pair(0.1, 8.0, sources=names, **PROBS)
    for rep in range(3):
        for i, s in enumerate(names):
            if (i + rep) % 4 == 3:
                continue
            for k in range(1 + i % 2):
                both(g, o, "accumulate", s, cloud(900 + 37 * i, 100 * rep + 10 * i + k), [0.05 * i, 0.1 * rep, 0.0])
        both(g, o, "integrate")
        same_map(g, o)


def test_other_paths_in_between():
    """Hash-traversal accumulates into the same set, inserts of another source, edits, resets and re-added sources."""
    g, o = pair(0.1, 8.0, sources=("a", "b"), **PROBS)
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
    assert g.add_input_source("a", 8.0) == o.add_input_source("a", 8.0)  # an empty set again
    both(g, o, "accumulate", "b", cloud(600, 9), [0, 0, 0])
    both(g, o, "integrate")
    same_map(g, o)


def test_artificial_areas_and_noop_probabilities():
    """Probabilities of 0.5 create no leaf (no group is opened for one); walls are activated once after the sources."""
    g, o = pair(0.1, 8.0, sources=("a", "b"), prob_hit=0.7, prob_miss=0.5, prob_thres_min=0.12, prob_thres_max=0.97)
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
    g, _ = pair(0.1, 8.0, **PROBS)
    bytes_at = []
    for k in range(6):
        assert g.accumulate("test", cloud(20000, k), [0, 0, 0]) == V.OK
        bytes_at.append(g.stats()["scratch_bytes"])
    leaves = len(g.export_update("test")[0])
    assert bytes_at[1] - bytes_at[0] <= 2 * 140 * leaves and bytes_at[5] - bytes_at[1] <= 2 * 140 * leaves
