"""The first scan of a new map is cast once: its record set is guessed large enough (a set too small means a second cast)."""
import numpy as np
import pytest

import vdb_mapping_amd as V
from vdb_mapping_amd import workloads as W
from parity import same_map, pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scene,n,res,R", [("room", 2003, 0.1, 15.0), ("room", 32768, 0.1, 15.0), ("outdoor", 20000, 0.1, 35.0),
                                           ("outdoor", 65536, 0.1, 50.0), ("outdoor", 65536, 0.2, 50.0)])
def test_one_cast(scene, n, res, R):
    pose = W.trajectory(7, 1, 1.0, 5.0, 1.8)[0] if scene == "outdoor" else np.zeros(6)
    s = W.outdoor_scene(7, pose[None]) if scene == "outdoor" else W.room_scene(7)
    rings = 16 if n < 8192 else 32 if n < 65536 else 128
    elev = 22.5 if scene == "outdoor" else 15.0
    p = W.lidar_scan(s, pose, rings, (n + rings - 1) // rings, n, -elev, elev, 0.03, 7)
    g, o = pair(res, R, **W.PROBS)
    g.set_profiling(True)
    assert g.insert("test", p, pose[:3], check=True) == V.OK
    g.synchronize()
    assert g.stats()["n_walk"] == 1
    if n < 8192:
        assert o.insert("test", p, pose[:3]) == 0
        same_map(g, o)


def test_sets_that_hold_a_scan_stay():
    """The first scan's set is guessed larger than the ring's others. A scan that any of them holds makes none grow,
    also when it lies in the larger one; a scan that none holds does."""
    g, o = pair(0.1, 15.0, **W.PROBS)
    assert g.set_tuning(defer=1) == V.OK
    d = np.random.default_rng(3).normal(size=(20000, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    at = []
    for r in (10.0, 10.5, 14.5):  # a ball of about 9,200 leaves, 10,500, 26,000; sets are sized for a quarter more
        p = (d * r).astype(np.float32)
        for k in range(8):  # four sets in the ring
            assert g.insert("test", p, [0, 0, 0], check=True) == V.OK
            assert o.insert("test", p, [0, 0, 0]) == 0
        g.synchronize()
        at.append(g.stats()["scratch_bytes"])
    assert at[1] == at[0] and at[2] > at[1]
    same_map(g, o)
