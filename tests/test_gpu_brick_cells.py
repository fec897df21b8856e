"""The brick tables of a scan (cells of the cube around the sensor up to a range of 1,597 voxels, hashed keys beyond)
and the size of its work items (256 segments up to 65,536 rays, 1,024 beyond) against the oracle, bit for bit. The
accumulated clouds beside them take the brick path at 200 voxels only (test_gpu_accumulate.py has the larger ones)."""
import numpy as np
import pytest

import vdb_mapping_amd as V
from parity import both, pair, same_map, same_update

pytestmark = pytest.mark.gpu

PROBS = dict(prob_hit=0.7, prob_miss=0.4, prob_thres_min=0.12, prob_thres_max=0.97)


def rays(n, R, org, seed):
    """Endpoints around `org`: the six axes at full range and truncated, then all directions and lengths."""
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(n, 3))
    p = d / np.linalg.norm(d, axis=1, keepdims=True) * rng.uniform(0, 1.3 * R, (n, 1))
    for k, f in enumerate([1.0, 3.0]):
        p[6 * k: 6 * k + 6] = np.concatenate([np.eye(3), -np.eye(3)]) * R * f
    p[12:14] = [[R, R, R], [-R, -R, -R]]
    return (p + org).astype(np.float32)


ORIGINS = [[0.5, 0.5, 0.5], [31.5, 32.0, -0.5], [-32.5, -4095.5, 4096.5]]


@pytest.mark.parametrize("R", [1.0, 29.0, 30.0, 31.0, 200.0, 1597.0, 1598.0, 1600.0, 3000.0])
@pytest.mark.parametrize("path", ["insert", "accumulate"])
def test_ranges(R, path):
    g, o = pair(1.0, R, **PROBS)
    for k, org in enumerate(ORIGINS):
        p = rays(250, R, org, int(R) + k)
        both(g, o, path, "test", p, org)
        if path == "accumulate":
            same_update(g, o, "test")
            both(g, o, "integrate")
    same_map(g, o)


def test_ranges_take_turns():
    """One map's sources on both sides of the line, inserted and accumulated, with the scratch memory given back."""
    names, R = ["near", "edge", "far"], [40.0, 1597.0, 1700.0]
    g, o = pair(1.0, 10.0, sources=names, source_ranges=R, **PROBS)
    for rep in range(3):
        for k, s in enumerate(names):
            org = ORIGINS[(rep + k) % 3]
            both(g, o, "insert" if (rep + k) % 2 else "accumulate", s, rays(300, R[k], org, 9 * rep + k), org)
        both(g, o, "integrate")
        if rep == 1:
            assert V.lib().vdbgpu_release_scratch(g.h) == V.OK
    same_map(g, o)


@pytest.mark.parametrize("n", [257, 1025, 65535, 65536, 65537])
def test_item_sizes(n):
    """Most rays through a few bricks: items of 256 and of 1,024 segments, split bricks on both sides of the line."""
    g, o = pair(1.0, 60.0, **PROBS)
    rng = np.random.default_rng(n)
    for k in range(2):
        p = rng.normal(0, 1, (n, 3)) * [4.0, 4.0, 4.0] + [40.0, 3.0 * k, -20.0]
        both(g, o, "insert", "test", p.astype(np.float32), [0.5, 0.5, 0.5 + k])
    same_map(g, o)
