"""Scan sizes around the tiles of the per-scan kernels: 256 rays per prep workgroup (its sums carry visits and
valid rays in one word), 1,024 records per append of the map insert and the group set-up, 2,048 update-set slots
per append of the listing. Map, update set and counters against the oracle, bit for bit."""
import numpy as np
import pytest

import vdb_mapping_amd as V
from parity import pair, same_map, same_update

pytestmark = pytest.mark.gpu

PROBS = dict(prob_hit=0.7, prob_miss=0.4, prob_thres_min=0.12, prob_thres_max=0.97)


def cloud(n, seed, nan_every=7):
    rng = np.random.default_rng(seed)
    p = rng.uniform(-8, 8, (n, 3)).astype(np.float32)
    p[::nan_every, 1] = np.nan
    return p


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 511, 1024, 3071, 4097, 20001])
@pytest.mark.parametrize("path", ["insert", "accumulate"])
def test_sizes_around_tiles(n, path):
    g, o = pair(0.1, 6.0, **PROBS)
    rays = leaves = 0
    for k in range(3):
        p, org = cloud(n, 10 * n + k), [0.05 + 0.3 * k, -0.2, 0.1 * k]
        rays += int((~np.isnan(p).any(1)).sum())
        o.accumulate("test", p, org)
        leaves += len(o.export_update("test")[0])
        if path == "insert":
            g.insert("test", p, org, check=True)
        else:
            g.accumulate("test", p, org, check=True)
            same_update(g, o, "test")
            g.integrate(check=True)
        o.integrate()
    same_map(g, o)
    st = g.stats()
    assert st["rays"] == rays and st["update_leaves"] == leaves


def test_no_valid_ray():
    g, o = pair(0.1, 6.0, **PROBS)
    p = np.full((700, 3), np.nan, np.float32)
    assert g.insert("test", p, [0, 0, 0]) == V.OK
    assert g.stats()["rays"] == 0 and g.leaf_count() == 0
