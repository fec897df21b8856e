"""Map sections by the cells of their box against the oracle: boxes cut through leaves on every side, one voxel, one
leaf, around the 16 cells of a workgroup, at the ends of the coordinate range, larger than the map, more cells than
the path takes, staging that grows between calls (pinned chunks, the rest in device memory), and caps one too small."""
import numpy as np
import pytest

import vdb_mapping_amd as V
from parity import both, pair

pytestmark = pytest.mark.gpu

PROBS = dict(prob_hit=0.9, prob_miss=0.4, prob_thres_min=0.12, prob_thres_max=0.6)


@pytest.fixture(scope="module")
def maps():
    g, o = pair(0.1, 8.0, **PROBS)
    rng = np.random.default_rng(3)
    for k in range(3):
        both(g, o, "insert", "test", rng.uniform(-6, 6, (2500, 3)).astype(np.float32), [0.3 * k, 0.1, 0.2])
    return g, o


def same_section(g, o, box, full):
    a, b = g.export_section(box, full), o.export_section(box, full)
    assert a[0].shape == b[0].shape, (a[0].shape, b[0].shape)
    assert np.array_equal(a[0], b[0])
    assert np.array_equal(a[1].view(np.uint32), np.asarray(b[1]).view(np.uint32))
    assert np.array_equal(a[2], b[2])
    return len(a[0])


BOXES = [[0, 0, 0, 0, 0, 0], [0, 0, 0, 7, 7, 7], [-1, -1, -1, 0, 0, 0], [3, -5, 2, 11, 6, 9], [-8, -8, 0, 7, 23, 7],
         [-24, -8, 0, -1, 31, 7], [-8, -8, -8, 7, 7, 127], [-61, -63, -59, 60, 62, 58], [-200, -200, -200, 199, 199, 199],
         [5, 5, 5, 4, 9, 9], [-(1 << 23), 0, 0, -(1 << 23) + 40, 9, 9], [(1 << 23) - 9, 0, 0, (1 << 30), 9, 9],
         [-(1 << 30), -3, -3, 1 << 30, 3, 3], [-2000, -2000, -2000, 2000, 2000, 2000]]


@pytest.mark.parametrize("box", BOXES)
@pytest.mark.parametrize("full", [True, False])
def test_boxes(maps, box, full):
    same_section(*maps, box, full)


def test_staging_grows_and_caps(maps):
    g, o = maps
    g.synchronize()
    assert V.lib().vdbgpu_release_scratch(g.h) == V.OK
    n = [same_section(g, o, [-h, -h, -h, h, h, h], True) for h in (3, 20, 9, 60, 100)]
    assert n[0] < n[1] < n[3]
    box = np.array([-60] * 3 + [60] * 3, np.int32)
    v = np.full((n[3], 512), 7.0, np.float32)
    call = V.lib().vdbgpu_export_section
    assert call(g.h, box.ctypes.data, 1, None, v.ctypes.data, None, n[3] - 1) == -n[3]
    assert (v == 7.0).all()
    assert call(g.h, box.ctypes.data, 1, None, v.ctypes.data, None, n[3]) == n[3]
    assert np.array_equal(v, np.asarray(o.export_section(box, True)[1]))


def test_tiles_are_not_section_leaves():
    g, o = pair(0.1, 8.0, **PROBS)
    rng = np.random.default_rng(4)
    p = rng.uniform(-3, 3, (400, 3)).astype(np.float32)
    both(g, o, "create_map_from_points", p, True, True)
    for full in (True, False):
        same_section(g, o, [-30] * 3 + [30] * 3, full)


@pytest.mark.parametrize("sizes", [[255, 256, 257], [300, 300, 512, 513, 511], [4096, 4097, 4095, 1], [6000] * 20 + [100]])
def test_staging_chunks(sizes):
    """Sections around the 256 leaves of a pinned chunk and the 16 chunks of a map, read while the chunks still grow."""
    g, o = pair(1.0, 8.0, **PROBS)
    p = np.zeros((6000, 3), np.float32) + 0.5
    p[:, 0] += 8 * np.arange(6000)  # a row of leaves: a box of n cells holds n of them
    both(g, o, "add_points_to_grid", p)
    for k, n in enumerate(sizes):
        assert same_section(g, o, [0, 0, 0, 8 * n - 1, 7, 7], k % 3 != 1) == n
