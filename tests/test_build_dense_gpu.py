"""The dense build of small grids (a table of one word per voxel instead of
the sort) against the oracle's arrays: every edge that takes it, both sides of
the rule that chooses it, edits, many records of one voxel, solid grids, grids
of one voxel, and deletions that leave nothing."""
import numpy as np
import pytest

import oracle_py as O
from scenes import random_points, scene_grid, grid_to_points
from test_build_gpu import assert_same_build

pytestmark = pytest.mark.gpu


def _build(log2, pts, dense=True, old=None, **kw):
    from pyrit_amd import gpu as g

    g.set_timing(True)
    try:
        b = g.build(log2, pts, old=old, **kw)
        finish = g.last_build_times()["finish"]
    finally:
        g.set_timing(False)
    assert (finish == 0) == dense, finish
    return b


@pytest.mark.parametrize("log2", [3, 4, 5, 6, 7])
@pytest.mark.parametrize("fill", ["rule", "full", "few"])
def test_random_grids(hip_device, log2, fill):
    cells = 8 ** log2
    n = {"rule": max(2, cells // 16 + 1), "full": min(cells, 1 << 21), "few": 37}[fill]
    pts = random_points(n, log2, seed=log2 * 7, dup_frac=0.25, delete_frac=0.05, out_frac=0.03)
    b = _build(log2, pts, dense=cells <= 1 << 18 or 16 * len(pts) >= cells)
    assert_same_build(b, O.gb_build(log2, pts), log2)


def test_rule_edge(hip_device):
    for count, dense in ((8 ** 7 // 16 - 1, False), (8 ** 7 // 16, True)):
        pts = random_points(count, 7, seed=3, dup_frac=0.0)
        assert_same_build(_build(7, pts, dense), O.gb_build(7, pts), 7)
    cube = random_points(1 << 21, 8, seed=4, dup_frac=0.0)  # an edge of 2^8 never takes it
    assert_same_build(_build(8, cube, False), O.gb_build(8, cube), 8)
    # a named setting gets its own path, the default value of one does not change anything
    pts = random_points(5000, 5, seed=9)
    ref = O.gb_build(5, pts)
    assert_same_build(_build(5, pts, False, finish=1), ref, 5)
    assert_same_build(_build(5, pts, False, sort_items=8), ref, 5)
    assert_same_build(_build(5, pts, True, sort_items=20), ref, 5)


def test_many_records_are_sorted(hip_device):
    """The last record count of a 2^7 grid that the table takes, and one more
    (a record outside the grid): the same voxels, by the table and sorted."""
    from pyrit_amd import abi

    count = 1 << 24
    pts = np.zeros(count + 1, abi.VOXEL)
    rng = np.random.default_rng(24)
    i = np.arange(count) // 8  # in voxel order, eight records each
    pts["x"][1:], pts["y"][1:], pts["z"][1:] = i % 128, i // 128 % 128, i // 16384
    pts["attribute"][1:] = rng.integers(0, 5, count)
    pts["x"][0], pts["attribute"][0] = -1, 7
    a, b = _build(7, pts[1:], True), _build(7, pts, False)
    # the last record of a voxel wins; attribute 0 removes it
    assert a.voxel_count == np.count_nonzero(pts["attribute"][8::8])
    for what in ("nodes", "leaves", "keys", "attrs"):
        assert np.array_equal(getattr(a, what)(), getattr(b, what)()), what
    assert a.root == b.root


@pytest.mark.parametrize("log2,edits", [(3, 1), (5, 700), (6, 4096), (7, 311)])
def test_edits(hip_device, log2, edits):
    from pyrit_amd import gpu as g

    size = 1 << log2
    rng = np.random.default_rng(log2)
    z, y, x = np.nonzero(rng.random((size, size, size)) < 0.3)
    pts = np.zeros(len(x), O.VOXEL)
    pts["x"], pts["y"], pts["z"], pts["attribute"] = x, y, z, rng.integers(1, 9, len(x))
    old = g.build(log2, pts)
    ed = random_points(edits, log2, seed=5, dup_frac=0.5, delete_frac=0.3, out_frac=0.1)
    b = _build(log2, ed, old=old)
    ref0 = O.gb_build(log2, pts)
    assert_same_build(b, O.gb_build(log2, ed, ref0["keys"], ref0["attrs"]), log2)
    # everything removed
    gone = pts.copy()
    gone["attribute"] = 0
    e = _build(log2, gone, old=old)
    assert e.voxel_count == 0 and e.nodes().tolist() == [0, 0] and e.root == 0 and e.leaf_count == 0


def test_one_voxel_many_records(hip_device):
    for log2 in (3, 6, 7):
        pts = np.zeros(1 << 18, O.VOXEL)
        pts["x"], pts["y"], pts["z"] = 5, 3, 6
        pts["attribute"] = np.arange(1, len(pts) + 1)
        pts["x"][::1000] = 2
        assert_same_build(_build(log2, pts), O.gb_build(log2, pts), log2)
        last = pts.copy()
        last["attribute"][-1] = 0
        assert_same_build(_build(log2, last), O.gb_build(log2, last), log2)


@pytest.mark.parametrize("log2", [3, 5, 6, 7])
def test_solid_and_corners(hip_device, log2):
    n = 1 << log2
    edge = min(n, 128)
    solid = np.zeros(edge ** 3, O.VOXEL)
    i = np.arange(edge ** 3)
    solid["x"], solid["y"], solid["z"], solid["attribute"] = i % edge, i // edge % edge, i // edge // edge, 1 + i % 7
    assert_same_build(_build(log2, solid), O.gb_build(log2, solid), log2)
    if log2 <= 6:
        corners = np.array([(0, 0, 0, 1), (n - 1, n - 1, n - 1, 2), (n, 0, 0, 3), (0, -1, 0, 4), (2 ** 31 - 1, 0, 0, 5),
                            (0, 0, -2 ** 31, 6)], O.VOXEL)
        assert_same_build(_build(log2, corners), O.gb_build(log2, corners), log2)
        for c in corners[:2]:
            one = np.array([c], O.VOXEL)
            assert_same_build(_build(log2, one), O.gb_build(log2, one), log2)


def test_scene_and_reuse(hip_device):
    # builds of different sizes one after another reuse the cached memory
    for log2 in (7, 5, 7, 6, 3):
        pts = grid_to_points(scene_grid(1 << log2))
        np.random.default_rng(log2).shuffle(pts)
        assert_same_build(_build(log2, pts, dense=8 ** log2 <= 1 << 18 or 16 * len(pts) >= 8 ** log2),
                          O.gb_build(log2, pts), log2)


@pytest.mark.parametrize("log2,count,mixed", [(3, 1, False), (6, 1, True), (5, 3, True), (8, 3, True), (7, 65, True),
                                              (8, 64, True), (4, 513, True), (3, 4096, False), (3, 4097, False),
                                              (9, 5, False)])
def test_batch_levels(hip_device, log2, count, mixed):
    """Batches whose upper levels are dense, from all levels to none: chunks
    that end on every level, empty chunks, and counts around the last kernel's
    cells."""
    from pyrit_amd import gpu as g

    rng = np.random.default_rng(count)
    l2 = rng.integers(3, log2 + 1, count).astype(np.uint8) if mixed else None
    chunks = []
    for c in range(count):
        edge = int(l2[c]) if mixed else log2
        n = 0 if c % 7 == 3 else int(rng.integers(1, min(8 ** edge, 200000 // count + 40)))
        chunks.append(random_points(n, edge, int(rng.integers(1 << 30)), dup_frac=0.1, delete_frac=0.02) if n else
                      np.zeros(0, O.VOXEL))
    offs = np.concatenate([[0], np.cumsum([len(c) for c in chunks])]).astype(np.uint32)
    vox = np.concatenate(chunks)
    ref, rroots, rfirst = O.gb_build_chunks(log2, vox, offs, l2)
    for levels in (0, 1, 2):
        b, roots, first = g.build_chunks(log2, vox, offs, l2, levels=levels)
        assert_same_build(b, ref, log2)
        assert np.array_equal(roots, rroots) and np.array_equal(first, rfirst)


@pytest.mark.parametrize("log2,n", [(7, 40000), (8, 300000), (9, 40000), (10, 600000), (13, 50000)])
def test_upper_levels(hip_device, log2, n):
    from pyrit_amd import gpu as g

    pts = random_points(n, log2, seed=n, dup_frac=0.1, delete_frac=0.02)
    ref = O.gb_build(log2, pts)
    for levels in (0, 1):
        assert_same_build(g.build(log2, pts, levels=levels), ref, log2)
    one = pts[:1].copy()
    one["x"] = one["y"] = one["z"] = (1 << log2) - 1
    many = np.repeat(one, 70000)  # one voxel of many records in a large grid
    assert_same_build(g.build(log2, many), O.gb_build(log2, many), log2)


def _patch(log2, bricks, per, seed):
    """`per` random voxels in each of `bricks` bricks side by side"""
    rng = np.random.default_rng(seed)
    side = min(1 << (log2 - 2), int(np.ceil(np.sqrt(bricks))))
    b = np.repeat(np.arange(bricks), per)
    bit = np.argsort(rng.random((bricks, 64)), 1)[:, :per].ravel()
    pts = np.zeros(len(b), O.VOXEL)
    pts["x"] = b % side * 4 + (bit & 3)
    pts["y"] = b // side // side * 4 + (bit >> 2 & 3)
    pts["z"] = b // side % side * 4 + (bit >> 4)
    pts["attribute"] = rng.integers(1, 1 << 20, len(b))
    rng.shuffle(pts)
    return pts


@pytest.mark.parametrize("log2,bricks,repeat,small", [(9, 3072, 1, True), (9, 3073, 1, False), (13, 700, 4, True),
                                                      (8, 2048, 3, True), (8, 2049, 3, False), (8, 1024, 20, True),
                                                      (8, 1025, 20, False)])
def test_levels_of_few_bricks(hip_device, log2, bricks, repeat, small):
    """Builds of many records in few bricks of a large grid: the levels of one
    workgroup up to the brick count where dense ones become faster (a build
    that takes those holds the same memory as one asked to), and equal arrays."""
    from pyrit_amd import gpu as g

    pts = np.tile(_patch(log2, bricks, 32, bricks), repeat)
    ref = O.gb_build(log2, pts)
    held = {}
    g.set_timing(True)
    try:
        for levels in (0, 2, 1):
            assert_same_build(g.build(log2, pts, levels=levels), ref, log2)
            held[levels] = g.last_build_times()["device_bytes"]
    finally:
        g.set_timing(False)
    assert (held[0] == held[2]) == small, held
    assert held[1] == held[2]


def test_memory_of_dense_levels(hip_device):
    """2.1e6 records in 20000 bricks of a 2^8 grid: the brick-sized buffers for
    the most bricks there can be hold 16.2 MB, within 8 bytes a record plus
    1 MiB (17.8 MB), but 20.5 MB with the dense levels: such a build counts its
    bricks and holds less than one without dense levels."""
    from pyrit_amd import gpu as g

    pts = np.tile(_patch(8, 20000, 35, 1), 3)
    ref = O.gb_build(8, pts)
    held = []
    g.set_timing(True)
    try:
        for levels in (0, 1):
            assert_same_build(g.build(8, pts, levels=levels), ref, 8)
            held.append(g.last_build_times()["device_bytes"])
    finally:
        g.set_timing(False)
    assert held[0] < held[1], held


@pytest.mark.parametrize("count", [16384, 16385])
def test_many_chunks(hip_device, count):
    """The most chunks whose roots the last kernel writes to the host, and one
    more (they are copied): as a batch, and replayed as a graph with fewer."""
    from pyrit_amd import gpu as g

    rng = np.random.default_rng(count)
    sizes = rng.integers(0, 5, count)
    offs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
    vox = random_points(int(offs[-1]), 3, 1, dup_frac=0.0)
    vox["attribute"][::50] = 0
    ref, rroots, rfirst = O.gb_build_chunks(3, vox, offs)
    graph = g.BuildGraph(3, count, len(vox))
    try:
        for few in (count, 100, count):
            cut = offs.copy()
            cut[few:] = offs[few]
            want, wroots, wfirst = (ref, rroots, rfirst) if few == count else O.gb_build_chunks(3, vox[:cut[-1]], cut)
            for b, roots, first in (graph.launch(vox[:cut[-1]], cut), g.build_chunks(3, vox[:cut[-1]], cut)):
                assert_same_build(b, want, 3)
                assert np.array_equal(roots, wroots) and np.array_equal(first, wfirst)
    finally:
        graph.destroy()
