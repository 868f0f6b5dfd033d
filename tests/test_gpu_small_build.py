"""Trees and query orders that one workgroup makes (GPU) against the oracle: sizes around its tiles,
all-equal and two-valued codes, points and spheres, and one tree object rebuilt across the limits."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def nb():
    import neighbor_amd
    return neighbor_amd


@pytest.fixture(scope="module")
def orc():
    import oracle
    return oracle


def points_of(n, kind):
    rng = np.random.default_rng(n)
    p = rng.random((n, 3)).astype(np.float32) * np.float32(10)
    if kind == "equal":
        p[:] = p[0]
    if kind == "two":
        p = p[rng.integers(0, min(n, 2), n)]
    if kind == "outside":
        p = p * np.float32(3) - np.float32(10)
    return np.ascontiguousarray(p)


def compare(lb, orc, pts, radius):
    arr = {k: v.cpu().numpy() for k, v in lb.arrays().items()}
    t = orc.build(pts, [0.0] * 3, [10.0] * 3, sphere_r=-1.0 if radius is None else radius)
    for k in ("codes", "primitive"):
        assert np.array_equal(arr[k].view(np.uint32), t[k]), k
    for k in ("parent", "left", "right", "lo", "hi"):
        assert np.array_equal(arr[k], t[k]), k
    assert lb.error_word() == 0


# 64: wave and chunk of keys; 1024: block; 2048: one launch; 16384: sort by counting
@pytest.mark.parametrize("kind", ["uniform", "equal", "two", "outside"])
@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 1023, 1025, 2047, 2048, 2049, 4096, 4161, 16383, 16384, 16385])
def test_small_build(nb, orc, n, kind):
    import torch
    pts = points_of(n, kind)
    x = torch.from_numpy(pts).cuda()
    for radius in (None, 0.4):
        lb = nb.LBVH()
        lb.build(x, [0.0] * 3, [10.0] * 3, radius=radius)
        compare(lb, orc, pts, radius)
        lb.refit(x, radius=radius)
        compare(lb, orc, pts, radius)


def test_sizes_in_turn(nb, orc):
    """One object's workspaces serve builds on both sides of each limit."""
    import torch
    lb = nb.LBVH()
    for n in (2000, 30000, 1, 2048, 16384, 16385, 5000, 2, 20000, 700):
        pts = points_of(n, "uniform")
        lb.build(torch.from_numpy(pts).cuda(), [0.0] * 3, [10.0] * 3)
        if n > 1:
            compare(lb, orc, pts, None)


@pytest.mark.parametrize("n", [65, 257, 1025, 2049, 4097, 16384, 16385])
def test_query_order(nb, orc, n):
    """Queries that a launch orders itself: counts as the oracle's, also for queries that have no code."""
    import torch
    pts = points_of(9000, "uniform")
    rng = np.random.default_rng(n)
    sph = (rng.random((n, 4)) * [12, 12, 12, 0.6] - [1, 1, 1, 0]).astype(np.float32)
    sph[::97, 0] = np.inf
    sph[1::97, 1] = np.nan
    lb, tr = nb.LBVH(), nb.LBVHTraverser()
    lb.build(torch.from_numpy(pts).cuda(), [0.0] * 3, [10.0] * 3)
    got = tr.count(lb, torch.from_numpy(sph).cuda()).cpu().numpy()
    want = orc.traverse(len(pts), orc.compress(orc.build(pts, [0.0] * 3, [10.0] * 3)), sph)["counts"]
    assert np.array_equal(got, want)
