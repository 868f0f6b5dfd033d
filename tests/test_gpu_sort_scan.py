"""Sorts on both sides of the tile sizes, scans on both sides of their launch rule, displacements
around half a box (GPU), against the oracle and NumPy."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 2048 keys per tile up to 393,216 keys, then 6144; windows of eight tiles
@pytest.mark.parametrize("n", [16385, 18432, 18433, 393216, 393217])
def test_build_order(n):
    import torch
    import neighbor_amd as nb
    import oracle as orc
    rng = np.random.default_rng(n)
    pts = np.ascontiguousarray(np.round(rng.random((n, 3)) * 64) / 8, np.float32)      # many equal codes
    t = orc.build(pts, [0.0] * 3, [9.0] * 3)
    lb = nb.LBVH()
    lb.build(torch.from_numpy(pts).cuda(), [0.0] * 3, [9.0] * 3)
    arr = lb.arrays()
    assert np.array_equal(arr["codes"].cpu().numpy().view(np.uint32), t["codes"])
    assert np.array_equal(arr["primitive"].cpu().numpy().view(np.uint32), t["primitive"])
    assert lb.error_word() == 0


# 2048: tile; 2048 tiles: no launch between the tile sums and the scans
@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, 2048 * 257 + 5, 2048 * 2048, 2048 * 2048 + 1])
@pytest.mark.parametrize("permuted", [False, True])
def test_scan(n, permuted):
    import torch
    from neighbor_amd.api import exclusive_scan
    rng = np.random.default_rng(n)
    counts = rng.integers(0, 2 ** 31 - 1, n).astype(np.int32)
    perm = rng.permutation(n).astype(np.int32) if permuted else None
    got = exclusive_scan(torch.from_numpy(counts).cuda(), perm=None if perm is None else torch.from_numpy(perm).cuda()).cpu().numpy()
    in_order = counts.astype(np.int64) if perm is None else counts[perm].astype(np.int64)
    ends = np.cumsum(in_order)
    want = np.empty(n + 1, np.int64)
    want[np.arange(n) if perm is None else perm] = ends - in_order
    want[n] = ends[-1]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n", [1, 1023, 1025, 262145, 300007])
def test_displacement(n):
    """The largest squared displacement (rounded up by 2^-40, and the FP64 sums' own 2^-51) and the
    number of wrapped points, with differences at 0.49 and 0.5 of the box and beyond."""
    import torch
    from neighbor_amd.api import max_displacement2
    rng = np.random.default_rng(n)
    box = np.array([10.0, 12.5, 20.0], np.float32)
    ref = (rng.random((n, 3)) * box).astype(np.float32)
    step = rng.normal(0, 0.05, (n, 3))
    step[::5] += box * rng.choice([0.0, 0.4899, 0.4901, 0.5, -0.5, 0.75, 1.0, -1.6], (len(step[::5]), 3))
    x = (ref + step).astype(np.float32)
    for periodic in (False, True):
        d = x.astype(np.float64) - ref.astype(np.float64)
        images = np.rint(d / box.astype(np.float64)) if periodic else np.zeros_like(d)
        d = d - box.astype(np.float64) * images
        want = (d * d).sum(1).max()
        wrapped = torch.full((), 7, dtype=torch.int32, device="cuda")
        got = float(max_displacement2(torch.from_numpy(x).cuda(), torch.from_numpy(ref).cuda(),
                                      box=[float(b) for b in box] if periodic else None, wrapped=wrapped).item())
        assert want * (1 - 2.0 ** -50) <= got <= want * (1 + 2.0 ** -39)
        assert int(wrapped.item()) == int((images != 0).any(1).sum())
