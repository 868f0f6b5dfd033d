"""Packing of rows (GPU): every row length around the copy's group size, against numpy."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, longest", [(1, 9), (63, 5), (64, 9), (257, 3), (1000, 130), (70, 5000)])
@pytest.mark.parametrize("image, stream", [(True, True), (False, True), (True, False)])
def test_pack_rows_lengths(n, longest, image, stream):
    import torch
    from neighbor_amd.api import pack_rows
    rng = np.random.default_rng(1000 * n + longest)
    counts = rng.integers(0, longest + 1, n)
    counts[: min(n, longest + 1)] = np.arange(longest + 1)[: min(n, longest + 1)]      # every length
    rng.shuffle(counts)
    gap = rng.integers(0, 4, n)
    place = rng.permutation(n)                              # rows laid out in another order, with gaps
    ends = np.cumsum((counts + gap)[place])
    start = np.empty(n, np.int64)
    start[place] = ends - (counts + gap)[place] + 1         # odd starts among them
    size = int(ends[-1]) + 2
    neigh = rng.integers(0, 2 ** 31 - 1, size).astype(np.int32)
    img = rng.integers(0, 256, size).astype(np.uint8)
    out = pack_rows(torch.from_numpy(start).cuda(), torch.from_numpy(counts.astype(np.int32)).cuda(),
                    torch.from_numpy(neigh).cuda(), torch.from_numpy(img).cuda() if image else None, pair_stream=stream)
    torch.cuda.synchronize()
    pos = np.repeat(start, counts) + np.arange(counts.sum()) - np.repeat(np.cumsum(counts) - counts, counts)
    assert np.array_equal(np.diff(out["offsets"].cpu().numpy()), counts)
    assert np.array_equal(out["neigh"].cpu().numpy(), neigh[pos])
    assert out["image"] is None if not image else np.array_equal(out["image"].cpu().numpy(), img[pos])
    assert out["first"] is None if not stream else np.array_equal(out["first"].cpu().numpy(), np.repeat(np.arange(n), counts))
