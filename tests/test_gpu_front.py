"""The walk by node fronts (GPU) against the oracle: sizes around its groups, batches, buckets and
launch rules, query orders, scattered and unusual queries, every traversal variant and output."""
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


def host(t):
    return t.cpu().numpy()


def points_of(n, rng, kind):
    L = max((n / 0.85) ** (1.0 / 3.0), 1.0)
    p = rng.random((n, 3)).astype(np.float32) * np.float32(L)
    if kind == "lattice":       # many equal distances and coordinates
        p = np.round(p * 2) / np.float32(2)
    if kind == "copies":        # runs of coincident points
        p = p[rng.integers(0, max(n // 40, 1), n)]
    return np.ascontiguousarray(p, np.float32), float(np.float32(L))


# 16 / 32 / 64: group, run and wave; 2048: chunk; 16384, 32768, 65536: queries per team
SIZES = [1, 2, 15, 16, 17, 32, 33, 63, 64, 65, 130, 1023, 1025, 2049, 16384, 16385, 32769, 65537]


@pytest.mark.parametrize("kind", ["uniform", "lattice", "copies"])
@pytest.mark.parametrize("n", SIZES)
def test_reference_query(nb, orc, n, kind):
    """Counts and lists of every variant equal the oracle's traversal, in order, for queries in
    particle, Morton and random order, with and without images."""
    import torch
    from neighbor_amd.workloads import images27
    if kind != "uniform" and n > 20000:
        pytest.skip("large sizes with uniform points only")
    rng = np.random.default_rng(n)
    pts, L = points_of(n, rng, kind)
    rad = 0.25 if kind == "copies" else None
    r = 1.0 if kind == "copies" else 1.7
    # the points themselves, some outside the box, some with other radii (zero, large, negative)
    sph = np.concatenate([pts, np.full((n, 1), r, np.float32)], 1).astype(np.float32)
    sph[::7, 3] = 0.0
    if n <= 3000:
        sph[3::11, 3] = 0.6 * L
        sph[5::13, :3] += np.float32(1.5 * L)
        sph[6::17, 3] = -r
    tree = orc.build(pts, [0, 0, 0], [L] * 3, -1.0 if rad is None else rad)
    records = orc.compress(tree)
    lb = nb.LBVH()
    lb.build(torch.from_numpy(pts).cuda(), [0, 0, 0], [L] * 3, radius=rad)
    shuffled = rng.permutation(n).astype(np.int32)
    d_sph = torch.from_numpy(sph).cuda()
    images = images27(L) if n < 40000 else images27(L)[9:18]
    for imgs in (images, None):
        ref = orc.traverse(n, records, sph, imgs, triplets=True)
        counts = ref["counts"].astype(np.int64)
        most = int(counts.max()) if n else 0
        for variant in (nb.NB_VARIANT_QUANTIZED, nb.NB_VARIANT_FLOAT_ROPE, nb.NB_VARIANT_WAVE_QUANTIZED):
            tr = nb.LBVHTraverser(variant=variant)
            tr.set_bucket_size(24)
            tr.setup(lb)
            d_img = None if imgs is None else torch.from_numpy(imgs).cuda()
            for order in (None, lb.device_pointers()["primitive"], torch.from_numpy(shuffled).cuda()):
                got = host(tr.count(lb, d_sph, images=d_img, order=order)).view(np.uint32)
                assert np.array_equal(got, ref["counts"]), (variant, imgs is None)
            cut = max(min(most, 40), 1)
            lst, nn = tr.neighbor_list(lb, d_sph, cut, images=d_img)
            assert np.array_equal(host(nn).view(np.uint32), ref["counts"])
            pos = np.concatenate([[0], np.cumsum(counts)])[:-1]
            want = np.zeros((n, cut), np.int64)
            for k in range(cut):
                have = counts > k
                want[have, k] = ref["prim"][pos[have] + k]
            assert np.array_equal(host(lst).astype(np.int64), want)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("bucket", [1, 16, 33, 64])
def test_exact_query(nb, orc, n, bucket):
    """Exact counts and rows (image-major, then Morton order) equal the FP64 cell list."""
    import torch
    from neighbor_amd.api import exact_rows, exclusive_scan
    from neighbor_amd.workloads import images27
    if n > 2049 and bucket not in (16, 64):
        pytest.skip("large sizes with two bucket sizes only")
    rng = np.random.default_rng(n + 77)
    pts, L = points_of(n, rng, "lattice" if n % 2 and n < 3000 else "uniform")
    r = 1.5
    sph = np.concatenate([pts, np.full((n, 1), r, np.float32)], 1).astype(np.float32)
    ref = orc.exact_bruteforce(pts, sph, images27(L, dtype=np.float64)) if n < 3000 else orc.exact_celllist(pts, sph, [L] * 3, r)
    d_pts, d_sph = torch.from_numpy(pts).cuda(), torch.from_numpy(sph).cuda()
    d_img = torch.from_numpy(images27(L, dtype=np.float64)).cuda()
    lb = nb.LBVH()
    lb.build(d_pts, [0, 0, 0], [L] * 3)
    tr = nb.LBVHTraverser(variant=nb.NB_VARIANT_WAVE)
    tr.set_bucket_size(bucket)
    tr.setup(lb)
    counts = ref["counts"].astype(np.int64)
    offs = np.concatenate([[0], np.cumsum(counts)])
    for order in (None, lb.device_pointers()["primitive"], torch.from_numpy(rng.permutation(n).astype(np.int32)).cuda()):
        got = tr.exact_count(lb, d_sph, d_pts, images=d_img, order=order)
        assert np.array_equal(host(got).view(np.uint32), ref["counts"])
        start = exclusive_scan(got)
        neigh = torch.full((int(offs[-1]) + 1,), -1, dtype=torch.int32, device="cuda")
        img = torch.full((int(offs[-1]) + 1,), 77, dtype=torch.uint8, device="cuda")
        filled = exact_rows(tr, lb, d_sph, d_pts, start, got, neigh, img, images=d_img, order=order)
        assert np.array_equal(host(filled).view(np.uint32), ref["counts"])
        nj, nk = host(neigh)[:-1].astype(np.int64), host(img)[:-1].astype(np.int64)
        assert int(neigh[-1]) == -1 and int(img[-1]) == 77
        i = np.repeat(np.arange(n), counts)
        assert np.array_equal(np.lexsort((nk, i)), np.arange(i.size)), "rows are not image by image"
        a = np.lexsort((nj, nk, i))
        b = np.lexsort((ref["j"], ref["k"], i))
        assert np.array_equal(nk[a], ref["k"].astype(np.int64)[b]) and np.array_equal(nj[a], ref["j"].astype(np.int64)[b])


@pytest.mark.parametrize("n", [40, 5000, 70000])
def test_unusual_queries(nb, orc, n):
    """Queries at infinity, NaN, and radii beyond the walk's range beside ordinary ones: the
    ordinary rows are the oracle's, the others those of the definition."""
    import torch
    rng = np.random.default_rng(5)
    pts, L = points_of(n, rng, "uniform")
    sph = np.concatenate([pts, np.full((n, 1), 1.5, np.float32)], 1).astype(np.float32)
    odd = rng.choice(n, 8, replace=False)
    sph[odd[0], 0] = np.inf
    sph[odd[1], 1] = np.nan
    sph[odd[2], 3] = np.inf
    sph[odd[3], 3] = 1e30
    sph[odd[4], 3] = np.nan
    sph[odd[5], :3] = 1e20
    sph[odd[6], :3] = -3e38
    sph[odd[7], 3] = 3e38
    d_pts, d_sph = torch.from_numpy(pts).cuda(), torch.from_numpy(sph).cuda()
    lb = nb.LBVH()
    lb.build(d_pts, [0, 0, 0], [L] * 3)
    ref = orc.traverse(n, orc.compress(orc.build(pts, [0, 0, 0], [L] * 3)), sph, None)["counts"]
    for variant in (nb.NB_VARIANT_QUANTIZED, nb.NB_VARIANT_FLOAT_ROPE, nb.NB_VARIANT_WAVE_QUANTIZED):
        tr = nb.LBVHTraverser(variant=variant)
        tr.setup(lb)
        assert np.array_equal(host(tr.count(lb, d_sph)).view(np.uint32), ref)
    tr = nb.LBVHTraverser(variant=nb.NB_VARIANT_WAVE)
    tr.setup(lb)
    got = host(tr.exact_count(lb, d_sph, d_pts)).astype(np.int64)
    plain = np.setdiff1d(np.arange(n), odd)
    check = np.concatenate([plain[:: max(1, plain.size // 400)], odd])
    with np.errstate(all="ignore"):
        for q in check:
            d = sph[q, :3].astype(np.float64) - pts.astype(np.float64)
            d2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
            want = int((d2 <= np.float64(sph[q, 3]) * np.float64(sph[q, 3])).sum())
            assert got[q] == want, (q, sph[q])


@pytest.mark.parametrize("n", [40, 5000, 70000])
@pytest.mark.parametrize("batched", [False, True])
def test_unusual_queries_beside_rows(nb, n, batched):
    """Exact rows of waves with a few unusual queries: the others' rows are those of a call without
    them, NaN and infinite centers have no hits, a radius beyond the walk's range has every point."""
    import torch
    from neighbor_amd.api import exact_rows, exclusive_scan
    from neighbor_amd.batch import LBVHBatch
    rng = np.random.default_rng(n + 3)
    pts, L = points_of(n, rng, "uniform")
    plain = np.concatenate([pts, np.full((n, 1), 1.3, np.float32)], 1).astype(np.float32)
    none, every = rng.choice(n, 8, replace=False).reshape(2, 4)
    odd = plain.copy()
    plain[none, :3] = -50.0 * L
    odd[none[0], 0] = np.nan
    odd[none[1], 3] = np.nan
    odd[none[2], 1] = np.inf
    odd[none[3], :3] = -np.inf
    odd[every, 3] = (1e30, np.inf, -3e38, 1e15)
    plain[every, 3] = 4.0 * L
    d_pts = torch.from_numpy(pts).cuda()
    box = torch.tensor([[0.0] * 3, [L] * 3], device="cuda")

    def rows(sph):
        d = torch.from_numpy(sph).cuda()
        if batched:
            b = LBVHBatch()
            b.build(d_pts, torch.tensor([0, n], dtype=torch.int32, device="cuda"), box[:1].contiguous(), box[1:].contiguous())
            b.setup()
            counts = b.count(d, periodic=False)
            start = exclusive_scan(counts)
            return host(counts), host(start), host(b.pairs(d, start, periodic=False)[0])
        lb = nb.LBVH()
        lb.build(d_pts, [0, 0, 0], [L] * 3)
        tr = nb.LBVHTraverser(variant=nb.NB_VARIANT_WAVE)
        tr.setup(lb)
        order = lb.device_pointers()["primitive"]
        counts = tr.exact_count(lb, d, d_pts, order=order)
        start = exclusive_scan(counts)
        neigh = torch.full((int(start[-1]),), -1, dtype=torch.int32, device="cuda")
        exact_rows(tr, lb, d, d_pts, start, counts, neigh, order=order)
        return host(counts), host(start), host(neigh)

    got, want = rows(odd), rows(plain)
    assert (got[0][none] == 0).all() and (got[0][every] == n).all()
    for g, w in zip(got, want):
        assert np.array_equal(g, w)


def test_two_streams_share_a_traverser(nb, orc):
    """Unordered queries (sorted on the device in the traverser's workspaces) on two streams and
    with other numbers of queries in turn."""
    import torch
    rng = np.random.default_rng(9)
    pts, L = points_of(30000, rng, "uniform")
    lb = nb.LBVH()
    lb.build(torch.from_numpy(pts).cuda(), [0, 0, 0], [L] * 3)
    tr = nb.LBVHTraverser()
    tr.setup(lb)
    records = orc.compress(orc.build(pts, [0, 0, 0], [L] * 3))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(6)]
    sets, outs = [], []
    for i in range(12):
        sph = np.concatenate([rng.random((2000 + 3001 * (i % 4), 3)) * L, np.full((2000 + 3001 * (i % 4), 1), 1.6)], 1).astype(np.float32)
        sets.append((sph, torch.from_numpy(sph).cuda()))
    torch.cuda.synchronize()
    for i, (_, d) in enumerate(sets):
        with torch.cuda.stream(streams[i % 6]):
            outs.append(tr.count(lb, d, stream=streams[i % 6]))
    torch.cuda.synchronize()
    for (sph, _), out in zip(sets, outs):
        assert np.array_equal(host(out).view(np.uint32), orc.traverse(30000, records, sph, None)["counts"])


@pytest.mark.parametrize("grid", [0, 1, 3, 500])
def test_batch_grids(nb, orc, grid):
    """Boxes of sizes around a wave's 64 queries, by grids of fewer and of more waves than items."""
    import torch
    from neighbor_amd.batch import LBVHBatch
    from neighbor_amd.workloads import batched_boxes, images27, spheres_from_points
    sizes = [1, 2, 63, 64, 65, 128, 129, 700, 3, 2049]
    pts, offsets, lo, hi = batched_boxes(sizes=sizes, seed=3)
    r = 1.2
    sph = spheres_from_points(pts, r)
    b = LBVHBatch()
    b.set_params(bucket=16, grid=grid)
    b.build(torch.from_numpy(pts).cuda(), torch.from_numpy(offsets.astype(np.int32)).cuda(), torch.from_numpy(lo).cuda(),
            torch.from_numpy(hi).cuda())
    b.setup()
    d_sph = torch.from_numpy(sph).cuda()
    counts = host(b.count(d_sph)).astype(np.int64)
    offs = np.concatenate([[0], np.cumsum(counts)])
    neigh, image = b.pairs(d_sph, torch.from_numpy(offs).cuda(), total=int(offs[-1]))
    nj, nk = host(neigh).astype(np.int64), host(image).astype(np.int64)
    for k in range(len(sizes)):
        s, e = int(offsets[k]), int(offsets[k + 1])
        ref = orc.exact_bruteforce(pts[s:e], sph[s:e], images27(hi[k], dtype=np.float64))
        assert np.array_equal(counts[s:e], ref["counts"].astype(np.int64))
        i = np.repeat(np.arange(e - s), counts[s:e])
        rows = slice(int(offs[s]), int(offs[e]))
        a = np.lexsort((nj[rows], nk[rows], i))
        c = np.lexsort((ref["j"], ref["k"], i))
        assert np.array_equal(nk[rows][a], ref["k"].astype(np.int64)[c]) and np.array_equal(nj[rows][a] - s, ref["j"].astype(np.int64)[c])


@pytest.mark.parametrize("n", [1, 2, 31, 33, 64, 65, 500, 2049])
def test_exact_query_rope_records(nb, orc, n):
    """Exact rows of the rope variants, whose records hold the leaves' values only: the pairs of the
    FP64 sum over all points, in the rope walk's order, with and without a transform map."""
    import torch
    from neighbor_amd.api import exact_rows, exclusive_scan
    from neighbor_amd.workloads import images27
    rng = np.random.default_rng(n + 5)
    pts, L = points_of(n, rng, "lattice" if n % 2 else "uniform")
    r = 1.5
    sph = np.concatenate([pts, np.full((n, 1), r, np.float32)], 1).astype(np.float32)
    sph[::5, 3] = 0.0
    sph[1::9, 3] = np.float32(0.45 * L)
    ref = orc.exact_bruteforce(pts, sph, images27(L, dtype=np.float64))
    counts = ref["counts"].astype(np.int64)
    d_sph = torch.from_numpy(sph).cuda()
    d_img = torch.from_numpy(images27(L, dtype=np.float64)).cuda()
    lb = nb.LBVH()
    lb.build(torch.from_numpy(pts).cuda(), [0, 0, 0], [L] * 3)
    prim = host(lb.arrays()["primitive"]).view(np.uint32).astype(np.int64)
    place = np.empty(n, np.int64)
    place[prim] = np.arange(n)
    tag = rng.permutation(n + 3)[:n].astype(np.int32)       # values of the points, and the points by value
    by_tag = np.full((n + 3, 3), 1e6, np.float32)
    by_tag[tag] = pts
    for variant in (nb.NB_VARIANT_QUANTIZED, nb.NB_VARIANT_FLOAT_ROPE, nb.NB_VARIANT_FLOAT_ROPE_EXACT):
        for mapped in (False, True):
            tr = nb.LBVHTraverser(variant=variant)
            kw = dict(transform_map=torch.from_numpy(tag).cuda()) if mapped else {}
            d_pts = torch.from_numpy(by_tag if mapped else pts).cuda()
            for order in (None, lb.device_pointers()["primitive"]):
                got = tr.exact_count(lb, d_sph, d_pts, images=d_img, order=order, **kw)
                assert np.array_equal(host(got).view(np.uint32), ref["counts"])
                start = exclusive_scan(got)
                total = int(counts.sum())
                neigh = torch.full((total + 1,), -1, dtype=torch.int32, device="cuda")
                img = torch.full((total + 1,), 77, dtype=torch.uint8, device="cuda")
                exact_rows(tr, lb, d_sph, d_pts, start, got, neigh, img, images=d_img, order=order, **kw)
                i = np.repeat(np.arange(n), counts)
                key = np.lexsort((place[ref["j"]], ref["k"], ref["i"] if "i" in ref else i))
                want_j = ref["j"].astype(np.int64)[key]
                assert np.array_equal(host(img)[:-1].astype(np.int64), ref["k"].astype(np.int64)[key])
                assert np.array_equal(host(neigh)[:-1].astype(np.int64), tag[want_j] if mapped else want_j)


@pytest.mark.parametrize("n", [1, 3, 40, 700])
def test_exact_query_other_points(nb, n):
    """Points that need not lie in the tree's boxes: a hit is a point within the radius whose leaf's
    box is, too (the quantized boxes: up to two bins larger)."""
    import torch
    rng = np.random.default_rng(n + 11)
    L = 9.0
    centers = (rng.random((n, 3)) * L).astype(np.float32)
    other = (centers + rng.normal(0, 0.6, (n, 3))).astype(np.float32)
    other[::9, 1] = np.nan
    other[4::9] = centers[4::9]
    nq = 200
    sph = np.concatenate([rng.random((nq, 3)) * L, rng.uniform(0.2, 2.5, (nq, 1))], 1).astype(np.float32)
    box_r = 0.25
    lb = nb.LBVH()
    lb.build(torch.from_numpy(centers).cuda(), [0, 0, 0], [L] * 3, radius=box_r)
    q, R = sph[:, None, :3].astype(np.float64), sph[:, None, 3].astype(np.float64)
    near = ((q - other[None].astype(np.float64)) ** 2).sum(2) <= R * R
    gap = np.sqrt((np.maximum(np.abs(q - centers[None]) - box_r, 0.0) ** 2).sum(2))
    least = (near & (gap <= R - 1e-4)).sum(1)
    for variant, more in ((nb.NB_VARIANT_FLOAT_ROPE_EXACT, 1e-4), (nb.NB_VARIANT_FLOAT_ROPE, 0.06), (nb.NB_VARIANT_QUANTIZED, 0.06)):
        tr = nb.LBVHTraverser(variant=variant)
        got = host(tr.exact_count(lb, torch.from_numpy(sph).cuda(), torch.from_numpy(other).cuda())).astype(np.int64)
        most = (near & (gap <= R + more)).sum(1)
        assert (got >= least).all() and (got <= most).all()


@pytest.mark.parametrize("n", [262144, 262145])
def test_exact_query_rope_records_by_size(nb, n):
    """Both sides of the size from which exact queries over rope records take a path each: the counts
    of the bucket records' walk."""
    import torch
    rng = np.random.default_rng(n)
    pts, L = points_of(n, rng, "uniform")
    d_pts = torch.from_numpy(pts).cuda()
    sph = torch.cat([d_pts, torch.full((n, 1), 1.1, device="cuda")], 1).contiguous()
    lb = nb.LBVH()
    lb.build(d_pts, [0, 0, 0], [L] * 3)
    order = lb.device_pointers()["primitive"]
    want = nb.LBVHTraverser(variant=nb.NB_VARIANT_WAVE).exact_count(lb, sph, d_pts, order=order)
    for variant in (nb.NB_VARIANT_QUANTIZED, nb.NB_VARIANT_FLOAT_ROPE, nb.NB_VARIANT_FLOAT_ROPE_EXACT):
        got = nb.LBVHTraverser(variant=variant).exact_count(lb, sph, d_pts, order=order)
        assert torch.equal(got, want)


def test_exact_query_negative_radius(nb):
    """Only the square of an exact query's radius counts, also at distances of exactly the radius and
    where queries take a path each: lattice points have themselves and up to six neighbors."""
    import torch
    k = torch.arange(65, device="cuda", dtype=torch.float32)
    pts = torch.stack(torch.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3).contiguous()
    lb = nb.LBVH()
    lb.build(pts, [0, 0, 0], [65.0] * 3)
    want = 1 + sum((pts[:, a] > 0).int() + (pts[:, a] < 64).int() for a in range(3))
    for radius in (1.0, -1.0):
        sph = torch.cat([pts, torch.full((pts.shape[0], 1), radius, device="cuda")], 1).contiguous()
        for variant in (nb.NB_VARIANT_FLOAT_ROPE_EXACT, nb.NB_VARIANT_QUANTIZED, nb.NB_VARIANT_WAVE):
            tr = nb.LBVHTraverser(variant=variant)
            for order in (None, lb.device_pointers()["primitive"]):
                assert torch.equal(tr.exact_count(lb, sph, pts, order=order), want), (radius, variant)
            assert torch.equal(tr.exact_count(lb, sph[:3000].contiguous(), pts), want[:3000])


# around the launches that one rope path per wave serves: from 2^18 queries, by rows or counts, leaves
# per bucket, images and (counts) radius
@pytest.mark.parametrize("n,bucket,images,radius", [
    (262144, 64, False, 1.0), (262145, 64, False, 1.0), (262145, 24, False, 1.4), (262145, 23, False, 1.4),
    (600001, 64, False, 1.0), (600001, 64, False, 1.9), (800003, 64, True, 1.0), (1048577, 32, True, 0.9),
    (1048577, 64, True, 0.8)])
@pytest.mark.parametrize("given", ["tree", "random", None])
def test_many_exact_queries(nb, n, bucket, images, radius, given):
    """Counts and rows, as given, placed and all moved, equal those of a path per query."""
    import torch
    from neighbor_amd.api import exact_rows, exclusive_scan
    from neighbor_amd.learned import exact_rows_placed
    from neighbor_amd.workloads import images27
    if given != "tree" and n > 600001:
        pytest.skip("the largest in the tree's order only")
    rng = np.random.default_rng(n + bucket)
    pts, L = points_of(n, rng, "uniform")
    d_pts = torch.from_numpy(pts).cuda()
    sph = torch.cat([d_pts, torch.full((n, 1), radius, device="cuda")], 1).contiguous()
    sph[12345, 0] = float("nan")
    sph[54321, 3] = -radius
    img = torch.from_numpy(images27(L, dtype=np.float64)).cuda() if images else None
    lb = nb.LBVH()
    lb.build(d_pts, [0, 0, 0], [L] * 3)
    prim = lb.arrays()["primitive"].long()
    tree = lb.device_pointers()["primitive"]
    order = {"tree": tree, "random": torch.from_numpy(rng.permutation(n).astype(np.int32)).cuda(), None: None}[given]

    def rows(variant, order):
        tr = nb.LBVHTraverser(variant=variant)
        tr.set_bucket_size(bucket)
        tr.setup(lb)
        counts = tr.exact_count(lb, sph, d_pts, images=img, order=order)
        start = exclusive_scan(counts, perm=tree)
        neigh = torch.full((int(counts.sum()),), -1, dtype=torch.int32, device="cuda")
        image = torch.full((neigh.numel(),), 77, dtype=torch.uint8, device="cuda")
        exact_rows(tr, lb, sph, d_pts, start, counts, neigh, image, images=img, order=order)
        return tr, counts, start, neigh, image

    _, counts, start, neigh, image = rows(nb.NB_VARIANT_FLOAT_ROPE_EXACT, tree)
    tr, *got = rows(nb.NB_VARIANT_WAVE, order)
    for g, w in zip(got, (counts, start, neigh, image)):
        assert torch.equal(g, w)
    if given != "tree":
        return
    for moved in (False, True):
        cap = counts // 2 if moved else counts.clone()
        sums = torch.zeros(((n + 255) // 256 * 256,), dtype=torch.int64, device="cuda")
        sums[:n] = cap[prim].long()
        base = torch.zeros((n + 255) // 256 + 1, dtype=torch.int64, device="cuda")
        base[1:] = sums.view(-1, 256).sum(1).cumsum(0)
        used = int(base[-1])
        spill = torch.tensor([used, 0], dtype=torch.int64, device="cuda")
        to = torch.full((used + neigh.numel(),), -1, dtype=torch.int32, device="cuda")
        to_image = torch.full((to.numel(),), 77, dtype=torch.uint8, device="cuda")
        at, nn = torch.zeros(n + 1, dtype=torch.int64, device="cuda"), torch.zeros_like(counts)
        exact_rows_placed(tr, lb, sph, d_pts, base, at, cap, to, to_image, nn, spill=spill, images=img)
        assert torch.equal(nn, counts)
        rest = torch.arange(neigh.numel(), device="cuda") - torch.repeat_interleave(start[:n][prim], counts[prim].long())
        where = torch.repeat_interleave(at[:n][prim], counts[prim].long()) + rest
        assert torch.equal(to[where], neigh) and torch.equal(to_image[where], image)


@pytest.mark.parametrize("nq", [20000, 32768, 40001])
@pytest.mark.parametrize("images", [False, True])
def test_scattered_teams(nb, orc, nq, images):
    """Queries in random order served by teams of 32 and 64, in a tree in which such queries take a path
    each: lists and exact rows in the walks' order, and rows that all move."""
    import torch
    from neighbor_amd.api import exact_rows, exclusive_scan
    from neighbor_amd.workloads import images27
    rng = np.random.default_rng(nq)
    n = 40001
    pts, L = points_of(n, rng, "uniform")
    sph = np.concatenate([rng.random((nq, 3)) * L, rng.uniform(0.5, 1.4, (nq, 1))], 1).astype(np.float32)
    sph[77, 1] = np.nan
    imgs = images27(L)
    d_pts, d_sph = torch.from_numpy(pts).cuda(), torch.from_numpy(sph).cuda()
    lb = nb.LBVH()
    lb.build(d_pts, [0, 0, 0], [L] * 3)
    order = torch.from_numpy(rng.permutation(nq).astype(np.int32)).cuda()
    ref = orc.traverse(n, orc.compress(orc.build(pts, [0, 0, 0], [L] * 3)), sph, imgs if images else None, triplets=True)
    want = ref["counts"].astype(np.int64)
    starts = np.concatenate([[0], np.cumsum(want)])
    f32 = torch.from_numpy(imgs).cuda() if images else None
    f64 = torch.from_numpy(imgs.astype(np.float64)).cuda() if images else None
    for variant in (nb.NB_VARIANT_QUANTIZED, nb.NB_VARIANT_WAVE_QUANTIZED):
        tr = nb.LBVHTraverser(variant=variant)
        assert np.array_equal(host(tr.count(lb, d_sph, images=f32, order=order)).astype(np.int64), want)
        neigh, image = tr.pairs(lb, d_sph, torch.from_numpy(starts).cuda(), images=f32, order=order)
        assert np.array_equal(host(neigh).astype(np.int64), ref["prim"].astype(np.int64))
        assert np.array_equal(host(image), ref["image"])
    rows = []
    for variant in (nb.NB_VARIANT_FLOAT_ROPE_EXACT, nb.NB_VARIANT_WAVE):
        tr = nb.LBVHTraverser(variant=variant)
        counts = tr.exact_count(lb, d_sph, d_pts, images=f64, order=order)
        start = exclusive_scan(counts)
        total = int(start[-1])
        neigh = torch.full((total,), -1, dtype=torch.int32, device="cuda")
        exact_rows(tr, lb, d_sph, d_pts, start, counts, neigh, images=f64, order=order)
        # no room at first: every row that has pairs moves
        moved, cap = start.clone(), torch.zeros_like(counts)
        to = torch.full((2 * total,), -1, dtype=torch.int32, device="cuda")
        spill = torch.tensor([total, 0], dtype=torch.int64, device="cuda")
        got = exact_rows(tr, lb, d_sph, d_pts, moved, cap, to, images=f64, order=order, spill=spill)
        assert torch.equal(got, counts) and int(spill[0]) == 2 * total
        at = torch.arange(total, device="cuda") + torch.repeat_interleave(moved[:nq] - start[:nq], counts.long())
        assert torch.equal(to[at], neigh)
        rows.append((host(counts), host(neigh)))
    assert np.array_equal(rows[0][0], rows[1][0]) and np.array_equal(rows[0][1], rows[1][1])
    ref = orc.exact_bruteforce(pts, sph[:2000], imgs.astype(np.float64) if images else np.zeros((1, 3)), pairs=False)
    assert np.array_equal(rows[0][0][:2000].view(np.uint32), ref["counts"])


@pytest.mark.parametrize("n", [4096, 4097, 12288, 12289, 28672, 28673, 49152, 49153])
def test_rows_by_team_size(nb, n):
    """Rows and lists on both sides of the lines between teams, and between teams and waves, equal the
    one-by-one emission of a path per query."""
    import torch
    from neighbor_amd.api import exact_rows, exclusive_scan
    from neighbor_amd.workloads import images27
    rng = np.random.default_rng(n + 9)
    nt = 300000     # exact queries over float rope records take a path each above 2^18
    pts, L = points_of(nt, rng, "uniform")
    d_pts = torch.from_numpy(pts).cuda()
    lb = nb.LBVH()
    lb.build(d_pts, [0, 0, 0], [L] * 3)
    sph = torch.cat([d_pts, torch.full((nt, 1), 1.2, device="cuda")], 1).contiguous()
    img = torch.from_numpy(images27(L, dtype=np.float64)).cuda()
    paths = nb.LBVHTraverser(variant=nb.NB_VARIANT_FLOAT_ROPE_EXACT)
    every = paths.exact_count(lb, sph, d_pts, images=img)
    all_start = exclusive_scan(every)
    all_neigh = torch.empty(int(all_start[-1]), dtype=torch.int32, device="cuda")
    exact_rows(paths, lb, sph, d_pts, all_start, every, all_neigh, images=img)
    few = sph[:n].contiguous()
    total = int(all_start[n])
    for variant in (nb.NB_VARIANT_WAVE, nb.NB_VARIANT_FLOAT_ROPE_EXACT):
        tr = nb.LBVHTraverser(variant=variant)
        neigh = torch.full((total,), -1, dtype=torch.int32, device="cuda")
        got = exact_rows(tr, lb, few, d_pts, all_start[:n].contiguous(), every[:n].contiguous(), neigh, images=img)
        assert torch.equal(got, every[:n]) and torch.equal(neigh, all_neigh[:total])
    counts = nb.LBVHTraverser().count(lb, sph, images=img.float())
    lst, nn = nb.LBVHTraverser().neighbor_list(lb, few, 24, images=img.float())
    want, _ = nb.LBVHTraverser(variant=nb.NB_VARIANT_FLOAT_ROPE).neighbor_list(lb, sph, 24, images=img.float())
    assert torch.equal(nn, counts[:n]) and torch.equal(lst, want[:n])
