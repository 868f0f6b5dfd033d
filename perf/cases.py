"""Performance cases of the neighbor library: what its users have it do, through its public API.

``listed()`` names the cases, ``draw(rng)`` gives another one of the same ranges, ``prepare``
makes what a program holds before the call (positions, trees' handles, output buffers with
headroom), ``run`` is one pass, ``work`` what a pass cannot do without and ``exact`` its
floating outputs in 64 bits.

Kinds of passes (case["kind"]):

raw      tree build, traverser set-up and one traversal with the float sphere query (the
         reference library's semantics): neighbor counts or a fixed-stride neighbor list, over
         27 periodic images or none, with the spheres in particle order or in Morton order.
exact    build, set-up, exact FP64 count, scan of the counts into row starts and exact fill of
         the (neighbor, image) rows, over float3 positions or 16-byte records.
learned  the single-pass form: row capacities from the trained network beside the build, one
         fill with placed rows, rows packed without gaps.
boxes    many independent periodic boxes in one forest: a captured plan (count, scan, fill), or
         the single pass over rows sized by each box's density, packed.
mixture  per-type lists of a size-asymmetric mixture (one tree per type, a cutoff per pair),
         packed into particle order.
md       a step of a dynamics loop that keeps the hierarchy: displacement test, refit, set-up,
         exact count, scan, fill.
tree     the build alone; its arrays are the output.
"""
import math

import numpy as np
import torch

import neighbor_amd as nb
from neighbor_amd.api import LBVH, LBVHTraverser, exact_rows, exclusive_scan, max_displacement2
from neighbor_amd.batch import BatchPlan, BatchRows, LBVHBatch
from neighbor_amd.learned import CapacityPredictor, LearnedFill, exact_rows_placed, learned_exact_pairs
from neighbor_amd.typed import TypedNeighborList
from neighbor_amd.workloads import box_length, images27

VARIANTS = {
    "quantized": nb.NB_VARIANT_QUANTIZED,
    "float": nb.NB_VARIANT_FLOAT_ROPE,
    "wave_quantized": nb.NB_VARIANT_WAVE_QUANTIZED,
}


def listed():
    return [
        # the smallest call: a list over the ideal gas of the reference's own test (1000 points),
        # spheres as they come, the default traverser
        dict(name="raw list 1k", kind="raw", n=1000, rho=1.0, r=2.8, periodic=True, variant="quantized", sorted=False,
             output="list", insert="points"),
        # the small benchmark configuration (N = 10,000, rho = 1), Morton-ordered spheres
        dict(name="raw count 10k", kind="raw", n=10_000, rho=1.0, r=2.8, periodic=True, variant="quantized", sorted=True,
             output="count", insert="points"),
        # the large benchmark configuration, the reference benchmark's traversal
        dict(name="raw count 1m", kind="raw", n=1_000_000, rho=0.85, r=2.8, periodic=True, variant="quantized", sorted=True,
             output="count", insert="points"),
        # a small simulation's exact list
        dict(name="exact 10k", kind="exact", n=10_000, rho=1.0, r=2.8, periodic=True, bucket=32, records=False, image=True),
        # a middle-sized cluster without periodic images, odd count, records read in place
        dict(name="exact 131k open", kind="exact", n=131_071, rho=0.85, r=2.0, periodic=False, bucket=16, records=True,
             image=False),
        # the large benchmark configuration, count then fill
        dict(name="exact 1m", kind="exact", n=1_000_000, rho=0.85, r=2.8, periodic=True, bucket=48, records=False, image=True),
        # the headline step (single pass), rows packed for the consumer
        dict(name="learned 1m", kind="learned", n=1_000_000, rho=0.85, r=2.8, clusters=0, bucket=48),
        # the clustered configuration at half its size, odd count
        dict(name="learned clustered 2m", kind="learned", n=2_000_003, rho=0.85, r=2.8, clusters=500, bucket=48),
        # batched boxes: 512 of the benchmark's 4096, log-uniform sizes
        dict(name="boxes 512", kind="boxes", nbox=512, nmin=256, nmax=16384, rho=0.85, r=2.8, mode="plan", bucket=32),
        # the colloid mixture at a fifth of its size
        dict(name="mixture 400k", kind="mixture", n=400_000, phi=0.3, skin=0.4, half=False, records=False),
        # one recompute of a dynamics loop that keeps its hierarchy
        dict(name="md refit 300k", kind="md", n=300_007, rho=0.85, r=2.8, step=0.1, bucket=32),
        # the largest build, above the size where the build's chunks change
        dict(name="tree 6m", kind="tree", n=6_300_001, rho=0.85, insert="points"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges: sizes log-uniform, odd ones among them, other options."""
    kind = rng.choice(["raw", "raw", "exact", "exact", "learned", "boxes", "mixture", "md", "tree"])
    rho = round(rng.uniform(0.6, 1.0), 3)
    r = round(rng.uniform(1.5, 2.8), 3)
    bucket = rng.choice([16, 32, 48, 64])
    if kind == "raw":
        return dict(kind=kind, n=_log_uniform(rng, 500, 800_000), rho=rho, r=r, periodic=rng.random() < 0.7,
                    variant=rng.choice(["quantized", "quantized", "float", "wave_quantized"]), sorted=rng.random() < 0.6,
                    output=rng.choice(["count", "list"]), insert=rng.choice(["points", "points", "spheres"]))
    if kind == "exact":
        return dict(kind=kind, n=_log_uniform(rng, 500, 900_000), rho=rho, r=r, periodic=rng.random() < 0.7, bucket=bucket,
                    records=rng.random() < 0.4, image=rng.random() < 0.7)
    if kind == "learned":
        return dict(kind=kind, n=_log_uniform(rng, 50_000, 900_000), rho=rho, r=r, clusters=rng.choice([0, 100]),
                    bucket=bucket)
    if kind == "boxes":
        return dict(kind=kind, nbox=_log_uniform(rng, 8, 400), nmin=_log_uniform(rng, 64, 512),
                    nmax=_log_uniform(rng, 1024, 16384), rho=rho, r=r, mode=rng.choice(["plan", "single"]), bucket=bucket)
    if kind == "mixture":
        return dict(kind=kind, n=_log_uniform(rng, 20_000, 350_000), phi=round(rng.uniform(0.15, 0.3), 3), skin=0.4,
                    half=rng.random() < 0.5, records=rng.random() < 0.5)
    if kind == "md":
        return dict(kind=kind, n=_log_uniform(rng, 3000, 300_000), rho=rho, r=r, step=round(rng.uniform(0.02, 0.2), 3),
                    bucket=bucket)
    return dict(kind=kind, n=_log_uniform(rng, 700, 6_000_000), rho=rho, insert=rng.choice(["points", "spheres"]))


# ------------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _uniform(n, L, gen):
    """n points of [0, L)^3."""
    x = torch.rand((n, 3), generator=gen, device="cuda") * L
    return torch.where(x >= L, torch.zeros_like(x), x)


def _clustered(n, L, clusters, gen):
    """A fifth of the points uniform, the rest in Gaussian clusters of standard deviation 5."""
    x = torch.rand((n, 3), generator=gen, device="cuda", dtype=torch.float64) * L
    n_cl = n - n // 5
    centers = torch.rand((clusters, 3), generator=gen, device="cuda", dtype=torch.float64) * L
    which = torch.randint(clusters, (n_cl,), generator=gen, device="cuda")
    g = torch.randn((n_cl, 3), generator=gen, device="cuda", dtype=torch.float64)
    x[n - n_cl:] = torch.remainder(centers[which] + 5.0 * g, L)
    x = x.float()
    return torch.where(x >= L, torch.zeros_like(x), x)


def _points(case, seed):
    L = box_length(case["n"], case["rho"])
    gen = _generator(seed)
    if case.get("clusters"):
        return _clustered(case["n"], L, case["clusters"], gen), L
    return _uniform(case["n"], L, gen), L


def _spheres(points, r):
    s = torch.empty((points.shape[0], 4), dtype=torch.float32, device="cuda")
    s[:, :3] = points[:, :3]
    s[:, 3] = r
    return s


def _images(L, dtype):
    return torch.from_numpy(images27(L, dtype=np.float32 if dtype == torch.float32 else np.float64)).cuda()


def _mean_neighbors(case):
    """Mean neighbors of a particle: those of the mean density and, of a clustered point, those
    of its own Gaussian cluster."""
    own = 0.8 * (0.8 * case["n"] / case["clusters"]) / (4.0 * math.pi * 25.0) ** 1.5 if case.get("clusters") else 0.0
    return 4.0 / 3.0 * math.pi * case["r"] ** 3 * (case["rho"] + own)


class _Packed:
    """Kept buffers of rows packed without gaps, in particle order."""

    def __init__(self, n, capacity):
        self.n = n
        self.offsets = torch.empty(n + 1, dtype=torch.int64, device="cuda")
        self.neigh = torch.zeros(capacity, dtype=torch.int32, device="cuda")
        self.image = torch.zeros(capacity, dtype=torch.uint8, device="cuda")

    def pack(self, start, counts, neigh, image):
        exclusive_scan(counts, self.offsets)
        rc = nb.lib().nb_rows_pack(start.data_ptr(), counts.data_ptr(), self.n, None, self.offsets.data_ptr(), neigh.data_ptr(),
                                   image.data_ptr(), self.neigh.data_ptr(), self.image.data_ptr(), None,
                                   torch.cuda.current_stream().cuda_stream)
        if rc != 0:
            raise RuntimeError("nb_rows_pack failed (%d)" % rc)
        return {"counts": counts, "offsets": self.offsets, "neigh": self.neigh, "image": self.image}


def _pair_capacity(n, mean):
    """Positions of a pair buffer with headroom."""
    return int(n * (mean + 2.0) * 1.15) + 4096


def _mixture(case, seed):
    """Large spheres (1%, diameter 10) on random sites of a lattice, small ones (diameter 1)
    uniform outside them, in random particle order; total volume fraction phi."""
    gen = _generator(seed)
    n = case["n"]
    n_l = max(n // 100, 1)
    volume = (n_l * 1000.0 + (n - n_l)) * math.pi / 6.0
    L = float(torch.tensor((volume / case["phi"]) ** (1.0 / 3.0), dtype=torch.float32))
    side = max(int(L // 10.5), 1)
    cell = L / side
    site = torch.full((side ** 3,), -1, dtype=torch.long, device="cuda")
    chosen = torch.randperm(side ** 3, generator=gen, device="cuda")[:n_l]
    n_l = chosen.shape[0]
    site[chosen] = torch.arange(n_l, device="cuda")
    corner = torch.stack([chosen // (side * side), (chosen // side) % side, chosen % side], 1).double()
    large = (corner + 0.5) * cell + (torch.rand((n_l, 3), generator=gen, device="cuda", dtype=torch.float64) - 0.5) * (cell - 10.0)
    small = torch.empty((0, 3), dtype=torch.float64, device="cuda")
    while small.shape[0] < n - n_l:
        c = torch.rand((2 * (n - n_l - small.shape[0]) + 1024, 3), generator=gen, device="cuda", dtype=torch.float64) * L
        at = (c / cell).long().clamp_(max=side - 1)
        free = torch.ones(c.shape[0], dtype=torch.bool, device="cuda")
        for dx in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dz in (-1, 0, 1):
                    b = torch.remainder(at + torch.tensor([dx, dy, dz], device="cuda"), side)
                    k = site[(b[:, 0] * side + b[:, 1]) * side + b[:, 2]]
                    d = c - large[k.clamp(min=0)]
                    d -= L * torch.round(d / L)
                    free &= (k < 0) | ((d * d).sum(1) >= 5.5 ** 2)
        small = torch.cat([small, c[free]])[:n - n_l]
    x = torch.cat([small, large]).float()
    x = torch.where(x >= L, torch.zeros_like(x), x)
    types = torch.cat([torch.zeros(n - n_l, dtype=torch.int32, device="cuda"),
                       torch.ones(n_l, dtype=torch.int32, device="cuda")])
    p = torch.randperm(n, generator=gen, device="cuda")
    return x[p].contiguous(), types[p].cpu().numpy(), L


def _box_sizes(case):
    """Box sizes log-uniform in [nmin, nmax], spread evenly over the boxes."""
    lo, hi, n = math.log(case["nmin"]), math.log(case["nmax"] + 1), case["nbox"]
    return [min(int(math.exp(lo + (hi - lo) * ((b * 0.6180339887498949 + 0.5) % 1.0))), case["nmax"]) for b in range(n)]


# ------------------------------------------------------------------------------- states
def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["case"]["kind"]](state)


def _prepare_raw(case, seed):
    pts, L = _points(case, seed)
    n = case["n"]
    trav = LBVHTraverser(variant=VARIANTS[case["variant"]])
    if case["variant"] == "wave_quantized":
        trav.set_bucket_size(32)
    return dict(case=case, pts=pts, L=L, spheres=_spheres(pts, case["r"]), lbvh=LBVH(), trav=trav,
                images=_images(L, torch.float32) if case["periodic"] else None,
                counts=torch.empty(n, dtype=torch.int32, device="cuda"),
                max_neigh=int(1.5 * _mean_neighbors(case)) + 24, radius=0.25 if case["insert"] == "spheres" else None)


def _run_raw(s):
    case, lbvh, trav, L = s["case"], s["lbvh"], s["trav"], s["L"]
    lbvh.build(s["pts"], [0.0, 0.0, 0.0], [L, L, L], radius=s["radius"])
    trav.setup(lbvh)
    order = lbvh.device_pointers()["primitive"] if case["sorted"] else None
    if case["output"] == "count":
        return {"counts": trav.count(lbvh, s["spheres"], images=s["images"], order=order, nneigh=s["counts"])}
    neigh, counts = trav.neighbor_list(lbvh, s["spheres"], s["max_neigh"], images=s["images"], order=order)
    return {"counts": counts, "neigh": neigh}


def _rows_state(case, seed, pts, L):
    n = case["n"]
    trav = LBVHTraverser(variant=nb.NB_VARIANT_WAVE)
    trav.set_bucket_size(case["bucket"])
    cap = _pair_capacity(n, _mean_neighbors(case))
    return dict(case=case, pts=pts, L=L, spheres=_spheres(pts, case["r"]), lbvh=LBVH(), trav=trav,
                counts=torch.empty(n, dtype=torch.int32, device="cuda"),
                filled=torch.empty(n, dtype=torch.int32, device="cuda"),
                offsets=torch.empty(n + 1, dtype=torch.int64, device="cuda"),
                neigh=torch.zeros(cap, dtype=torch.int32, device="cuda"),
                image=torch.zeros(cap, dtype=torch.uint8, device="cuda") if case.get("image", True) else None,
                images=_images(L, torch.float64) if case.get("periodic", True) else None)


def _prepare_exact(case, seed):
    pts, L = _points(case, seed)
    s = _rows_state(case, seed, pts, L)
    if case["records"]:
        s["pts"] = torch.cat([pts, torch.zeros((case["n"], 1), device="cuda")], 1)
    return s


def _count_and_fill(s):
    lbvh, trav = s["lbvh"], s["trav"]
    order = lbvh.device_pointers()["primitive"]
    counts = trav.exact_count(lbvh, s["spheres"], s["pts"], images=s["images"], order=order, nneigh=s["counts"])
    exclusive_scan(counts, s["offsets"], perm=order)
    exact_rows(trav, lbvh, s["spheres"], s["pts"], s["offsets"], counts, s["neigh"], s["image"], images=s["images"],
               order=order, nneigh=s["filled"])
    out = {"counts": counts, "offsets": s["offsets"], "neigh": s["neigh"]}
    if s["image"] is not None:
        out["image"] = s["image"]
    return out


def _run_exact(s):
    lo, hi = [0.0, 0.0, 0.0], [s["L"]] * 3
    if s["case"]["records"]:
        s["lbvh"].build_postype(s["pts"], lo, hi)
    else:
        s["lbvh"].build(s["pts"], lo, hi)
    s["trav"].setup(s["lbvh"])
    return _count_and_fill(s)


def _prepare_learned(case, seed):
    # the network is trained on an earlier configuration of the same system, which also sizes
    # the row buffer
    train, L = _points(case, seed + 7_000_003)
    n, r = case["n"], case["r"]
    lo, hi = [0.0, 0.0, 0.0], [L] * 3
    lbvh = LBVH()
    trav = LBVHTraverser(variant=nb.NB_VARIANT_WAVE)
    trav.set_bucket_size(case["bucket"])
    images = _images(L, torch.float64)
    spheres = _spheres(train, r)
    lbvh.build(train, lo, hi)
    trav.setup(lbvh)
    counts = trav.exact_count(lbvh, spheres, train, images=images, order=lbvh.device_pointers()["primitive"])
    pred = CapacityPredictor(seed=1)
    pred.features(lbvh, lo, hi, r)
    pred.train(lbvh, counts, steps=300, batch=16384, lr=3e-3)
    margin = pred.margin(lbvh, 0.999)
    buf = LearnedFill(n)
    learned_exact_pairs(trav, lbvh, pred, spheres, train, images, margin, pad=8, buffers=buf, placed=(lo, hi, r))
    buf.grow(int(buf.neigh.numel() * 1.15), keep=False)
    packed = _Packed(n, _pair_capacity(n, 1.1 * _mean_neighbors(case)))
    lbvh.enable_sorted_event(True)
    pts, _ = _points(case, seed)
    return dict(case=case, pts=pts, L=L, spheres=_spheres(pts, r), lbvh=lbvh, trav=trav, pred=pred, margin=margin, buf=buf,
                packed=packed, images=images, side=torch.cuda.Stream(), ready=torch.cuda.Event())


def _run_learned(s):
    case, lbvh, trav, buf, L = s["case"], s["lbvh"], s["trav"], s["buf"], s["L"]
    lo, hi = [0.0, 0.0, 0.0], [L] * 3
    lbvh.build(s["pts"], lo, hi)
    # the prediction needs only the sorted points: beside the rest of the build
    lbvh.wait_sorted(stream=s["side"])
    with torch.cuda.stream(s["side"]):
        s["pred"].predict_rows(lbvh, lo, hi, case["r"], s["margin"], 8, buf.cap, buf.base, buf.spill, stream=s["side"])
    s["ready"].record(s["side"])
    trav.setup(lbvh)
    torch.cuda.current_stream().wait_event(s["ready"])
    exact_rows_placed(trav, lbvh, s["spheres"], s["pts"], buf.base, buf.start, buf.cap, buf.neigh, buf.image, buf.count,
                      spill=buf.spill, images=s["images"])
    return s["packed"].pack(buf.start, buf.count, buf.neigh, buf.image)


def _prepare_boxes(case, seed):
    gen = _generator(seed)
    sizes = _box_sizes(case)
    Ls = [box_length(m, case["rho"]) for m in sizes]
    n = sum(sizes)
    size_t = torch.tensor(sizes, device="cuda")
    L_t = torch.tensor(Ls, dtype=torch.float32, device="cuda")
    offsets = torch.zeros(len(sizes) + 1, dtype=torch.int64, device="cuda")
    offsets[1:] = torch.cumsum(size_t, 0)
    L_p = torch.repeat_interleave(L_t, size_t)[:, None]
    pts = torch.rand((n, 3), generator=gen, device="cuda") * L_p
    pts = torch.where(pts >= L_p, torch.zeros_like(pts), pts).contiguous()
    box_lo = torch.zeros((len(sizes), 3), dtype=torch.float32, device="cuda")
    box_hi = L_t[:, None].expand(-1, 3).contiguous()
    offsets32 = offsets.to(torch.int32)
    spheres = _spheres(pts, case["r"])
    cap = _pair_capacity(n, _mean_neighbors(case))
    batch = LBVHBatch()
    batch.set_params(block=256, bucket=case["bucket"])
    s = dict(case=case, pts=pts, offsets=offsets32, lo=box_lo, hi=box_hi, spheres=spheres, batch=batch)
    if case["mode"] == "plan":
        s["plan"] = BatchPlan(batch, pts, offsets32, box_lo, box_hi, spheres, cap)
        s["plan"].neigh.zero_()
        s["plan"].image.zero_()
    else:
        s["rows"] = BatchRows(n, 2 * cap)
        s["packed"] = _Packed(n, cap)
    return s


def _run_boxes(s):
    if s["case"]["mode"] == "plan":
        plan = s["plan"]
        plan.launch()
        return {"counts": plan.nneigh, "offsets": plan.offsets, "neigh": plan.neigh, "image": plan.image}
    batch, rows = s["batch"], s["rows"]
    batch.build(s["pts"], s["offsets"], s["lo"], s["hi"])
    batch.setup()
    batch.single_pass(s["spheres"], rows)
    return s["packed"].pack(rows.start, rows.count, rows.neigh, rows.image)


def _prepare_mixture(case, seed):
    pts, types, L = _mixture(case, seed)
    lists = TypedNeighborList(2)
    # the choices the tuner makes on this mixture
    lists.choice[(0, 1)] = (nb.NB_VARIANT_WAVE, 16)
    lists.choice[(1, 0)] = (nb.NB_VARIANT_FLOAT_ROPE_EXACT, 1)
    lists.set_types(types)
    if case["records"]:
        pts = torch.cat([pts, torch.from_numpy(types).cuda().float()[:, None]], 1).contiguous()
    skin = case["skin"]
    return dict(case=case, pts=pts, L=L, lists=lists, R=[[1.0 + skin, 5.5 + skin], [5.5 + skin, 10.0 + skin]],
                packed=_Packed(case["n"], 4 * case["n"] + 4096))


def _run_mixture(s):
    lists = s["lists"]
    lists.build(s["pts"], s["L"])
    res = lists.compute(s["R"], half=s["case"]["half"])
    return s["packed"].pack(res["start"], res["counts"], res["neigh"], res["image"])


def _md_points(case, seed):
    """(reference positions, positions a few steps later): no particle has crossed the box."""
    ref, L = _points(case, seed)
    d = (torch.rand((case["n"], 3), generator=_generator(seed + 1_000_003), device="cuda") * 2.0 - 1.0) * case["step"]
    pts = ref + d
    top = torch.nextafter(torch.tensor(L, device="cuda"), torch.tensor(0.0, device="cuda"))
    return ref, torch.minimum(torch.clamp(pts, min=0.0), top).contiguous(), L


def _prepare_md(case, seed):
    ref, pts, L = _md_points(case, seed)
    s = _rows_state(case, seed, pts, L)
    s["ref"] = ref
    s["disp2"] = torch.zeros((), dtype=torch.float64, device="cuda")
    s["wrapped"] = torch.zeros((), dtype=torch.int32, device="cuda")
    s["lbvh"].build(ref, [0.0, 0.0, 0.0], [L, L, L])
    return s


def _run_md(s):
    disp2 = max_displacement2(s["pts"], s["ref"], box=[s["L"]] * 3, out=s["disp2"], wrapped=s["wrapped"])
    s["lbvh"].refit(s["pts"])
    s["trav"].setup(s["lbvh"])
    out = _count_and_fill(s)
    out["disp2"], out["wrapped"] = disp2, s["wrapped"]
    return out


class _Array:
    """A tree array in device memory, for torch.as_tensor (the tensor keeps this object, and so
    the tree that owns the memory, alive)."""

    def __init__(self, lbvh, address, shape, typestr):
        self.lbvh = lbvh
        self.__cuda_array_interface__ = dict(data=(address, False), shape=shape, typestr=typestr, version=2)


def _tree_tensors(lbvh):
    """The tree's arrays as tensors over its own memory."""
    n, ni, nn, _ = lbvh.info()
    p = lbvh.device_pointers()
    shapes = dict(parent=(nn,), left=(ni,), right=(ni,), primitive=(n,), lo=(nn, 3), hi=(nn, 3), rope=(nn,), codes=(n,))
    return {k: torch.as_tensor(_Array(lbvh, p[k], shapes[k], "<f4" if k in ("lo", "hi") else "<i4"), device="cuda") for k in shapes}


def _prepare_tree(case, seed):
    pts, L = _points(case, seed)
    return dict(case=case, pts=pts, L=L, lbvh=LBVH(), radius=0.25 if case["insert"] == "spheres" else None)


def _run_tree(s):
    s["lbvh"].build(s["pts"], [0.0, 0.0, 0.0], [s["L"]] * 3, radius=s["radius"])
    return _tree_tensors(s["lbvh"])


_PREPARE = dict(raw=_prepare_raw, exact=_prepare_exact, learned=_prepare_learned, boxes=_prepare_boxes,
                mixture=_prepare_mixture, md=_prepare_md, tree=_prepare_tree)
_RUN = dict(raw=_run_raw, exact=_run_exact, learned=_run_learned, boxes=_run_boxes, mixture=_run_mixture, md=_run_md,
            tree=_run_tree)


# ------------------------------------------------------------------------------- work
def work(case):
    """Bytes: positions, spheres and images read once, counts, row starts and pairs (or the tree's
    arrays) written once.  Operations: 8 per pair found (its distance test)."""
    kind = case["kind"]
    if kind == "tree":
        # parent, left, right, primitive, lo, hi, rope, codes
        return {"bytes": case["n"] * (12 + 8 + 4 + 4 + 4 + 24 + 24 + 8 + 4), "flops": 30.0 * case["n"]}
    if kind == "boxes":
        n = sum(_box_sizes(case))
        mean = _mean_neighbors(case)
    elif kind == "mixture":
        n = case["n"]
        # pairs of the radii (d_i + d_j) / 2 + skin at this density, without the packing's structure
        volume = (0.01 * 1000.0 + 0.99) * math.pi / 6.0 / case["phi"]
        reach = [4.0 / 3.0 * math.pi * (d + case["skin"]) ** 3 for d in (1.0, 5.5, 10.0)]
        free = [reach[0], max(reach[1] - 4.0 / 3.0 * math.pi * 5.5 ** 3, 0.0), max(reach[2] - 4.0 / 3.0 * math.pi * 1e3, 0.0)]
        mean = 1.0 + (0.99 * 0.99 * free[0] + 2 * 0.99 * 0.01 * free[1] + 0.01 * 0.01 * free[2]) / volume
        mean *= 0.5 if case["half"] else 1.0
    else:
        n = case["n"]
        mean = _mean_neighbors(case)
    pairs = n * mean
    if kind == "raw":
        out = 4 * n + (4 * pairs if case["output"] == "list" else 0)
    else:
        out = 12 * n + (5 if case.get("image", True) else 4) * pairs
    read = 12 * n + 16 * n + (12 * n if kind == "md" else 0)
    return {"bytes": read + out, "flops": 8.0 * pairs}


# ------------------------------------------------------------------------------- exact values
def exact(case, seed):
    """Floating outputs in 64 bits: the displacement of an md step, the boxes of a tree.  The
    other outputs are whole numbers."""
    if case["kind"] == "md":
        ref, pts, L = _md_points(case, seed)
        d = pts.double() - ref.double()
        box = float(torch.tensor(L, dtype=torch.float32))
        d -= box * torch.round(d / box)
        return {"counts": None, "offsets": None, "neigh": None, "image": None, "disp2": (d * d).sum(1).max(), "wrapped": None}
    if case["kind"] != "tree":
        return None
    pts, L = _points(case, seed)
    lo, hi = _exact_boxes(pts, L, 0.25 if case["insert"] == "spheres" else 0.0)
    return {k: None for k in ("parent", "left", "right", "primitive", "rope", "codes")} | {"lo": lo, "hi": hi}


def _codes(pts, L):
    """30-bit Morton codes of 32-bit positions in [0, L)^3 (the definition is in 32 bits)."""
    q = torch.clamp(pts / torch.tensor(L, dtype=torch.float32, device=pts.device) * 1023.0, 0.0, 1023.0).long()
    code = torch.zeros(pts.shape[0], dtype=torch.long, device=pts.device)
    for bit in range(10):
        for axis in range(3):
            code |= ((q[:, axis] >> bit) & 1) << (3 * bit + 2 - axis)
    return code


def _exact_boxes(pts, L, radius):
    """Boxes of the binary radix tree over (Morton code, input order): internal node i covers the
    range of sorted leaves with i at one end, found by bisection; its box by range minima."""
    n = pts.shape[0]
    # a sphere's code is that of its box center, (lo + hi) / 2 in 32 bits
    center = 0.5 * ((pts - radius) + (pts + radius)) if radius else pts
    code, order = torch.sort(_codes(center, L), stable=True)
    leaf_lo, leaf_hi = pts.double()[order] - radius, pts.double()[order] + radius
    if n == 1:
        return leaf_lo, leaf_hi
    key = (code << 32) | torch.arange(n, device=pts.device)     # all different
    i = torch.arange(n - 1, device=pts.device)

    def differ(j):
        """key[i] ^ key[j]: the longer the common prefix, the smaller; past the ends the largest."""
        inside = (j >= 0) & (j < n)
        return torch.where(inside, key[i] ^ key[j.clamp(0, n - 1)], torch.full_like(j, 1 << 62))

    def top_bit(x):
        """Position of the highest set bit of x (0 < x <= 2^62), from 1."""
        high = (x >> 31).double()
        low = (x & ((1 << 31) - 1)).double()
        return torch.where(high > 0, torch.frexp(high)[1].long() + 31, torch.frexp(low)[1].long())

    forward = top_bit(differ(i + 1)) < top_bit(differ(i - 1))
    d = torch.where(forward, 1, -1)
    limit = top_bit(differ(i - d))
    length = torch.zeros_like(i)
    step = 1 << (n - 1).bit_length()
    while step:
        longer = length + step
        j = i + longer * d
        ok = (j >= 0) & (j < n) & (top_bit(differ(j)) < limit)
        length = torch.where(ok, longer, length)
        step >>= 1
    first = torch.where(forward, i, i - length)
    count = length + 1
    level = torch.frexp(count.double())[1].long() - 1           # floor(log2(count))
    lo = torch.empty((n - 1, 3), dtype=torch.float64, device=pts.device)
    hi = torch.empty_like(lo)
    tlo, thi = leaf_lo, leaf_hi                                 # minima of [j, j + 2^k)
    for k in range(int(level.max()) + 1):
        if k:
            half = 1 << (k - 1)
            tlo = torch.minimum(tlo[:-half], tlo[half:])
            thi = torch.maximum(thi[:-half], thi[half:])
        at = torch.nonzero(level == k)[:, 0]
        a, b = first[at], first[at] + count[at] - (1 << k)
        lo[at] = torch.minimum(tlo[a], tlo[b])
        hi[at] = torch.maximum(thi[a], thi[b])
    return torch.cat([lo, leaf_lo]), torch.cat([hi, leaf_hi])
