"""Output ops of a program's own (template API, tests/device/custom_output.hip) against the oracle:
set up and finalized once per query whatever lanes walk for it, hits handed to their process()."""
from __future__ import annotations

import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "tests", "device", "custom_output.bin")
QUANTIZED, FLOAT_ROPE, WAVE, WAVE_QUANTIZED = 0, 1, 3, 4


def log(msg):
    print(msg, flush=True)


@pytest.fixture(scope="module")
def orc():
    import oracle
    return oracle


def run(mode, tmp_path, pts, sph, imgs, L, variant, order, exact, bucket=16, starts=None):
    head = np.array([len(pts), len(sph), variant, bucket, 2 if isinstance(order, np.ndarray) else order, len(imgs), int(exact)], np.uint32)
    src, dst = str(tmp_path / "in"), str(tmp_path / "out")
    with open(src, "wb") as f:
        for a in (head, np.float32(L), pts.astype(np.float32), sph.astype(np.float32), imgs.astype(np.float64)):
            f.write(np.ascontiguousarray(a).tobytes())
        if isinstance(order, np.ndarray):
            f.write(order.astype(np.uint32).tobytes())
        if starts is not None:
            f.write(starts.astype(np.uint64).tobytes())
    r = subprocess.run([EXE, mode, src, dst], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    return np.fromfile(dst, np.uint32)


def hits(orc, pts, sph, imgs, L, exact):
    """(query, primitive, image) of the oracle's hits."""
    if exact:
        if len(pts) < 3000:
            ref = orc.exact_bruteforce(pts, sph, imgs)
        else:
            ref = orc.exact_celllist(pts, sph, [L] * 3, float(sph[0, 3]), pairs=True)
        return np.repeat(np.arange(len(sph)), ref["counts"].astype(np.int64)), ref["j"].astype(np.int64), ref["k"].astype(np.int64)
    tree = orc.build(pts, [0, 0, 0], [L] * 3)
    ref = orc.traverse(len(pts), orc.compress(tree), sph, imgs.astype(np.float32), triplets=True)
    return np.repeat(np.arange(len(sph)), ref["counts"].astype(np.int64)), ref["prim"].astype(np.int64), ref["image"].astype(np.int64)


# 70,001 queries: split blocks, whose waves have lanes without a query; 40,000: more nodes than the
# trees in which scattered queries still walk together
@pytest.mark.parametrize("variant,exact", [(QUANTIZED, False), (FLOAT_ROPE, False), (WAVE_QUANTIZED, False), (WAVE, True), (QUANTIZED, True)])
@pytest.mark.parametrize("n,order", [(37, 0), (1000, 0), (70001, 1), (40000, 2)])
def test_set_up_once(orc, tmp_path, n, order, variant, exact):
    from neighbor_amd.workloads import images27
    log(f"own output op: n={n} order={order} variant={variant} exact={exact}")
    rng = np.random.default_rng(n)
    L = float(np.float32((n / 0.85) ** (1.0 / 3.0)))
    pts = (rng.random((n, 3)) * L).astype(np.float32)
    pts[pts >= np.float32(L)] = 0.0
    sph = np.concatenate([pts, np.full((n, 1), 1.2)], 1).astype(np.float32)
    imgs = images27(L, dtype=np.float64)
    perm = rng.permutation(n).astype(np.uint32) if order == 2 else order
    got = run("log", tmp_path, pts, sph, imgs, L, variant, perm, exact).reshape(3, n)
    i, j, k = hits(orc, pts, sph, imgs, L, exact)
    want = np.bincount(i, weights=31.0 * j + 7.0 * k + 1.0, minlength=n).astype(np.int64)
    assert (got[1] == 1).all() and (got[2] == 1).all()
    assert np.array_equal(got[0].astype(np.int64), want % (1 << 32))


@pytest.mark.parametrize("variant,exact", [(QUANTIZED, False), (FLOAT_ROPE, True), (WAVE_QUANTIZED, False), (WAVE, True)])
@pytest.mark.parametrize("n,order", [(50, 0), (2000, 0), (70001, 1)])
def test_derived_rows(orc, tmp_path, n, order, variant, exact):
    """An op derived from the library's pair rows that keeps some of the hits."""
    from neighbor_amd.workloads import images27
    log(f"derived pair rows: n={n} order={order} variant={variant} exact={exact}")
    rng = np.random.default_rng(n + 1)
    L = float(np.float32((n / 0.85) ** (1.0 / 3.0)))
    pts = (rng.random((n, 3)) * L).astype(np.float32)
    pts[pts >= np.float32(L)] = 0.0
    sph = np.concatenate([pts, np.full((n, 1), 1.1)], 1).astype(np.float32)
    imgs = images27(L, dtype=np.float64)
    i, j, _ = hits(orc, pts, sph, imgs, L, exact)
    keep = j >= i
    counts = np.bincount(i[keep], minlength=n)
    starts = np.concatenate([[0], np.cumsum(counts)])
    got = run("half", tmp_path, pts, sph, imgs, L, variant, order, exact, starts=starts)
    assert np.array_equal(got[:n].astype(np.int64), counts)
    rows = np.repeat(np.arange(n), counts)
    pairs = got[n:].astype(np.int64)
    assert np.array_equal(pairs[np.lexsort((pairs, rows))], j[keep][np.lexsort((j[keep], i[keep]))])
