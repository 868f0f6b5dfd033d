"""One traverser's unordered queries, which it sorts in workspaces of its own, from several host
threads and streams (template API, tests/device/shared_traverser.hip): counts equal those in the
tree's order."""
from __future__ import annotations

import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EXE = os.path.join(ROOT, "tests", "device", "shared_traverser.bin")


def run(mode):
    print(f"shared traverser: {mode}", flush=True)
    r = subprocess.run([EXE, mode], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr


def test_threads_on_their_own_streams():
    """Two threads on hipStreamPerThread: one handle value, two streams."""
    run("threads")


def test_no_memory_for_the_sort():
    """Any of the workspaces' allocations may fail: the call is served unsorted, the next one right."""
    run("memory")


def test_beside_a_capture():
    """Workspaces made and grown while another thread captures in global mode."""
    run("capture")


def test_unordered_under_capture():
    """Unordered queries captured in a graph (not sorted there), replayed with eager calls between."""
    import torch
    import neighbor_amd as nb
    n = 50000
    rng = np.random.default_rng(23)
    L = float(np.float32((n / 0.85) ** (1.0 / 3.0)))
    pts = torch.from_numpy((rng.random((n, 3)) * L).astype(np.float32)).cuda()
    lb = nb.LBVH()
    lb.build(pts, [0, 0, 0], [L] * 3)
    tr = nb.LBVHTraverser()
    tr.setup(lb)
    sets = [torch.cat([pts, torch.full((n, 1), r, device="cuda")], 1).contiguous() for r in (1.1, 1.4, 0.9)]
    want = [tr.count(lb, s, order=lb.device_pointers()["primitive"]) for s in sets]
    sph, out = sets[0].clone(), torch.zeros(n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        tr.count(lb, sph, nneigh=out, stream=stream)
    for s, w in zip(sets, want):
        sph.copy_(s)
        out.zero_()
        graph.replay()
        assert torch.equal(tr.count(lb, sph), w)
        torch.cuda.synchronize()
        assert torch.equal(out, w)


def test_streams_across_the_sorts_limits():
    """Two streams and numbers of queries on both sides of the sorts' limits, in turn."""
    import torch
    import neighbor_amd as nb
    n = 400001
    rng = np.random.default_rng(21)
    L = float(np.float32((n / 0.85) ** (1.0 / 3.0)))
    pts = torch.from_numpy((rng.random((n, 3)) * L).astype(np.float32)).cuda()
    lb = nb.LBVH()
    lb.build(pts, [0, 0, 0], [L] * 3)
    sph = torch.cat([pts, torch.full((n, 1), 1.2, device="cuda")], 1).contiguous()
    want = nb.LBVHTraverser().count(lb, sph, order=lb.device_pointers()["primitive"])
    tr = nb.LBVHTraverser()
    tr.setup(lb)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    sizes = [2000, 20000, 400000, 30000, 16384, 16385, 393216, 393217]
    outs = []
    for i in range(16):
        s = streams[i % 2]
        with torch.cuda.stream(s):
            outs.append((sizes[i % 8], tr.count(lb, sph[:sizes[i % 8]], stream=s)))
    torch.cuda.synchronize()
    for m, got in outs:
        assert torch.equal(got, want[:m]), m


def test_long_codes():
    """More unordered queries than 16-bit codes serve: three digit passes."""
    import torch
    import neighbor_amd as nb
    n, nq = 5000, (1 << 20) + 1
    rng = np.random.default_rng(22)
    pts = torch.from_numpy(rng.random((n, 3)).astype(np.float32) * 18.0).cuda()
    lb = nb.LBVH()
    lb.build(pts, [0, 0, 0], [18.0] * 3)
    gen = torch.Generator(device="cuda").manual_seed(5)
    sph = torch.rand((nq, 4), generator=gen, device="cuda") * torch.tensor([18.0, 18.0, 18.0, 0.9], device="cuda")
    tr = nb.LBVHTraverser()
    tr.setup(lb)
    got = tr.count(lb, sph)
    want = torch.cat([tr.count(lb, sph[i:i + (1 << 18)].contiguous()) for i in range(0, nq, 1 << 18)])
    assert torch.equal(got, want)
