"""Split prefills of many caches share a few workspaces: calls of several
streams and threads under way at once, and one captured among them, give the
bits of each call by itself; a model's layer caches hold one between them."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from common import log, make_workload, new_cache, to_dev
import oracle as O

pytestmark = pytest.mark.gpu


def _caches(gpu, n, T):
    import torch
    out = []
    for i in range(n):
        w = make_workload(8600 + i, B=1, Hq=32, Hkv=8, T=T, Tb=64, dtype="bf16", top_k=4)
        c = new_cache(w)
        c.append(to_dev(w.keys[0][None], "bf16", gpu), to_dev(w.values[0][None], "bf16", gpu))
        q = to_dev(O.fill_normal(8650 + i, 0, 0, (1, 32, 64, 128), "bf16"), "bf16", gpu)
        out.append((c, q, w.scale))
    torch.cuda.synchronize()
    return out


def test_split_prefills_on_several_streams(gpu):
    import torch
    log("[prefill streams]")
    caches = _caches(gpu, 6, 1500)
    want = []
    for c, q, scale in caches:
        want.append(c.prefill(q, scale))
        torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(6)]
    for n in range(5):
        got = [None] * 6
        for i, (c, q, scale) in enumerate(caches):
            with torch.cuda.stream(streams[(i + n) % 6]):
                for _ in range(4):
                    got[i] = c.prefill(q, scale)
        torch.cuda.synchronize()
        for i in range(6):
            assert torch.equal(got[i], want[i]), f"round {n} cache {i}"
    # threads
    bad = []

    def work(i):
        c, q, scale = caches[i]
        with torch.cuda.stream(streams[i]):
            for _ in range(20):
                o = c.prefill(q, scale)
            streams[i].synchronize()
            if not torch.equal(o, want[i]):
                bad.append(i)
            streams[i].synchronize()

    th = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    # a captured call keeps its own workspace: replays beside eager calls
    c, q, scale = caches[0]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = c.prefill(q, scale)
    for n in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        with torch.cuda.stream(streams[1]):
            got = caches[1][0].prefill(caches[1][1], caches[1][2])
        torch.cuda.synchronize()
        assert torch.equal(out, want[0]) and torch.equal(got, want[1]), f"replay {n}"


def test_layers_share_a_workspace(gpu):
    import torch
    log("[prefill streams] memory")
    caches = _caches(gpu, 8, 1500)
    outs = [torch.empty_like(q) for _, q, _ in caches]
    free = torch.cuda.mem_get_info()[0]
    for (c, q, scale), o in zip(caches, outs):
        o.copy_(c.prefill(q, scale))
    torch.cuda.synchronize()
    held = free - torch.cuda.mem_get_info()[0]
    assert held <= 100 << 20, f"{held >> 20} MiB for 8 caches"
    assert all(np.isfinite(o.float().cpu().numpy()).all() for o in outs)


def test_the_merge_is_timed(gpu):
    """A profiled split prefill: its merge is a combine launch of its own."""
    import torch
    from bsattn import _lib
    log("[prefill streams] profile")
    (c, q, scale), = _caches(gpu, 1, 1500)
    want = c.prefill(q, scale)
    c.profile(True)
    for _ in range(3):
        assert torch.equal(c.prefill(q, scale), want)
    for kind in (_lib.KERNEL_PREFILL, _lib.KERNEL_COMBINE):
        ms, n = c.profileRead(kind)
        assert n == 3 and ms > 0.0
    c.profile(False)
    assert torch.equal(c.prefill(q, scale), want)
