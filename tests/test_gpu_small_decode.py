"""The one-launch decode of small batches: the selection that each wave makes
for itself (up to 256 candidates) against the separate selection kernels, over
sizes around its 64-candidate steps, ties, infinities and NaN; and the split
merge inside the launch against the combine launch (which a profiled call
takes): the same bytes, call after call, with two to more than sixteen splits,
without allocation, and in replayed graphs."""
from __future__ import annotations

import pytest

from common import fill, log, make_workload, new_cache, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("what", ["normal", "ties", "few-values", "inf-nan"])
@pytest.mark.parametrize("blocks", [2, 3, 33, 64, 65, 66, 67, 129, 130, 194, 257, 258, 259, 300])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_selection_per_wave(gpu, dtype, blocks, what):
    import torch
    log(f"[small decode] {dtype} {blocks} blocks {what}")
    for K in (1, 5, blocks - 3, blocks - 2):
        if K < 1:
            continue
        w = make_workload(7000 + blocks, B=1, Hq=8, Hkv=2, T=32 * blocks - 5, Tb=32, dtype=dtype, top_k=K)
        c = new_cache(w)
        td = torch.float16 if dtype == "f16" else torch.bfloat16
        g = torch.Generator().manual_seed(blocks)
        k = torch.randn((1, 2, 32 * blocks - 5, 128), generator=g)
        q = torch.randn((1, 8, 1, 128), generator=g)
        if what == "ties":
            k[:] = k[:, :, :1]
        elif what == "few-values":
            k = torch.randint(0, 2, (1, 2, blocks, 1), generator=g).repeat_interleave(32, 2)[:, :, :32 * blocks - 5].expand_as(k)
        elif what == "inf-nan":
            k[:, 0, 40::97] = float("inf")
            k[:, 1, 50::111] = float("nan")
            k[:, 1, 60::77] = -float("inf")
        k = k.to(td).to(gpu).contiguous()
        c.append(k, torch.randn(k.shape, generator=g).to(td).to(gpu))
        q = q.to(td).to(gpu)
        want = c.selectBlocks(q)
        got = torch.empty_like(want)
        out = c.decode(q, w.scale, idx_out=got)
        torch.cuda.synchronize()
        assert torch.equal(got, want), f"top_k {K}"
        ref = c.attend(q, want, w.scale)
        assert torch.equal(out.view(torch.int16), ref.view(torch.int16)), f"top_k {K}"


# B, Hkv, G, top_k: splits of 4 slots, as many as about 256 workgroups allow
SPLITS = [(1, 8, 4, 8), (1, 2, 2, 3), (1, 1, 4, 30), (2, 1, 1, 62), (1, 1, 4, 66), (3, 8, 4, 14), (6, 8, 1, 30)]


@pytest.mark.parametrize("B,Hkv,G,K", SPLITS, ids=[f"b{b}-h{h}-g{g}-k{k}" for b, h, g, k in SPLITS])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_merge_in_the_launch(gpu, dtype, B, Hkv, G, K):
    import torch
    lens = [64 * 90 - 7 - 300 * b for b in range(B)]
    w = make_workload(7300 + K, B=B, Hq=Hkv * G, Hkv=Hkv, T=max(lens), Tb=64, dtype=dtype, top_k=K, lens=lens)
    c = new_cache(w)
    fill(c, w, gpu)
    q = to_dev(w.q[:, :, None, :], dtype, gpu)
    c.profile(True)
    ref = c.decode(q, w.scale).view(torch.int16)
    c.profile(False)
    out = torch.empty_like(q)
    for n in range(12):
        qn = torch.roll(q, n, 1)
        assert torch.equal(c.decode(q, w.scale).view(torch.int16), ref), f"call {n}"
        c.decode(qn, w.scale)
        c.decodeNoAlloc(q, w.scale, out)
        assert torch.equal(out.view(torch.int16), ref), f"call {n} without allocation"
        if B > 1:  # fewer sequences: other splits on the same counters
            one = c.decode(q[:1].contiguous(), w.scale, seq_ids=[0])
            c.profile(True)
            assert torch.equal(one.view(torch.int16), c.decode(q[:1].contiguous(), w.scale, seq_ids=[0]).view(torch.int16))
            c.profile(False)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        c.decode(q, w.scale)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o = c.decode(q, w.scale)
    for n in range(4):
        o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o.view(torch.int16), ref), f"replay {n}"
        assert torch.equal(c.decode(q, w.scale).view(torch.int16), ref)


@pytest.mark.parametrize("L", [2, 3, 4, 16])
def test_merge_of_a_multi_token_decode(gpu, L):
    """128 workgroups for each query token: up to 1.5 per CU the launch merges
    its splits, with more the combine launch does, as when profiled."""
    import torch
    log(f"[small decode] multi L={L}")
    w = make_workload(7350, B=2, Hq=32, Hkv=8, T=4000, Tb=64, dtype="bf16", top_k=30, lens=[4000, 3700])
    c = new_cache(w)
    fill(c, w, gpu)
    q = torch.randn((2, 32, L, 128), generator=torch.Generator().manual_seed(L)).to(torch.bfloat16).to(gpu)
    c.profile(True)
    ref = c.decodeMulti(q, w.scale)
    c.profile(False)
    for n in range(4):
        assert torch.equal(c.decodeMulti(q, w.scale).view(torch.int16), ref.view(torch.int16)), f"call {n}"
