"""Prefill attention at the edges of its workgroup tiles (8 waves x 32
columns: 256 / G query tokens), of its parts (a short chunk's tokens are
split over the chip and merged) and past the 64 blocks whose pages a wave
holds at a time; and the split prefill inside a captured graph."""
from __future__ import annotations

import numpy as np
import pytest

from common import log, make_workload, new_cache, to_dev
import oracle as O
from test_gpu_prefill import _check, _run, test_prefill_quantized_cache as check_quantized

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,Hq,Hkv,Tb,lens,L", [
    ("f16", 32, 8, 64, [4700, 4129], 64),     # a whole tile; 74 blocks
    ("bf16", 32, 8, 32, [2500], 65),          # one token more than a tile; 79 blocks
    ("f16", 64, 4, 64, [4500, 4230, 4353, 4416], 256),  # 256 tiles: not split; 71 blocks
    ("bf16", 8, 8, 64, [255], 255),           # one token less than a tile, from an empty cache
    ("f16", 16, 2, 32, [33], 32),             # one token before the chunk
])
def test_prefill_tile_edges(gpu, dtype, Hq, Hkv, Tb, lens, L):
    log(f"[prefill tiles] {dtype} Hq={Hq} Hkv={Hkv} Tb={Tb} lens={lens} L={L}")
    w = make_workload(8100 + Hq + Tb + L, B=len(lens), Hq=Hq, Hkv=Hkv, T=max(lens), Tb=Tb, dtype=dtype,
                      top_k=4, lens=lens, salient_frac=0.01)
    got, qm, _ = _run(w, gpu, L)
    _check(w, got, qm, L, sorted({0, 1, L // 2, L - 2, L - 1}))


@pytest.mark.parametrize("bits,Hq,Hkv,Tb,lens,L", [
    (4, 32, 8, 64, [4700], 63),
    (8, 64, 4, 32, [2200, 2117], 17),
])
def test_prefill_tile_edges_quantized(gpu, bits, Hq, Hkv, Tb, lens, L):
    check_quantized(gpu, bits, Hq, Hkv, Tb, lens, L)


def test_split_prefill_in_a_graph(gpu):
    """A cache's first split prefill under capture: its workspace is had
    there, and every replay equals the eager call."""
    import torch
    log("[prefill tiles] graph")
    L, T = 40, 900
    w = make_workload(8200, B=1, Hq=32, Hkv=8, T=T, Tb=64, dtype="bf16", top_k=4)
    a, b = new_cache(w), new_cache(w)
    for c in (a, b):
        c.append(to_dev(w.keys[0][None], "bf16", gpu), to_dev(w.values[0][None], "bf16", gpu))
    q = to_dev(O.fill_normal(8201, 0, 0, (1, 32, L, 128), "bf16"), "bf16", gpu)
    want = a.prefill(q, w.scale)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = b.prefill(q, w.scale)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(a.prefill(q, w.scale), want)
        torch.cuda.synchronize()
    assert np.isfinite(want.float().cpu().numpy()).all()
