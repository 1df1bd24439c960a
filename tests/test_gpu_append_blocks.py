"""Appends and exports of many tokens, which move whole blocks: every split of
a conversation into chunks (inside a block, across its edges, whole blocks;
with and without the pages passed in the launch) stores the same bytes and
summaries, which are the ones that the reference arithmetic of the tests gives
(16-bit: the tokens themselves and their means in token order; quantized: the
oracle's codec), and an append leaves its neighbours' slots alone."""
from __future__ import annotations

import numpy as np
import pytest

from common import from_dev, log, make_workload, new_cache, to_dev
import oracle as O

pytestmark = pytest.mark.gpu

# total tokens, chunk sizes (the last is repeated): around 8-token pieces,
# 32-token segments and blocks; 13000 tokens of 32-token blocks (407 pages)
# take the metadata launch, as the arguments hold 192
CHUNKS = [(1, [1]), (7, [3, 4]), (64, [64]), (65, [65]), (200, [1, 6, 1, 25, 31, 33, 64]), (333, [17, 16, 2, 100]),
          (129, [127, 2]), (13000, [12345, 655])]


def split(total, sizes):
    at, i, out = 0, 0, []
    while at < total:
        n = min(sizes[min(i, len(sizes) - 1)], total - at)
        out.append((at, at + n))
        at, i = at + n, i + 1
    return out


@pytest.mark.parametrize("total,sizes", CHUNKS, ids=[f"{t}-{s[0]}" for t, s in CHUNKS])
@pytest.mark.parametrize("kind", ["f16", "bf16", "int4", "int8"])
@pytest.mark.parametrize("Tb", [32, 64])
def test_append_and_export_blocks(gpu, Tb, kind, total, sizes):
    import torch
    bits = {"int4": 4, "int8": 8}.get(kind, 0)
    dtype = "f16" if bits else kind
    B, Hkv = 2, 2
    log(f"[append blocks] {kind} Tb={Tb} {total} {sizes}")
    lens = [total, total]
    w = make_workload(6100 + total, B=B, Hq=2, Hkv=Hkv, T=total, Tb=Tb, dtype=dtype, top_k=4, lens=lens)
    c = new_cache(w, kv_bits=bits)
    c.shuffleFreePages(total)
    k = to_dev(np.stack(w.keys), dtype, gpu)
    v = to_dev(np.stack(w.values), dtype, gpu)
    for a, b in split(total, sizes):
        c.append(k[:, :, a:b].contiguous(), v[:, :, a:b].contiguous())
    # both sequences at once, and one alone in a second cache through the state
    if not bits:
        ko, vo = c.export([1, 0])
        assert torch.equal(ko, k.flip(0)) and torch.equal(vo, v.flip(0))
    else:
        (kw, ks, kb), (vw, vs, vb) = c.exportQuantized([1, 0])
        for got, src in (((kw, ks, kb), w.keys), ((vw, vs, vb), w.values)):
            for b in range(B):
                for h in range(Hkv):
                    codes, sc, bs = O.quantize(src[1 - b][h], bits, 64)
                    assert np.array_equal(got[0][b, h].cpu().numpy().view(np.uint32), codes)
                    assert np.array_equal(from_dev(got[1][b, h]), sc) and np.array_equal(from_dev(got[2][b, h]), bs)
        other = new_cache(w, kv_bits=bits)
        for a, b in split(total, list(reversed(sizes))):
            cut = [[x[:, :, a:b].flip(0).contiguous() for x in t] for t in ((kw, ks, kb), (vw, vs, vb))]
            other.appendQuantized(*cut)
        for x, y in zip(c.state, other.state):
            assert torch.equal(x, y)
        for b in range(B):
            assert torch.equal(c.exportSummaries(b), other.exportSummaries(b))
    for b in range(B):
        got = from_dev(c.exportSummaries(b))
        for h in range(Hkv):
            want = (O.summaries_q(*O.quantize(w.keys[b][h], bits, 64), Tb, bits, 64) if bits
                    else O.summaries(w.keys[b][h], Tb, dtype))
            assert np.array_equal(got[h], want[:total // Tb])


@pytest.mark.parametrize("kind", ["bf16", "int4", "int8"])
def test_append_after_trim(gpu, kind):
    """Tokens appended over trimmed ones, one at a time and by chunks, read
    back as if the trimmed ones had never been there."""
    import torch
    bits = {"int4": 4, "int8": 8}.get(kind, 0)
    dtype = "f16" if bits else kind
    w = make_workload(6300, B=1, Hq=2, Hkv=2, T=170, Tb=64, dtype=dtype, top_k=2, lens=[170])
    k, v = to_dev(w.keys[0][None], dtype, gpu), to_dev(w.values[0][None], dtype, gpu)
    a, b = new_cache(w, kv_bits=bits), new_cache(w, kv_bits=bits)
    a.append(k, v)
    for at, n in ((61, 5), (66, 1), (67, 103)):
        b.trim(1 << 20, [0])
        b.append(v, k)          # other tokens
        b.trim(170 - at, [0])
        b.trim(at, [0])
        b.append(k[:, :, :at].contiguous(), v[:, :, :at].contiguous())
        b.append(k[:, :, at:at + n].contiguous(), v[:, :, at:at + n].contiguous())
        if at + n < 170:
            b.append(k[:, :, at + n:].contiguous(), v[:, :, at + n:].contiguous())
        for x, y in zip(a.state, b.state):
            assert torch.equal(x, y)
        assert torch.equal(a.exportSummaries(0), b.exportSummaries(0))
