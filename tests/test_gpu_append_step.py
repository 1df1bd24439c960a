"""bsattn_append_decode where the step's append runs inside the scoring launch:
affine caches (the token quantized there, the summary of the block it fills
folded there) and candidate sets past the selection inside the attention.
Outputs, selected blocks, the stored tokens and the summaries are the same
bytes as bsattn_append + bsattn_decode on a copy, at every step across a block
fill."""
from __future__ import annotations

import pytest

from common import fill, from_dev, log, make_workload, new_cache, to_dev

pytestmark = pytest.mark.gpu

# dtype, Tb, Hq, Hkv, top_k, sink, recent, kv_bits, starting lengths, steps
CASES = {
    # last slots of a block, its fill, and the next block's first slots
    "int4-tb64-g4": ("f16", 64, 16, 4, 3, 1, 1, 4, [64 * 9 - 3, 61, 64 * 4], 6),
    "int4-tb32-g1": ("f16", 32, 2, 2, 2, 0, 2, 4, [32 * 9 - 2, 31, 1], 40),
    "int8-tb64-g2": ("f16", 64, 4, 2, 2, 2, 1, 8, [64 * 6 - 2, 63], 5),
    "int8-tb32-g8": ("f16", 32, 16, 2, 4, 1, 4, 8, [32 * 12 - 2, 29, 32], 5),
    "int8-topk0": ("f16", 32, 4, 2, 0, 1, 2, 8, [32 * 6 - 1, 62], 4),
    # more candidates than the attention selects: MFMA scores (wide groups)
    # or exact scores, and a separate selection
    "int8-tb32-g16-mfma": ("f16", 32, 16, 1, 16, 1, 4, 8, [32 * 2060 - 2, 700], 4),
    "int4-tb32-g2-exact": ("f16", 32, 2, 1, 16, 1, 1, 4, [32 * 2052 - 2, 5], 4),
    "f16-tb32-g8-mfma": ("f16", 32, 8, 1, 9, 0, 1, 0, [32 * 2052 - 2], 4),
    "bf16-tb32-g16-mfma": ("bf16", 32, 16, 1, 9, 0, 1, 0, [32 * 2054 - 2], 4),
    # a selection wider than the attention holds
    "int8-tb32-k300": ("f16", 32, 4, 1, 300, 1, 1, 8, [32 * 320 - 2], 4),
}


@pytest.mark.parametrize("case", list(CASES))
def test_append_in_the_scoring_launch(gpu, case):
    import torch
    from bsattn import _lib
    dtype, Tb, Hq, Hkv, K, ns, nr, bits, lens0, steps = CASES[case]
    log(f"[append step] {case}")
    B = len(lens0)
    w = make_workload(5200 + len(case), B=B, Hq=Hq, Hkv=Hkv, T=max(lens0), Tb=Tb, dtype=dtype, top_k=K, ns=ns,
                      nr=nr, lens=lens0)
    a = new_cache(w, kv_bits=bits, mbps=-(-(max(lens0) + steps) // Tb))
    fill(a, w, gpu)
    b = a.copy()
    a.profile(True)
    q = to_dev(w.q[:, :, None, :], dtype, gpu)
    gen = torch.Generator().manual_seed(len(case))
    for s in range(steps):
        k, v = (torch.randn((B, Hkv, 1, 128), generator=gen).to(q.dtype).to(gpu) for _ in range(2))
        ia = torch.empty((B, Hkv, K + ns + nr), dtype=torch.int32, device=gpu)
        ib = torch.empty_like(ia)
        oa = a.appendDecode(k, v, q, w.scale, idx_out=ia)
        b.append(k, v)
        ob = b.decode(q, w.scale, idx_out=ib)
        torch.cuda.synchronize()
        assert torch.equal(ia, ib), f"step {s}: selected blocks differ"
        assert (from_dev(oa) == from_dev(ob)).all(), f"step {s}: outputs differ"
    # a step is the scoring launch (the append and the summaries inside), the
    # attention, and the selection between them where the attention has none
    separate = case.endswith(("mfma", "exact", "k300"))
    launches = {k: a.profileRead(getattr(_lib, "KERNEL_" + k))[1] for k in ("SCORE", "TOPK", "ATTEND", "APPEND")}
    assert launches == {"SCORE": steps, "TOPK": steps * separate, "ATTEND": steps, "APPEND": 0}
    a.profile(False)
    for i in range(B):
        assert torch.equal(a.exportSummaries(i), b.exportSummaries(i)), f"sequence {i}: summaries differ"
        sa, sb = ((x for t in c.exportQuantized([i]) for x in t) if bits else c.export([i]) for c in (a, b))
        for x, y in zip(sa, sb):
            assert torch.equal(x, y), f"sequence {i}: stored tokens differ"
