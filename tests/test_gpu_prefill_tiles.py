"""Prefill attention at the edges of its workgroup tiles (8 waves x 32
columns: 256 / G query tokens), of its parts (a short chunk's tokens are
split over the chip and merged) and past the 64 blocks whose pages a wave
holds at a time; and the split prefill inside a captured graph."""
from __future__ import annotations

import numpy as np
import pytest

from common import log, make_workload, new_cache, to_dev
import oracle as O
from test_gpu_prefill import TOL, _check, _run, ulp, test_prefill_quantized_cache as check_quantized

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,Hq,Hkv,Tb,lens,L", [
    ("f16", 32, 8, 64, [4700, 4129], 64),     # a whole tile; 74 blocks
    ("bf16", 32, 8, 32, [2500], 65),          # one token more than a tile; 79 blocks
    ("f16", 64, 4, 64, [4500, 4230, 4353, 4416], 256),  # 256 tiles: not split; 71 blocks
    ("bf16", 8, 8, 64, [255], 255),           # one token less than a tile, from an empty cache
    ("f16", 16, 2, 32, [33], 32),             # one token before the chunk
    ("bf16", 32, 8, 64, [97, 33], 33),        # half tiles of 32 tokens: one token more
    ("f16", 64, 4, 64, [200], 71),            # half tiles of 8 tokens: one token less
    # split with a sequence of fewer units than parts, in whole tiles and in half ones
    ("bf16", 32, 8, 64, [4700, 40, 65], 33),
    ("f16", 8, 2, 32, [20, 2000], 20),
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


@pytest.mark.parametrize("dtype,units,big", [
    ("f16", 1, ()), ("bf16", 2, ()), ("f16", 3, ()), ("bf16", 4, (3,)), ("bf16", 5, (1, 2)),
    ("bf16", 11, (2, 3, 7)), ("f16", 12, ()),
])
def test_prefill_unit_counts(gpu, dtype, units, big):
    """Prefills of a few 32-token units (the waves meet after every second
    one), odd and even; `big` units hold bf16 values that fp16 cannot, so
    that the steps leave their pairs at odd and even units."""
    log(f"[prefill units] {dtype} {units} {big}")
    L, T = 20, 32 * units - 3
    w = make_workload(8300 + units, B=1, Hq=32, Hkv=8, T=T, Tb=32, dtype=dtype, top_k=4)
    v = O.to_f32(w.values[0], dtype)
    for u in big:
        v[:, 32 * u + 5, :] *= 2.0 ** 17
    w.values[0] = O.from_f32(v, dtype)
    got, qm, _ = _run(w, gpu, L)
    # the error of sum_i p_i v_i scales with sum_i p_i |v_i| (each product and
    # weight is rounded on its own), which the oracle's dense attention over
    # |V| gives: TOL of that, and of 1 where it is smaller
    for i in (0, 1, L // 2, L - 1):
        for h in range(w.Hkv):
            qh, kh, vh = qm[0, h * w.G:(h + 1) * w.G, i], w.keys[0][h][:T - L + i + 1], w.values[0][h][:T - L + i + 1]
            ref = O.dense(qh, kh, vh, w.scale, dtype)
            mag = O.dense(qh, kh, vh & np.uint16(0x7FFF), w.scale, dtype)
            a = O.to_f32(got[0, h * w.G:(h + 1) * w.G, i], dtype).astype(np.float64)
            err = float(np.max((np.abs(a - ref) - 0.5 * ulp(ref, dtype)) / np.maximum(1.0, mag)))
            assert err <= TOL, f"query {i} head {h}: relative error {err:.3g}"


@pytest.mark.parametrize("dtype,bits,Hq,Hkv,Tb", [
    ("f16", 0, 32, 8, 64), ("bf16", 0, 32, 8, 32), ("f16", 4, 32, 8, 64), ("f16", 8, 64, 4, 32), ("bf16", 0, 8, 8, 64),
])
def test_prefill_widths(gpu, dtype, bits, Hq, Hkv, Tb):
    """Many sequences in a call take workgroups of 8 waves, one alone those of
    4 (neither is split): the same bits, at every count of units up to 13."""
    import torch
    log(f"[prefill widths] {dtype} int{bits} Hq={Hq} Hkv={Hkv} Tb={Tb}")
    L, B = 40, 40
    lens = [L + 9 * b for b in range(B)]
    w = make_workload(8400 + bits + Hq, B=B, Hq=Hq, Hkv=Hkv, T=max(lens), Tb=Tb, dtype=dtype, top_k=4, lens=lens)
    c = new_cache(w, kv_bits=bits)
    for b in range(B):
        v = to_dev(w.values[b][None], dtype, gpu)
        if dtype == "bf16" and b % 3 == 1:
            v[:, :, 7::29] *= 2.0 ** 17  # (beyond fp16)
        c.append(to_dev(w.keys[b][None], dtype, gpu), v, seq_ids=[b])
    q = to_dev(O.fill_normal(w.seed + 1, 0, 0, (B, Hq, L, 128), dtype), dtype, gpu)
    together = c.prefill(q, w.scale)
    for b in range(B):
        alone = c.prefill(q[b:b + 1].contiguous(), w.scale, seq_ids=[b])
        assert torch.equal(together[b], alone[0]), f"{lens[b]} tokens"
    assert torch.isfinite(together.float()).all()


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


@pytest.mark.parametrize("dtype,bits,Hq,Hkv,Tb,T,L", [
    ("f16", 0, 32, 8, 64, 200, 150),    # half tiles
    ("bf16", 0, 32, 8, 32, 130, 130),
    ("f16", 8, 64, 4, 32, 300, 200),
    ("f16", 4, 32, 8, 64, 900, 300),
    ("bf16", 0, 32, 8, 64, 4500, 200),  # split
    ("f16", 0, 8, 8, 64, 2100, 2000),   # whole tiles of 256 tokens
    ("bf16", 0, 8, 8, 64, 2100, 2000),
])
def test_prefill_values_that_are_not_finite(gpu, dtype, bits, Hq, Hkv, Tb, T, L):
    """An infinity or NaN in a token's V reaches the queries that see the token,
    in its dim and head, and no other output: those are the bits of a cache
    with a finite value there."""
    import torch
    log(f"[prefill not finite] {dtype} int{bits} Hq={Hq} Hkv={Hkv} Tb={Tb} T={T} L={L}")
    w = make_workload(8500 + T + Hq, B=1, Hq=Hq, Hkv=Hkv, T=T, Tb=Tb, dtype=dtype, top_k=4)
    G = Hq // Hkv
    k, v = to_dev(w.keys[0][None], dtype, gpu), to_dev(w.values[0][None], dtype, gpu)
    q = to_dev(O.fill_normal(w.seed + 1, 0, 0, (1, Hq, L, 128), dtype), dtype, gpu)
    inf, nan = float("inf"), float("nan")
    odd = [(T - L + 3, 0, 5, inf), (T - L // 2, 0, 70, nan), (T - 9, Hkv - 1, 127, -inf), (T - 1, 1, 64, inf)]
    caches = []
    for bad in (False, True):
        c = new_cache(w, kv_bits=bits)
        if bits:  # the whole 64-dim group of the token: V = scale * code + bias
            src = new_cache(w, kv_bits=bits)
            src.append(k, v)
            kq, vq = src.exportQuantized([0])
            if bad:
                for pos, h, d, x in odd:
                    vq[2][0, h, pos, d // 64] = x
            c.appendQuantized(kq, vq)
        else:
            vb = v.clone()
            if bad:
                for pos, h, d, x in odd:
                    vb[0, h, pos, d] = x
            c.append(k, vb)
        caches.append(c)
    good, got = (c.prefill(q, w.scale)[0].float() for c in caches)
    hit = torch.zeros_like(good, dtype=torch.bool)
    for pos, h, d, x in odd:
        dims = slice(d // 64 * 64, d // 64 * 64 + 64) if bits else slice(d, d + 1)
        seen = got[h * G:(h + 1) * G, max(0, pos - (T - L)):, dims]
        assert bool(torch.isnan(seen).all() if x != x else (seen == x).all()), f"token {pos}: its queries"
        hit[h * G:(h + 1) * G, max(0, pos - (T - L)):, dims] = True
    assert torch.isfinite(good).all()
    assert torch.equal(got[~hit], good[~hit]), f"{int((got[~hit] != good[~hit]).sum())} outputs differ"
