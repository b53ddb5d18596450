"""v1 decode attention at head_dim 64 and 256 on the matrix cores with split
operands (2-4 bit codes), against the oracle's float64 attention over the same
cache bytes, and the formats around it that stay on the FMA kernel.

Tolerance: operands carry 22 bits (f16 hi + lo), sums are fp32, scores reach
about 2^5 in log2 units: relative 2-norm error below 2^-22 * 2^5 / 2 = 4e-6.
"""
import math

import numpy as np
import pytest
import torch

from oracle import tq_oracle as O

pytestmark = pytest.mark.gpu


def _setup(cuda, d, kb, vb, hkv, lens, vrot, page, seed, kind="rht"):
    from fused_turboquant import v1 as V1
    g = torch.Generator().manual_seed(seed)
    layer = V1.TurboQuantV1Layer(d, kb, vb, v_rotate=vrot, device=cuda, kind=kind)
    pages = [(n + page - 1) // page for n in lens]
    nb = sum(pages) + 2
    perm = torch.randperm(nb, generator=g).to(torch.int32)
    bt = torch.full((len(lens), max(pages)), -1, dtype=torch.int32)
    cache = torch.zeros(layer.kv_cache_shape(nb, page, hkv), dtype=torch.uint8, device=cuda)
    at = 0
    for b, n in enumerate(lens):
        bt[b, :pages[b]] = perm[at:at + pages[b]]
        at += pages[b]
        k, v = torch.randn(n, hkv, d, generator=g), torch.randn(n, hkv, d, generator=g) + 0.25
        k[::41] *= 4.0
        pos = torch.arange(n)
        slots = bt[b].long()[pos // page] * page + pos % page
        layer.store(k.to(torch.bfloat16).to(cuda), v.to(torch.bfloat16).to(cuda), cache, slots.to(cuda))
    return layer, cache, bt.to(cuda), torch.tensor(lens, dtype=torch.int32, device=cuda), g


def _rel(got, want):
    return float(np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want))


@pytest.mark.parametrize("d,kb,vb,hkv,G,lens,vrot,page,splits,start,kind", [
    (64, 4, 4, 2, 4, (33, 1, 130), False, 16, None, None, "rht"),     # tile edges, a single position
    (64, 3, 3, 1, 8, (500,), True, 32, 3, None, "rht"),               # codes that start inside a 16-bit unit
    (64, 2, 3, 2, 9, (70, 64), False, 16, 1, None, "rht"),            # more than 8 heads, output by the kernel
    (64, 4, 2, 1, 16, (257,), True, 16, 2, (40,), "rht"),             # a start inside a tile
    (64, 2, 2, 2, 1, (31, 32), True, 64, 1, (0, 32), "rht"),          # an empty range
    (64, 3, 4, 1, 5, (200,), True, 16, 1, None, "planar"),            # matrix rotation, through the merge
    (256, 4, 4, 2, 2, (33, 1, 130), True, 16, None, None, "rht"),
    (256, 3, 3, 1, 8, (400,), False, 32, 4, None, "rht"),
    (256, 2, 4, 1, 12, (97,), True, 16, 1, (5,), "rht"),
    (256, 4, 2, 2, 3, (64, 65), False, 16, 2, None, "rht"),
    (256, 3, 2, 1, 4, (150,), True, 16, 1, None, "iso_full"),
])
def test_split_operands_match_oracle(cuda, d, kb, vb, hkv, G, lens, vrot, page, splits, start, kind):
    layer, cache, bt, sl, g = _setup(cuda, d, kb, vb, hkv, lens, vrot, page, seed=d + 8 * kb + vb + G, kind=kind)
    B = len(lens)
    q = torch.randn(B, hkv * G, d, generator=g)
    q[:, 0] *= 100.0  # heads of very different magnitude
    ks = None if start is None else torch.tensor(start, dtype=torch.int32, device=cuda)
    lse = torch.empty(B, hkv * G, device=cuda)
    got = layer.decode(q.to(cuda), cache, bt, sl, num_splits=splits, kv_start=ks, lse=lse, max_seq_len=max(lens)).cpu().numpy()
    rot = None if layer.rotation is None else layer.rotation.cpu().numpy()
    args = (cache.cpu().numpy(), bt.cpu().numpy(), np.array(lens), layer.centroids.cpu().numpy(), kb, vb, 1 / math.sqrt(d))
    kw = dict(kv_start=None if start is None else np.array(start), v_rotate=vrot, rotation=rot)
    want = O.v1_decode_attention(q.numpy(), *args, **kw)
    err = _rel(got[:, 1:] if hkv * G > 1 else got, want[:, 1:] if hkv * G > 1 else want)
    print(f"[split d{d} K{kb}V{vb} G{G} splits {splits}] rel {err:.2e}", flush=True)
    assert np.isfinite(got).all() and err < 4e-6
    assert _rel(got, want) < 2e-4  # the large head: scores near 2^11, so 2^6 the error
    empty = [b for b, n in enumerate(lens) if start is not None and start[b] >= n]
    assert all((got[b] == 0).all() and torch.isneginf(lse[b]).all() for b in empty)


def test_positions_without_a_page_and_bad_scales(cuda):
    """Entries of -1 or past num_blocks hide their positions; infinite fields of
    positions past the sequence do not reach the output."""
    layer, cache, bt, sl, g = _setup(cuda, 64, 4, 4, 1, (100,), False, 16, seed=9)
    q = torch.randn(1, 4, 64, generator=g).to(cuda)
    want = layer.decode(q, cache, bt, sl, operands="fp32")
    raw = cache.view(-1, cache.shape[2] * cache.shape[3])
    blk = int(bt[0, 6])
    cache[blk, 4:, :, 66:70] = torch.tensor([0, 0x7c, 0, 0x7c], dtype=torch.uint8, device=cuda)  # positions 100 .. 111
    del raw
    assert _rel(layer.decode(q, cache, bt, sl).cpu().numpy(), want.cpu().double().numpy()) < 4e-6
    bt2 = bt.clone()
    bt2[0, 1], bt2[0, 4] = -1, cache.shape[0] + 3
    a, b = layer.decode(q, cache, bt2, sl), layer.decode(q, cache, bt2, sl, operands="fp32")
    assert _rel(a.cpu().numpy(), b.cpu().double().numpy()) < 4e-6
