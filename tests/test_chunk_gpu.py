"""Chunk attention (``v1_chunk_attention``): n consecutive query tokens of one
sequence over its stored slots, against the oracle's float64 attention over
the same cache bytes with one row per query token.

Sizes sit where the kernels can go wrong: columns (n x group) around the 64- /
128-column workgroups, contexts around the 32- / 64-token tiles, windows whose
edge falls inside a tile, several splits, several segments.

Tolerances: fp32 outputs.  Formats whose decode runs fp32 products carry every
operand as f16 hi + lo (2^-22) with fp32 sums, so the relative error stays
below 1e-5; the d = 128, 2-4 bit formats carry K as f16 table values, whose
relative error is at most 2^-11 per score term (5e-4 on the outputs).
"""
import math

import numpy as np
import pytest
import torch

from oracle import tq_oracle as O

RAW = 16


def _case(cuda, d, kb, vb, hkv, L, vrot, page, seed, key_fp8=False, kind="rht"):
    from fused_turboquant import raw as R, v1 as V1
    g = torch.Generator().manual_seed(seed)
    pages = (L + page - 1) // page
    nb = pages + 3
    row = torch.randperm(nb, generator=g)[:pages].to(torch.int32)
    k = torch.randn(L, hkv, d, generator=g)
    k[:: 37] *= 6.0  # outlier keys
    v = torch.randn(L, hkv, d, generator=g) + 0.5
    pos = torch.arange(L)
    slots = (row.long()[pos // page] * page + pos % page).to(cuda)
    kd, vd = k.to(torch.bfloat16).to(cuda), v.to(torch.bfloat16).to(cuda)
    if kb == RAW:
        cache = torch.zeros(nb, page, hkv, 4 * d, dtype=torch.uint8, device=cuda)
        R.raw_store(kd, vd, cache, slots)
        return None, cache, row.to(cuda)
    layer = V1.TurboQuantV1Layer(d, kb, vb, v_rotate=vrot, device=cuda, key_fp8=key_fp8, kind=kind)
    cache = torch.zeros(layer.kv_cache_shape(nb, page, hkv), dtype=torch.uint8, device=cuda)
    layer.store(kd, vd, cache, slots)
    return layer, cache, row.to(cuda)


def _chunk(layer, q, cache, row, past, kb, vb, vrot, window=None, key_fp8=False):
    from fused_turboquant import v1 as V1
    cent = None if layer is None or key_fp8 else layer.centroids
    return V1.v1_chunk_attention(q, cache, row, past, cent, kb, vb, 1 / math.sqrt(q.shape[2]), v_rotate=vrot,
                                 window=window, rotation=None if layer is None else layer.rotation, key_fp8=key_fp8)


def _want(layer, q, cache, row, past, kb, vb, vrot, window=None, key_fp8=False):
    n, _, d = q.shape
    sl = np.arange(past + 1, past + n + 1)
    ks = np.maximum(sl - window, 0) if window else None
    bt = np.broadcast_to(row.cpu().numpy(), (n, row.numel()))
    c, qn = cache.cpu().numpy(), q.float().cpu().numpy()
    if layer is None:
        return O.raw_decode_attention(qn, c, bt, sl, 1 / math.sqrt(d), kv_start=ks)
    rot = None if layer.rotation is None else layer.rotation.cpu().numpy()
    return O.v1_decode_attention(qn, c, bt, sl, None if key_fp8 else layer.centroids.cpu().numpy(), kb, vb,
                                 1 / math.sqrt(d), kv_start=ks, v_rotate=vrot, rotation=rot, key_fp8=key_fp8)


def _rel(got, want):
    return float(np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want))


CASES = [
    # d, kb, vb, hkv, G, n, past, vrot, window, page, fp8, kind
    (128, 4, 4, 2, 4, 33, 31, False, None, 16, False, "rht"),     # one column over a workgroup, a tile edge
    (128, 3, 3, 2, 7, 19, 200, True, None, 32, False, "rht"),     # a group that does not divide the columns
    (128, 4, 2, 1, 8, 16, 1500, True, None, 16, False, "rht"),    # one workgroup: split over the context
    (128, 2, 4, 2, 4, 70, 300, False, 100, 16, False, "rht"),     # window edges inside tiles
    (128, 3, 4, 1, 1, 200, 0, True, 64, 16, False, "rht"),        # no past, one head per kv head
    (128, 4, 4, 2, 4, 40, 90, True, None, 16, False, "planar"),   # matrix un-rotation (through the merge)
    (64, 4, 4, 2, 4, 33, 63, False, None, 16, False, "rht"),
    (64, 3, 2, 1, 16, 9, 700, True, 130, 64, False, "rht"),
    (256, 4, 3, 2, 2, 33, 95, True, None, 16, False, "rht"),
    (256, 2, 2, 1, 5, 14, 640, False, 33, 16, False, "rht"),
    (128, 1, 1, 2, 4, 20, 77, True, None, 16, False, "rht"),
    (128, 8, 8, 1, 4, 20, 77, False, None, 16, False, "rht"),
    (64, 8, 8, 1, 4, 20, 77, True, None, 16, True, "rht"),        # fp8 keys
    (64, RAW, RAW, 2, 4, 20, 77, False, None, 16, False, "rht"),  # raw fp16 slots
    (128, RAW, RAW, 2, 8, 20, 300, False, 50, 16, False, "rht"),
    (256, RAW, RAW, 1, 2, 40, 77, False, None, 16, False, "rht"),
]


@pytest.mark.gpu
@pytest.mark.parametrize("d,kb,vb,hkv,G,n,past,vrot,window,page,fp8,kind", CASES)
def test_chunk_matches_oracle(cuda, d, kb, vb, hkv, G, n, past, vrot, window, page, fp8, kind):
    layer, cache, row = _case(cuda, d, kb, vb, hkv, past + n, vrot, page, seed=n + past, key_fp8=fp8, kind=kind)
    q = torch.randn(n, hkv * G, d, generator=torch.Generator().manual_seed(1)).to(cuda)
    got = _chunk(layer, q, cache, row, past, kb, vb, vrot, window, fp8).cpu().numpy()
    want = _want(layer, q, cache, row, past, kb, vb, vrot, window, fp8)
    f16_keys = d == 128 and kb in (2, 3, 4)
    err = _rel(got, want)
    print(f"[chunk d{d} k{kb}v{vb} G{G} n{n} past{past} w{window}] rel {err:.2e}", flush=True)
    assert np.isfinite(got).all() and err < (5e-4 if f16_keys else 1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_chunk_16bit_queries_and_outputs(cuda, dtype):
    layer, cache, row = _case(cuda, 64, 4, 4, 2, 150, True, 16, seed=3)
    q = torch.randn(40, 8, 64, generator=torch.Generator().manual_seed(1)).to(dtype).to(cuda)
    got = _chunk(layer, q, cache, row, 110, 4, 4, True)
    assert got.dtype == dtype
    want = _want(layer, q, cache, row, 110, 4, 4, True)
    # one rounding to the output type, at most half a unit in the last place
    assert _rel(got.float().cpu().numpy(), want) < (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)


@pytest.mark.gpu
def test_chunk_skips_positions_without_a_page(cuda):
    """A block-table entry of -1 (or past num_blocks) hides its positions."""
    layer, cache, row = _case(cuda, 64, 3, 3, 2, 160, False, 16, seed=4)
    q = torch.randn(32, 8, 64, generator=torch.Generator().manual_seed(1)).to(cuda)
    row = row.clone()
    row[2], row[5] = -1, cache.shape[0] + 7
    got = _chunk(layer, q, cache, row, 128, 3, 3, False).cpu().numpy()
    syn = torch.arange(129, 161, dtype=torch.int32, device=cuda)
    want = layer.decode(q, cache, row[None].expand(32, -1).contiguous(), syn, max_seq_len=160).cpu().numpy()
    assert _rel(got, want) < 1e-5


@pytest.mark.gpu
def test_chunk_several_segments(cuda):
    """A context whose dequantised fragments exceed one workspace segment."""
    d, hkv, n, past = 256, 16, 16, 12000
    layer, cache, row = _case(cuda, d, 2, 2, hkv, past + n, True, 16, seed=5)
    q = torch.randn(n, hkv, d, generator=torch.Generator().manual_seed(1)).to(cuda)
    got = _chunk(layer, q, cache, row, past, 2, 2, True).cpu().numpy()
    syn = torch.arange(past + 1, past + n + 1, dtype=torch.int32, device=cuda)
    want = layer.decode(q, cache, row[None].expand(n, -1).contiguous(), syn, max_seq_len=past + n).cpu().numpy()
    assert _rel(got, want) < 1e-5


def test_chunk_workspace_rejects():
    """Sizes without a plan return -1 (host only)."""
    import ctypes

    from fused_turboquant import _lib
    f = _lib.lib().ftq_v1_chunk_workspace_bytes
    f.restype, f.argtypes = ctypes.c_int64, [ctypes.c_int] * 9
    assert f(16, 8, 2, 128, 100, 4, 4, 0, 0) > 0
    assert f(16, 8, 2, 64, 100, 16, 16, 0, 0) > 0
    for bad in ((0, 8, 2, 128, 100, 4, 4, 0, 0), (16, 8, 3, 128, 100, 4, 4, 0, 0), (16, 8, 2, 96, 100, 4, 4, 0, 0),
                (16, 8, 2, 128, -1, 4, 4, 0, 0), (16, 8, 2, 128, 100, 5, 4, 0, 0), (16, 8, 2, 128, 100, 16, 4, 0, 0),
                (16, 8, 2, 128, 2 ** 30, 4, 4, 0, 0)):
        assert f(*bad) == -1, bad


@pytest.mark.gpu
@pytest.mark.parametrize("past", [40, 3000])  # one split, several
def test_a_nan_query_row_stays_nan(cuda, past):
    layer, cache, row = _case(cuda, 64, 4, 4, 1, past + 20, True, 16, seed=6)
    q = torch.randn(20, 4, 64, generator=torch.Generator().manual_seed(1)).to(cuda)
    want = _chunk(layer, q, cache, row, past, 4, 4, True)
    q[7, 2, 5] = float("nan")
    got = _chunk(layer, q, cache, row, past, 4, 4, True)
    assert torch.isnan(got[7, 2]).all()
    got[7, 2] = want[7, 2]
    assert _rel(got.cpu().numpy(), want.cpu().double().numpy()) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("below", [20, 24])
@pytest.mark.parametrize("d,bits", [(64, RAW), (128, RAW), (256, RAW), (64, 4), (256, 8)])
def test_one_dominant_key_and_a_long_tail(cuda, d, bits, below):
    """One key takes most of the weight; 30000 others, ``below`` log2 units
    under it, together still move the output."""
    from fused_turboquant import raw as R, v1 as V1
    n, past, G = 16, 30000, 2
    L, nb = past + n, (past + n + 15) // 16
    g = torch.Generator().manual_seed(d)
    k, v = torch.randn(L, 1, d, generator=g) * 0.02, torch.randn(L, 1, d, generator=g) * 0.5 + 0.5
    u = torch.randn(d, generator=g)
    u /= u.norm()
    k[0, 0] = 30 * u
    q = torch.randn(n, G, d, generator=g) * 0.05 + u * (below * math.log(2) * math.sqrt(d) / 30)
    row, slots = torch.arange(nb, dtype=torch.int32, device=cuda), torch.arange(L, device=cuda)
    layer = None if bits == RAW else V1.TurboQuantV1Layer(d, bits, bits, device=cuda)
    shape = (nb, 16, 1, 4 * d) if layer is None else layer.kv_cache_shape(nb, 16, 1)
    cache = torch.zeros(shape, dtype=torch.uint8, device=cuda)
    (R.raw_store if layer is None else layer.store)(k.to(cuda), v.to(cuda), cache, slots)
    got = _chunk(layer, q.to(cuda), cache, row, past, bits, bits, False).cpu().numpy()
    want = _want(layer, q, cache, row, past, bits, bits, False)
    err = _rel(got, want)
    print(f"[chunk tail d{d} bits {bits} below {below}] rel {err:.2e}", flush=True)
    assert err < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("d,past", [(64, 40), (128, 40), (256, 3000)])
def test_an_infinite_raw_value_stays_in_the_rows_that_attend_it(cuda, d, past):
    n, G, at = 30, 2, 12  # the 13th new token; 12 rows of its tile come before it
    _, cache, row = _case(cuda, d, RAW, RAW, 1, past + n, False, 16, seed=7)
    q = torch.randn(n, G, d, generator=torch.Generator().manual_seed(1)).to(cuda)
    want = _chunk(None, q, cache, row, past, RAW, RAW, False)
    v = cache[row[(past + at) // 16].long(), (past + at) % 16, 0].view(torch.float16)
    v[d + 5], v[2 * d - 1] = float("inf"), float("nan")
    got = _chunk(None, q, cache, row, past, RAW, RAW, False)
    assert torch.equal(got[:at], want[:at])
    assert torch.isnan(got[at:, :, [5, d - 1]]).all()


def test_chunk_rejects_tables_of_another_width():
    """Refused before a device is asked for: the kernel reads 2^key_bits centroids."""
    from fused_turboquant import v1 as V1
    q, row = torch.zeros(16, 4, 64), torch.zeros(4, dtype=torch.int32)
    cache = torch.zeros(4, 16, 1, V1.slot_bytes(64, 4, 4), dtype=torch.uint8)
    for cent in (None, torch.zeros(8), torch.zeros(32), torch.zeros(16, dtype=torch.float64)):
        with pytest.raises(ValueError, match="centroids"):
            V1.v1_chunk_attention(q, cache, row, 8, cent, 4, 4, 0.125)
    with pytest.raises(ValueError, match="slot"):
        V1.v1_chunk_attention(q, cache[..., :32], row, 8, torch.zeros(16), 4, 4, 0.125)


@pytest.mark.gpu
def test_chunk_operator_rejects_tables_of_another_width(cuda):
    """The operator's own check: an error from the host, no launch."""
    from fused_turboquant import _ops
    layer, cache, row = _case(cuda, 64, 4, 4, 1, 40, True, 16, seed=8)
    q = torch.zeros(20, 4, 64, device=cuda)
    for cent, rot in ((layer.centroids[:8].contiguous(), None), (layer.centroids, torch.zeros(32, 64, device=cuda))):
        with pytest.raises(ValueError):
            _ops.ops().v1_chunk_attention(q, cache, row, 20, cent, 4, 4, 0.125, 1, 0, torch.empty_like(q), rot)
