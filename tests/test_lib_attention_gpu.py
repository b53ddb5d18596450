"""Library-format attention kernels (``paged.lib_attention`` through the
HuggingFace cache): windowed and flat decode steps and multi-token steps,
against float64 attention over the oracle's decode of the stored codes (and,
for a multi-token step, the new tokens as given).

Tolerances (relative 2-norm): decode steps and float32 and float16 multi-token
steps carry f16 hi + lo operands (2^-22) with fp32 sums: 1e-5, and for float16
outputs their own rounding, at most 2^-11.  bfloat16 multi-token steps carry
f16 operands, each with a relative error of at most 2^-11 (1e-3 on the outputs,
whose own rounding is 2^-9).
"""
import math

import numpy as np
import pytest
import torch

from oracle import tq_oracle as O

pytestmark = pytest.mark.gpu


def _cache(cuda, d, bk, bv, B, hkv, lens, seed, dtype=torch.bfloat16):
    from fused_turboquant import TurboQuantMSE
    from fused_turboquant.hf import CompressedKVCache
    g = torch.Generator().manual_seed(seed)
    k_tq, v_tq = TurboQuantMSE(d, bits=bk, device=cuda), TurboQuantMSE(d, bits=bv, device=cuda)
    cache = CompressedKVCache(k_tq)
    cache.set_layer_quantizer(0, k_tq)
    cache.set_layer_quantizer_v(0, v_tq)
    L = max(lens)
    k, v = (torch.randn(B, hkv, L, d, generator=g) for _ in range(2))
    k[:, :, ::29] *= 5.0
    keep = torch.tensor([[i >= L - n for i in range(L)] for n in lens], device=cuda)
    cache.store_compressed_kv(k.to(dtype).to(cuda), v.to(dtype).to(cuda), 0, keep=None if all(n == L for n in lens) else keep)
    return cache, g


def _decoded(cache, which, B, hkv, d):
    e = cache.get_compressed_key(0) if which == "k" else cache.get_compressed_value(0)
    tq = cache.get_layer_quantizer(0) if which == "k" else cache.get_layer_quantizer_v(0)
    S = e["packed_indices"].shape[2]
    x = O.decode(e["packed_indices"].cpu().numpy().reshape(-1, d * tq.bits // 8), e["norms"].cpu().numpy().reshape(-1),
                 tq.quantizer.levels.cpu().numpy(), tq.rotation.signs.cpu().numpy(), tq.bits, d)
    return x.reshape(B, hkv, S, d).astype(np.float64)


def _attend(q, k, v, scale, ok):
    """q [n, d], k / v [S, d], ok [n, S] -> [n, d], float64."""
    s = np.where(ok, q @ k.T * scale, -np.inf)
    p = np.exp(s - s.max(axis=1, keepdims=True))
    return (p / p.sum(axis=1, keepdims=True)) @ v


def _rel(got, want):
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


@pytest.mark.parametrize("d,bk,bv,B,hkv,G,lens,window,sinks", [
    (128, 4, 4, 2, 2, 4, (300, 300), 100, 4),    # the window starts inside a page
    (128, 3, 2, 1, 2, 7, (97,), 33, 40),         # more sinks than one tile
    (256, 4, 3, 2, 1, 2, (200, 150), 64, 4),     # sequences of different lengths
    (128, 2, 4, 2, 2, 1, (40, 17), 512, 4),      # a window longer than the context
    (64, 4, 4, 2, 2, 4, (130, 130), None, 0),    # flat rows, the whole context
    (64, 3, 3, 3, 2, 16, (70, 33, 1), 32, 4),    # flat rows, a window, short sequences
    (64, 2, 4, 1, 1, 8, (2100,), 1000, 4),       # splits over the context
])
def test_decode_step(cuda, d, bk, bv, B, hkv, G, lens, window, sinks):
    cache, g = _cache(cuda, d, bk, bv, B, hkv, lens, seed=d + bk)
    q = torch.randn(B, hkv * G, d, generator=g)
    got = cache.decode_attention(q.to(cuda), 0, 1 / math.sqrt(d), sliding_window=window, sink_tokens=sinks).cpu().numpy()
    kd, vd = _decoded(cache, "k", B, hkv, d), _decoded(cache, "v", B, hkv, d)
    want = np.zeros(got.shape)
    for b, n in enumerate(lens):
        pos = np.arange(n)
        ok = np.ones(n, bool) if window is None else (pos >= n - window) | (pos < sinks)
        for h in range(hkv * G):
            want[b, h] = _attend(q[b, h:h + 1].double().numpy(), kd[b, h // G, :n], vd[b, h // G, :n], 1 / math.sqrt(d), ok[None])[0]
    err = _rel(got, want)
    print(f"[lib decode d{d} K{bk}V{bv} lens {lens} w{window}] rel {err:.2e}", flush=True)
    assert err < 1e-5


@pytest.mark.parametrize("d,bk,bv,B,hkv,G,past,n,window,dtype", [
    (128, 4, 4, 1, 2, 4, 200, 70, None, torch.bfloat16),   # past ends inside a tile
    (128, 3, 2, 2, 2, 7, 64, 33, 50, torch.float16),       # a window over past and new tokens
    (256, 4, 4, 2, 1, 2, 45, 20, None, torch.bfloat16),
    (64, 4, 3, 2, 2, 4, 100, 65, None, torch.bfloat16),
    (64, 4, 4, 1, 1, 16, 31, 2, 40, torch.float16),
    (128, 4, 4, 1, 2, 4, 90, 40, None, torch.float32),
    (64, 3, 3, 2, 1, 4, 33, 17, 20, torch.float32),
    (256, 2, 4, 1, 2, 2, 64, 31, None, torch.float32),
])
def test_multi_token_step(cuda, d, bk, bv, B, hkv, G, past, n, window, dtype):
    cache, g = _cache(cuda, d, bk, bv, B, hkv, (past,) * B, seed=d + past, dtype=dtype)
    kd, vd = (np.ascontiguousarray(_decoded(cache, w, B, hkv, d)[:, :, :past]) for w in "kv")
    k, v = (torch.randn(B, hkv, n, d, generator=g).to(dtype) for _ in range(2))
    q = torch.randn(B, hkv * G, n, d, generator=g).to(dtype)
    cache.store_compressed_kv(k.to(cuda), v.to(cuda), 0)
    got = cache.chunk_attention(q.to(cuda), k.to(cuda), v.to(cuda), 0, 1 / math.sqrt(d), sliding_window=window)
    assert got is not None and got.dtype == dtype and got.shape == q.shape
    want = np.zeros(q.shape)
    row, col = past + np.arange(n)[:, None], np.arange(past + n)[None]
    ok = (col <= row) & (col > row - window) if window else col <= row
    for b in range(B):
        for h in range(hkv * G):
            kk = np.concatenate([kd[b, h // G], k[b, h // G].double().numpy()])
            vv = np.concatenate([vd[b, h // G], v[b, h // G].double().numpy()])
            want[b, h] = _attend(q[b, h].double().numpy(), kk, vv, 1 / math.sqrt(d), ok)
    err = _rel(got.float().cpu().numpy(), want)
    print(f"[lib chunk d{d} K{bk}V{bv} past {past} n {n} w{window} {dtype}] rel {err:.2e}", flush=True)
    assert err < {torch.float32: 1e-5, torch.float16: 1e-5 + 2.0 ** -11, torch.bfloat16: 1e-3 + 2.0 ** -9}[dtype]


def test_large_values_stay_finite(cuda):
    """New values up to what an fp16 norm holds, and zero vectors."""
    cache, g = _cache(cuda, 64, 4, 4, 1, 1, (20,), seed=1)
    k, v = torch.zeros(1, 1, 8, 64), torch.randn(1, 1, 8, 64, generator=g) * 5000.0
    q = torch.randn(1, 4, 8, 64, generator=g)
    dt = torch.bfloat16
    cache.store_compressed_kv(k.to(dt).to(cuda), v.to(dt).to(cuda), 0)
    got = cache.chunk_attention(q.to(dt).to(cuda), k.to(dt).to(cuda), v.to(dt).to(cuda), 0, 0.125)
    assert torch.isfinite(got).all() and got.abs().max() > 1000


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,hq,hkv,n,d,cb", [(2, 8, 2, 5, 64, 2), (1, 4, 4, 1, 128, 1), (3, 7, 1, 33, 256, 1)])
def test_rope_kernel_is_the_torch_expression(cuda, dtype, B, hq, hkv, n, d, cb):
    """Bit for bit, on transposed views, with one or B sets of angles."""
    from fused_turboquant.hf import fused_cache as F
    from fused_turboquant import _ops
    g = torch.Generator().manual_seed(n)
    q = torch.randn(B, n, hq, d, generator=g).to(dtype).to(cuda).transpose(1, 2)
    k = torch.randn(B, n, hkv, d, generator=g).to(dtype).to(cuda).transpose(1, 2)
    ang = torch.randn(cb, n, d, generator=g) * 3
    cos, sin = ang.cos().to(dtype).to(cuda), ang.sin().to(dtype).to(cuda)
    assert F._rope_fused(q, k, cos, sin)
    got, want = _ops.ops().rope(q, k, cos, sin), F._apply_rotary_pos_emb(q, k, cos, sin)
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.transpose(1, 2).is_contiguous() and torch.equal(a, b)
    assert not F._rope_fused(q, k, cos[..., : d // 2], sin[..., : d // 2])  # partial rotary: the torch expression
    assert not F._rope_fused(q.requires_grad_(), k, cos, sin)


def test_append_slots(cuda):
    from fused_turboquant import _ops
    lens = torch.tensor([0, 7, 300], dtype=torch.int32, device=cuda)
    got = _ops.ops().append_slots(lens, 260, 1000)
    want = torch.cat([b * 1000 + n + torch.arange(260) for b, n in enumerate((0, 7, 300))])
    assert torch.equal(got.cpu(), want) and lens.tolist() == [260, 267, 560]


def _lib(cache, q, window=None, sinks=0, precise=None, new_kv=None, lens=None, max_len=None):
    """``paged.lib_attention`` on a cache's layer, query [B, Hq, n, d]."""
    from fused_turboquant import paged as P
    lp = cache._pages[0]
    src = dict(pages=(lp.kv_cache, lp.block_table)) if lp.d in (128, 256) else dict(flat=(lp.kp, lp.kn, lp.vp, lp.vn))
    return P.lib_attention(q, lp.lens_dev if lens is None else lens, max_len or max(lp.lens), lp.k_tq, lp.v_tq,
                           1 / math.sqrt(lp.d), new_kv=new_kv, window=window, sinks=sinks, precise=precise, **src)


@pytest.mark.parametrize("precise", [False, True])
@pytest.mark.parametrize("d,B,hkv,G,lens,window,sinks", [
    (128, 2, 2, 4, (300, 190), 100, 4),   # the window starts inside a page; sinks and tile padding
    (256, 1, 1, 2, (2100,), 1000, 5),     # splits over the context
    (64, 3, 2, 16, (70, 33, 1), 32, 4),   # flat rows, short sequences
    (64, 1, 2, 4, (130,), None, 0),       # no window
])
def test_decode_step_at_both_precisions(cuda, d, B, hkv, G, lens, window, sinks, precise):
    """Hidden positions take no weight in either form.  f16 operands: 2^-11
    per operand, three of them in a row's weights and values (1e-3)."""
    cache, g = _cache(cuda, d, 4, 4, B, hkv, lens, seed=d)
    q = torch.randn(B, hkv * G, 1, d, generator=g)
    got = _lib(cache, q.to(cuda), window, sinks, precise).cpu().numpy()[:, :, 0]
    kd, vd = _decoded(cache, "k", B, hkv, d), _decoded(cache, "v", B, hkv, d)
    want = np.zeros(got.shape)
    for b, n in enumerate(lens):
        pos = np.arange(n)
        ok = np.ones(n, bool) if window is None else (pos >= n - window) | (pos < sinks)
        for h in range(hkv * G):
            want[b, h] = _attend(q[b, h].double().numpy(), kd[b, h // G, :n], vd[b, h // G, :n], 1 / math.sqrt(d), ok[None])[0]
    err = _rel(got, want)
    print(f"[lib decode d{d} lens {lens} w{window} precise {precise}] rel {err:.2e}", flush=True)
    assert err < (1e-5 if precise else 1e-3)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,past", [(64, 90), (64, 2100), (128, 90), (128, 2100)])  # one split, several
def test_not_a_number_stays_in_its_rows(cuda, d, past, dtype):
    """A NaN query row, an infinite new key and an infinite new value: the rows
    that meet them are NaN (as softmax attention gives), the others as without."""
    hkv, G, n = 2, 2, 24
    cache, g = _cache(cuda, d, 4, 4, 1, hkv, (past,), seed=past, dtype=dtype)
    k, v = (torch.randn(1, hkv, n, d, generator=g).to(dtype).to(cuda) for _ in range(2))
    q = torch.randn(1, hkv * G, n, d, generator=g).to(dtype).to(cuda)
    cache.store_compressed_kv(k, v, 0)
    want = _lib(cache, q, new_kv=(k, v)).float().cpu()
    q2, k2, v2 = q.clone(), k.clone(), v.clone()
    q2[0, 1, 5, 3] = float("nan")        # kv head 0, row 5 of one head
    k2[0, 0, 15, 7] = float("inf")       # kv head 0, rows 15 ..
    v2[0, 1, 20, 9] = float("-inf")      # kv head 1, rows 20 ..
    got = _lib(cache, q2, new_kv=(k2, v2)).float().cpu()
    bad = torch.zeros(hkv * G, n, dtype=torch.bool)
    bad[1, 5] = True
    bad[:G, 15:] = True
    bad[G:, 20:] = True
    assert torch.isnan(got[0][bad]).all()
    assert _rel(got[0][~bad].numpy(), want[0][~bad].numpy()) < (1e-5 if dtype == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("ctx", [90, 2100])  # one split, several
def test_decode_step_with_an_infinite_key_norm(cuda, ctx):
    """A row with a NaN score is zeros in a windowed decode step (softmax's NaN
    weights count as 0), not an average of what the other splits hold."""
    d, hkv, G = 64, 2, 2
    cache, g = _cache(cuda, d, 4, 4, 1, hkv, (ctx,), seed=3)
    cache._pages[0].kn[0, 0, ctx - 50] = float("inf")
    q = torch.randn(1, hkv * G, d, generator=g).to(cuda)
    got = cache.decode_attention(q, 0, 0.125, sliding_window=ctx - 10, sink_tokens=4).cpu()
    assert (got[0, :G] == 0).all() and torch.isfinite(got).all() and (got[0, G:] != 0).any(dim=-1).all()


@pytest.mark.parametrize("d,past,n", [(64, 49, 300), (128, 27, 120), (256, 82, 31)])
def test_float16_step_keeps_its_operands(cuda, d, past, n):
    """float16 queries and new tokens are not rounded on their way to the
    products: with scores of up to 2^5, f16 operands would show (7e-4 to 8e-4)."""
    hkv, G, dt = 1, 4, torch.float16
    cache, g = _cache(cuda, d, 4, 4, 1, hkv, (past,), seed=d, dtype=dt)
    kd, vd = (np.ascontiguousarray(_decoded(cache, w, 1, hkv, d)[:, :, :past]) for w in "kv")
    k, v = (torch.randn(1, hkv, n, d, generator=g).to(dt) for _ in range(2))
    q = (6 * torch.randn(1, hkv * G, n, d, generator=g)).to(dt)
    cache.store_compressed_kv(k.to(cuda), v.to(cuda), 0)
    got = cache.chunk_attention(q.to(cuda), k.to(cuda), v.to(cuda), 0, 1 / math.sqrt(d)).float().cpu().numpy()[0]
    kk, vv = (np.concatenate([x[0, 0], y[0, 0].double().numpy()]) for x, y in ((kd, k), (vd, v)))
    ok = np.arange(past + n)[None] <= past + np.arange(n)[:, None]
    want = np.stack([_attend(q[0, h].double().numpy(), kk, vv, 1 / math.sqrt(d), ok) for h in range(G)])
    err = _rel(got, want)
    print(f"[lib chunk float16 d{d} past {past} n {n}] rel {err:.2e}", flush=True)
    assert err < 1e-5 + 2.0 ** -11  # the products, and one rounding of the output


def test_queries_beyond_f16(cuda):
    """bfloat16 queries larger than f16 holds, with keys so small that their
    scores are ordinary, beside ordinary rows."""
    d, hkv, G, past, n, dt = 128, 2, 2, 40, 20, torch.bfloat16
    cache, g = _cache(cuda, d, 4, 4, 1, hkv, (past,), seed=2, dtype=dt)
    k, v = (torch.randn(1, hkv, n, d, generator=g) for _ in range(2))
    q = torch.randn(1, hkv * G, n, d, generator=g)
    k, v, q = k.to(dt), v.to(dt), q.to(dt)
    cache.store_compressed_kv(k.to(cuda), v.to(cuda), 0)
    big = q.clone()
    big[:, 1, 3:] *= 2.0 ** 20  # powers of two: exact, so that the key's factor brings the same scores back
    cache._pages[0].kv_cache.zero_()  # the past's norms are 0: its scores are 0 for every query
    want = _lib(cache, q.to(cuda), new_kv=(k.to(cuda), v.to(cuda))).float().cpu()
    k2 = k.clone()
    k2[:, 0] *= 2.0 ** -20
    got = _lib(cache, big.to(cuda), new_kv=(k2.to(cuda), v.to(cuda))).float().cpu()
    assert torch.isfinite(got).all()
    assert _rel(got[0, 1, 3:].numpy(), want[0, 1, 3:].numpy()) < 1e-3 + 2.0 ** -8
    assert _rel(got[0, G:].numpy(), want[0, G:].numpy()) < 1e-6


@pytest.mark.parametrize("window,sinks,queries", [
    (0, 4, 1), (0, 0, 1), (-3, 2, 1),            # a window that holds no position
    (2 ** 40, 4, 1), (20, -1, 1), (20, 2 ** 40, 1),  # beyond the context, no sinks, all of them
    (20, 4, 3),                                  # one sequence read by three queries
])
@pytest.mark.parametrize("d", [64, 128])
def test_windows_sinks_and_batches_of_the_torch_form(cuda, d, window, sinks, queries, monkeypatch):
    """What the cache's torch form takes, the kernels or that form still take."""
    cache, g = _cache(cuda, d, 4, 4, 1, 2, (50,), seed=4)
    q = torch.randn(queries, 4, d, generator=g).to(cuda)
    got = cache.decode_attention(q, 0, 0.1, sliding_window=window, sink_tokens=sinks).cpu()
    monkeypatch.setattr(type(cache), "_fused_attention", staticmethod(lambda *a: False))
    want = cache.decode_attention(q, 0, 0.1, sliding_window=window, sink_tokens=sinks).cpu()
    assert got.shape == want.shape and (got - want).norm() <= 1e-5 * want.norm()


def _misaligned(t):
    """The same values, contiguous, at a storage offset of one element."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    flat[1:] = t.reshape(-1)
    return flat[1:].view(t.shape)


def _odd_strides(t):
    """The same values, with a dimension of size 1 and an odd stride in front, or rows that are not contiguous."""
    wide = torch.empty(*t.shape[:-1], 2 * t.shape[-1] + 1, dtype=t.dtype, device=t.device)
    wide[..., 1:] = t.repeat_interleave(2, -1)
    return wide[..., 1::2]


@pytest.mark.parametrize("form", [_misaligned, _odd_strides,
                                  lambda t: t.contiguous().as_strided(t.shape, (t[0].numel() + 3, *t.stride()[1:]))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_any_alignment_and_stride(cuda, form, dtype):
    """Queries, new tokens and angles at any storage offset and stride give what aligned ones give."""
    from fused_turboquant import _ops
    from fused_turboquant.hf import fused_cache as F
    d, n = 64, 6
    cache, g = _cache(cuda, d, 4, 4, 1, 2, (50,), seed=5, dtype=dtype)
    k, v = (torch.randn(1, 2, n, d, generator=g).to(dtype).to(cuda) for _ in range(2))
    q = torch.randn(1, 4, n, d, generator=g).to(dtype).to(cuda)
    cos, sin = (torch.randn(1, n, d, generator=g).to(dtype).to(cuda) for _ in range(2))
    q1 = q[:, :, 0].contiguous()
    want = cache.decode_attention(q1, 0, 0.125, sliding_window=20)
    assert torch.equal(cache.decode_attention(form(q1), 0, 0.125, sliding_window=20), want)
    cache.store_compressed_kv(k, v, 0)
    want = cache.chunk_attention(q, k, v, 0, 0.125)
    assert torch.equal(cache.chunk_attention(form(q), form(k), form(v), 0, 0.125), want)
    assert F._rope_fused(form(q), form(k), form(cos), form(sin))
    for a, b in zip(_ops.ops().rope(form(q), form(k), form(cos), form(sin)), _ops.ops().rope(q, k, cos, sin)):
        assert torch.equal(a, b)


def test_flat_rows_end_at_the_capacity(cuda):
    """A length beyond the rows' capacity counts as the capacity."""
    cache, g = _cache(cuda, 64, 4, 4, 2, 2, (100, 100), seed=6)
    cap = cache._pages[0].cap
    q = torch.randn(2, 4, 1, 64, generator=g).to(cuda)
    lens = torch.tensor([cap, 70], dtype=torch.int32, device=cuda)
    want = _lib(cache, q, window=60, lens=lens, max_len=cap)
    lens[0] = cap + 40
    got = _lib(cache, q, window=60, lens=lens, max_len=cap)
    assert torch.equal(got, want)


@pytest.mark.parametrize("d,dtype", [(64, torch.float32), (128, torch.bfloat16), (256, torch.float16)])
def test_multi_token_step_lengths_strides_and_streams(cuda, d, dtype):
    """Sequences of different lengths, queries and new tokens as the transposed
    views a projection gives, on a stream other than the default one."""
    B, hkv, G, n, lens = 2, 2, 3, 25, (90, 33)
    cache, g = _cache(cuda, d, 4, 3, B, hkv, lens, seed=d + 7, dtype=dtype)
    kd, vd = (_decoded(cache, w, B, hkv, d) for w in "kv")
    k, v = (torch.randn(B, n, hkv, d, generator=g).to(dtype).transpose(1, 2) for _ in range(2))
    q = torch.randn(B, n, hkv * G, d, generator=g).to(dtype).transpose(1, 2)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        qc, kc, vc = (t.transpose(1, 2).to(cuda).transpose(1, 2) for t in (q, k, v))
        assert not (qc.is_contiguous() or kc.is_contiguous())
        cache.store_compressed_kv(kc, vc, 0)
        got = cache.chunk_attention(qc, kc, vc, 0, 1 / math.sqrt(d), sliding_window=60).float().cpu().numpy()
    for b, past in enumerate(lens):
        row, col = past + np.arange(n)[:, None], np.arange(past + n)[None]
        ok = (col <= row) & (col > row - 60)
        for h in range(hkv * G):
            kk = np.concatenate([kd[b, h // G, :past], k[b, h // G].double().numpy()])
            vv = np.concatenate([vd[b, h // G, :past], v[b, h // G].double().numpy()])
            want = _attend(q[b, h].double().numpy(), kk, vv, 1 / math.sqrt(d), ok)
            tol = {torch.float32: 1e-5, torch.float16: 1e-5 + 2.0 ** -11, torch.bfloat16: 1e-3 + 2.0 ** -9}[dtype]
            assert _rel(got[b, h], want) < tol, (b, h)


def test_several_segments(cuda):
    """A context whose dequantised fragments exceed one workspace segment (192
    MiB: 5952 positions of 64 kv heads at d = 64), in a decode step and in a
    multi-token step."""
    d, B, hkv, past, n = 64, 4, 16, 6100, 6
    cache, g = _cache(cuda, d, 2, 3, B, hkv, (past,) * B, seed=9)
    kd, vd = (_decoded(cache, w, B, hkv, d) for w in "kv")
    q = torch.randn(B, hkv, n, d, generator=g)
    got = cache.decode_attention(q[:, :, 0].to(cuda), 0, 0.125).cpu().numpy()
    every = np.ones((1, past), bool)
    want = np.stack([[_attend(q[b, h, :1].double().numpy(), kd[b, h, :past], vd[b, h, :past], 0.125, every)[0]
                      for h in range(hkv)] for b in range(B)])
    assert _rel(got, want) < 1e-5
    k, v = (torch.randn(B, hkv, n, d, generator=g) for _ in range(2))
    cache.store_compressed_kv(k.to(cuda), v.to(cuda), 0)
    got = cache.chunk_attention(q.to(cuda), k.to(cuda), v.to(cuda), 0, 0.125).cpu().numpy()
    ok = np.arange(past + n)[None] <= past + np.arange(n)[:, None]
    want = np.stack([[_attend(q[b, h].double().numpy(), np.concatenate([kd[b, h, :past], k[b, h].double().numpy()]),
                              np.concatenate([vd[b, h, :past], v[b, h].double().numpy()]), 0.125, ok)
                      for h in range(hkv)] for b in range(B)])
    assert _rel(got, want) < 1e-5
