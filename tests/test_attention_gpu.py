"""GPU parity of the KV append (bh_kv_store) and of grouped-query attention
over the cache (bh_attention) against the oracle's restatement of
src/forward.rs:273-375 (the reference's one-token loop, run per query).

Bars: the f32 store bit for bit, the f16 store = gguf::f32_to_half bit for
bit (specials and the subnormal range included); attention outputs
max|gpu-ref| / max(|ref|, |gpu|) <= 1e-5 (scores and P.V summed in another
order; the generic path keeps the reference's sequence except the f64 sum's
order).
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-5
MODEL = (24, 4, 256)  # n_head, n_kv, hd of the model (24 q / 4 kv heads x 256)


def _say(*a):
    print(*a, flush=True)


def _t(a, dev):
    import torch
    if a.dtype == np.uint16:
        return torch.from_numpy(a.view(np.int16).copy()).to(dev)
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dev)


def _h(t):
    import torch
    torch.cuda.synchronize()
    a = t.cpu().numpy()
    return a.view(np.uint16) if a.dtype == np.int16 else a


def _case(synth, n_q, pos0, n_head, n_kv, hd, seed, qscale=2.0):
    r = synth.Rng(seed)
    n = pos0 + n_q
    q = r.normal(n_q * n_head * hd).reshape(n_q, n_head, hd) * np.float32(qscale)
    kc = r.normal(n * n_kv * hd).reshape(n, n_kv * hd)
    vc = r.normal(n * n_kv * hd).reshape(n, n_kv * hd)
    return q.astype(np.float32), kc, vc


def _run(bh, dev, q, pos0, kc, vc, n_kv):
    return _h(bh.attention(_t(q, dev), pos0, _t(kc, dev), _t(vc, dev), n_kv))


@pytest.mark.parametrize("n_q,pos0,f16", [
    (1, 0, False), (1, 6, False), (1, 63, False), (1, 64, False), (1, 999, False),
    (1, 4095, False), (1, 4095, True), (1, 130, True),
    (1, 9000, False), (1, 20000, True),   # one query, chunks of several tiles (ragged last chunk)
    (3, 100, False),     # a few tokens at once (speculative verification)
    (3, 63, False),      # query 0 sees no position of the last chunk (merged as empty)
    (5, 4093, False),    # several queries over several merge groups
    (17, 0, False),      # a causal batch from the first position
    (64, 2000, True),
])
def test_attention_model_heads(bh, oracle, synth, dev, n_q, pos0, f16):
    n_head, n_kv, hd = MODEL
    _say("attention", n_q, pos0, "f16" if f16 else "f32")
    q, kc, vc = _case(synth, n_q, pos0, n_head, n_kv, hd, 300 + n_q + pos0)
    if f16:
        kc = kc.astype(np.float16).view(np.uint16)
        vc = vc.astype(np.float16).view(np.uint16)
    ref = oracle.attention(q, pos0, kc, vc, n_kv)
    got = _run(bh, dev, q, pos0, kc, vc, n_kv)
    err = rel_err(got, ref)
    _say("  rel", err)
    assert err <= TOL


@pytest.mark.parametrize("n_head,n_kv,hd,n_q,pos0", [
    (8, 2, 256, 2, 50),    # grouping 4
    (8, 8, 256, 1, 300),   # grouping 1
    (16, 2, 256, 1, 70),   # grouping 8
    (6, 2, 64, 3, 40),     # other head size: generic path
    (5, 1, 80, 2, 9),      # grouping 5, hd 80: generic path
    (12, 4, 256, 1, 33),   # grouping 3
    (8, 2, 256, 1, 40000), # one query, long context: 3-tile chunks
])
def test_attention_other_shapes(bh, oracle, synth, dev, n_head, n_kv, hd, n_q, pos0):
    _say("attention shape", n_head, n_kv, hd, n_q, pos0)
    q, kc, vc = _case(synth, n_q, pos0, n_head, n_kv, hd, 400 + hd + pos0)
    ref = oracle.attention(q, pos0, kc, vc, n_kv)
    assert rel_err(_run(bh, dev, q, pos0, kc, vc, n_kv), ref) <= TOL


def test_attention_unaligned_q_uses_generic(bh, oracle, synth, dev):
    import torch
    n_head, n_kv, hd = MODEL
    q, kc, vc = _case(synth, 1, 20, n_head, n_kv, hd, 500)
    buf = torch.zeros(q.size + 1, dtype=torch.float32, device=dev)
    buf[1:] = _t(q.reshape(-1), dev)
    got = _h(bh.attention(buf[1:].view(q.shape), 20, _t(kc, dev), _t(vc, dev), n_kv))
    assert rel_err(got, oracle.attention(q, 20, kc, vc, n_kv)) <= TOL


def test_attention_generic_skips_zero_probabilities(bh, oracle, synth, dev):
    """The generic path keeps src/forward.rs:363-366: a position whose
    probability is exactly 0 is skipped, so an inf in its v row does not
    reach the output."""
    q, kc, vc = _case(synth, 1, 1, 1, 1, 4, 501)
    q[0, 0] = [100.0, 0.0, 0.0, 0.0]
    kc[0] = [-100.0, 0.0, 0.0, 0.0]
    kc[1] = [100.0, 0.0, 0.0, 0.0]
    vc[0] = np.inf
    ref = oracle.attention(q, 1, kc, vc, 1)
    got = _run(bh, dev, q, 1, kc, vc, 1)
    assert np.array_equal(got, ref)


def test_kv_store_bits(bh, oracle, synth, dev):
    """f32 rows copied exactly; f16 rows = gguf::f32_to_half, including NaN,
    inf, overflow, ties and the subnormal range, at an offset position."""
    import torch
    r = synth.Rng(502)
    n_tok, elems, cap, pos0 = 3, 1024, 8, 4
    k = r.normal(n_tok * elems).reshape(n_tok, elems) * np.float32(3.0)
    v = r.normal(n_tok * elems).reshape(n_tok, elems)
    special = np.array([np.nan, np.inf, -np.inf, 65504.0, 65520.0, 1e6, -0.0, 1e-8, 6e-8,
                        3e-8, 2.98e-8, 5.96e-8, 1e-5, -6.1e-5, 1.0 + 2.0 ** -11, 1.0 + 3 * 2.0 ** -11,
                        0.1, 1e-40], dtype=np.float32)
    k[0, :special.size] = special
    v[1, :special.size] = special[::-1]
    for f16 in (False, True):
        dt = np.uint16 if f16 else np.float32
        kc0 = np.zeros((cap, elems), dt)
        vc0 = np.zeros((cap, elems), dt)
        want_k, want_v = oracle.kv_store(k, v, kc0, vc0, pos0)
        dk, dv = _t(kc0, dev), _t(vc0, dev)
        bh.kv_store(_t(k, dev), _t(v, dev), dk, dv, pos0)
        gk, gv = _h(dk), _h(dv)
        assert np.array_equal(gk.view(np.uint32 if not f16 else np.uint16),
                              want_k.view(np.uint32 if not f16 else np.uint16))
        assert np.array_equal(gv.view(np.uint32 if not f16 else np.uint16),
                              want_v.view(np.uint32 if not f16 else np.uint16))


def test_store_then_attend_token_loop(bh, oracle, synth, dev):
    """The reference's decode loop: per token, append k/v at pos then attend
    with n_q = 1; the same caches and outputs as one 6-token batch call."""
    import torch
    n_head, n_kv, hd = MODEL
    n_tok = 6
    r = synth.Rng(503)
    q = r.normal(n_tok * n_head * hd).reshape(n_tok, n_head, hd)
    k = r.normal(n_tok * n_kv * hd).reshape(n_tok, n_kv * hd)
    v = r.normal(n_tok * n_kv * hd).reshape(n_tok, n_kv * hd)
    dk = torch.zeros((n_tok, n_kv * hd), device=dev)
    dv = torch.zeros_like(dk)
    outs = []
    for t in range(n_tok):
        bh.kv_store(_t(k[t:t + 1], dev), _t(v[t:t + 1], dev), dk, dv, t)
        outs.append(_h(bh.attention(_t(q[t:t + 1], dev), t, dk, dv, n_kv)))
    ref = oracle.attention(q, 0, k, v, n_kv)
    assert rel_err(np.concatenate(outs), ref) <= TOL
    batch = _h(bh.attention(_t(q, dev), 0, dk, dv, n_kv))
    assert rel_err(batch, ref) <= TOL


@pytest.mark.parametrize("n_q,pos0,f16,n_head,n_kv,vscale,qscale", [
    (64, 4032, False, 24, 4, 1.0, 2.0),    # the bench's prefill case
    (64, 4032, True, 24, 4, 1.0, 2.0),
    (50, 17, False, 24, 4, 1.0, 2.0),      # ragged row tiles and position tiles
    (9, 300, False, 16, 2, 1.0, 2.0),      # grouping 8
    (40, 100, False, 8, 8, 1.0, 2.0),      # grouping 1
    (16, 500, False, 24, 4, 3e6, 1e-3),    # large v (scaled-down tiles), small q
    (16, 500, False, 24, 4, 1e-6, 10.0),   # tiny v, peaked attention (logits ~ N(0, 10^2))
    (33, 2000, True, 12, 4, 1.0, 0.05),    # f16 cache, near-flat attention
    # 8+ row tiles per kv head: the f32 cache is split into f16 hi / lo once
    (200, 37, False, 24, 4, 1.0, 2.0),     # ragged row and position tiles
    (176, 500, False, 24, 4, 3e6, 1e-3),   # large v, small q
    (176, 500, False, 24, 4, 1e-6, 10.0),  # tiny v, peaked attention
])
def test_attention_multi_query_matrix_cores(bh, oracle, synth, dev, n_q, pos0, f16, n_head, n_kv,
                                            vscale, qscale):
    """Many queries per kv head take the matrix-core path (f16 hi/lo
    products with power-of-two scaling); <= 1e-5 against the oracle's
    per-token loop, on magnitudes that stress the splits."""
    hd = 256
    _say("attention mq", n_q, pos0, "f16" if f16 else "f32", n_head, n_kv, vscale, qscale)
    q, kc, vc = _case(synth, n_q, pos0, n_head, n_kv, hd, 700 + n_q + pos0, qscale=qscale)
    vc = (vc * np.float32(vscale)).astype(np.float32)
    if f16:
        kc = kc.astype(np.float16).view(np.uint16)
        vc = vc.astype(np.float16).view(np.uint16)
    ref = oracle.attention(q, pos0, kc, vc, n_kv)
    got = _run(bh, dev, q, pos0, kc, vc, n_kv)
    err = rel_err(got, ref)
    _say("  rel", err)
    assert err <= TOL


@pytest.mark.parametrize("f16", [False, True])
def test_attention_prefill_2048_from_position_0(bh, oracle, synth, dev, f16):
    """The prefill shape behind config 4b's scores: 2048 causal queries from
    position 0 on the model's heads (src/forward.rs:273-375 run for a whole
    window, as GDev::prefill_batch does).  The whole batch runs in one call;
    sampled query rows (the first, chunk and tile edges, the last) are
    checked against the oracle's per-token loop at their own positions, and
    query 0 -- which sees position 0 alone, so its softmax is exactly 1 --
    must return v_0 of its kv head (to the f16 hi + lo products' 2^-21)."""
    n_head, n_kv, hd = MODEL
    n = 2048
    _say("attention prefill 2048", "f16" if f16 else "f32")
    q, kc, vc = _case(synth, n, 0, n_head, n_kv, hd, 911 + int(f16))
    if f16:
        kc = kc.astype(np.float16).view(np.uint16)
        vc = vc.astype(np.float16).view(np.uint16)
    got = _run(bh, dev, q, 0, kc, vc, n_kv)
    assert np.all(np.isfinite(got))
    v0 = (vc[0].view(np.float16).astype(np.float32) if f16 else vc[0]).reshape(n_kv, hd)
    grp = n_head // n_kv
    for h in range(n_head):
        assert rel_err(got[0, h], v0[h // grp]) <= 1e-6
    worst = 0.0
    for i in (1, 2, 63, 64, 127, 511, 1000, 1023, 1024, 1535, 2046, 2047):
        ref = oracle.attention(q[i:i + 1], i, kc[:i + 1], vc[:i + 1], n_kv)
        worst = max(worst, rel_err(got[i:i + 1], ref))
    _say("  rel (sampled rows)", worst)
    assert worst <= TOL


def test_attention_presplit_tile_scales(bh, oracle, synth, dev):
    """The pre-split f32 path (8+ row tiles per kv head) with V tiles whose
    magnitudes differ by up to 2^48 along the positions: each 32-position
    tile keeps its own power-of-two unit, and a block whose running unit
    has grown scales the tile's probabilities down instead.  <= 1e-5
    against the oracle's per-token loop."""
    n_head, n_kv, hd = MODEL
    n_q, pos0 = 192, 300
    q, kc, vc = _case(synth, n_q, pos0, n_head, n_kv, hd, 977)
    n = pos0 + n_q
    expo = np.round(24.0 * np.sin(np.arange(n) / 37.0)).astype(np.float32)
    vc = (vc * np.exp2(expo)[:, None]).astype(np.float32)
    ref = oracle.attention(q, pos0, kc, vc, n_kv)
    got = _run(bh, dev, q, pos0, kc, vc, n_kv)
    err = rel_err(got, ref)
    _say("  rel", err)
    assert err <= TOL


@pytest.mark.parametrize("n_q,pos0,f16,span", [
    (8, 1785, True, 0.0),    # 48 rows (two waves of four); the last chunk is one position
    (8, 1816, True, 0.0),    # whole tiles only
    (11, 1790, True, 0.0),   # 66 rows: a wave of two rows
    (22, 1000, True, 0.0),   # 132 rows: a second row tile of four rows; a 30-position last tile
    (64, 700, True, 32.0),   # scores that rise with the position: the reference moves many times
    (8, 1000, True, 0.0),    # four tiles a block: the 16-row form
    (256, 0, False, 0.0),    # a pre-split f32 cache, causal from position 0, one chunk
    (171, 86, False, 32.0),  # its last tile holds one position
    (172, 90, False, 64.0),  # each tile's scores far above the last one's
    (171, 30, False, 0.0),   # seven tiles a block: the 16-row form
])
def test_attention_wide_rows(bh, oracle, synth, dev, n_q, pos0, f16, span, n_kv=32):
    """The matrix-core forms (16-row ones on blocks of up to nine position
    tiles, the 32-row one from ten on, over f16 caches and f32 caches split beforehand; 32 kv heads, so that few
    positions make such blocks) at the edges of its row and position tiles, and with keys whose scores
    climb by `span` nats from the first position to the last, so that the
    running reference and the accumulators move many times.  A score of s
    nats is rounded to s * 2^-24 at best, which is the relative error of its
    probability, times the few roundings of its sum: centred, |s| <= 42, and
    the oracle is within 6e-6 of 64-bit arithmetic on these inputs (at the
    uncentred |s| of 390 it is 1e-4 away, past TOL by itself)."""
    n_head, hd = 6 * n_kv, 256
    _say("attention wide rows", n_q, pos0, "f16" if f16 else "f32", span)
    q, kc, vc = _case(synth, n_q, pos0, n_head, n_kv, hd, 1500 + n_q + pos0, qscale=1.0)
    if span:
        # q and k share a direction: a score is that of the position alone
        # plus noise of unit size
        u = np.float32(1.0 / np.sqrt(hd))
        q += u * np.float32(16.0)
        n = pos0 + n_q
        ramp = (np.arange(n, dtype=np.float32) / np.float32(n - 1) - np.float32(0.5)) * np.float32(span)
        kc = (kc + ramp[:, None] * u).astype(np.float32)
    if f16:
        kc = kc.astype(np.float16).view(np.uint16)
        vc = vc.astype(np.float16).view(np.uint16)
    ref = oracle.attention(q, pos0, kc, vc, n_kv)
    got = _run(bh, dev, q, pos0, kc, vc, n_kv)
    err = rel_err(got, ref)
    _say("  rel", err)
    assert err <= TOL


@pytest.mark.parametrize("n_q,pos0,f16,span,n_kv", [
    (8, 2873, True, 0.0, 25),     # ten tiles a block, 48 rows (two waves of four); the last chunk is one position
    (8, 2552, True, 0.0, 32),     # whole tiles only
    (11, 2300, True, 0.0, 32),    # 66 rows: a wave of two rows; a last chunk of three tiles
    (22, 1200, True, 0.0, 32),    # 132 rows: a second row tile of four rows; a 6-position last tile
    (8, 2240, True, 0.0, 32),     # nine tiles a block: the 16-row form
    (320, 0, False, 0.0, 32),     # a pre-split f32 cache, causal from position 0, one chunk
    (171, 118, False, 32.0, 32),  # its last tile holds one position
    (172, 154, False, 64.0, 32),  # each tile's scores far above the last one's
    (171, 100, False, 0.0, 32),   # nine tiles a block: the 16-row form
])
def test_attention_wide_rows_ten_tiles(bh, oracle, synth, dev, n_q, pos0, f16, span, n_kv):
    """The same edges on blocks of ten tiles and more, and of nine."""
    test_attention_wide_rows(bh, oracle, synth, dev, n_q, pos0, f16, span, n_kv)


@pytest.mark.parametrize("n_q,pos0,f16", [(22, 1200, True), (320, 0, False)])
def test_attention_wide_rows_first_tile(bh, oracle, synth, dev, n_q, pos0, f16):
    """The 32-row form's first staged tile is read by every wave before the
    third takes its place: most of each row's weight is on the first tile of
    its first chunk and keys of opposite sign stand two tiles later, so a
    wave that saw those instead would be far off; the same bits in ten calls
    of a full grid."""
    import torch
    n_head, n_kv, hd = 192, 32, 256
    _say("attention first tile", n_q, pos0, "f16" if f16 else "f32")
    q, kc, vc = _case(synth, n_q, pos0, n_head, n_kv, hd, 77 + n_q, qscale=1.0)
    u = np.float32(1.0 / np.sqrt(hd))
    q += u * np.float32(16.0)
    kc = kc.astype(np.float32)
    kc[:32] += u * np.float32(8.0)
    kc[64:96] -= u * np.float32(8.0)
    if f16:
        kc = kc.astype(np.float16).view(np.uint16)
        vc = vc.astype(np.float16).view(np.uint16)
    ref = oracle.attention(q, pos0, kc, vc, n_kv)
    tq, tk, tv = _t(q, dev), _t(kc, dev), _t(vc, dev)
    first = bh.attention(tq, pos0, tk, tv, n_kv)
    for _ in range(9):
        assert torch.equal(bh.attention(tq, pos0, tk, tv, n_kv), first)
    err = rel_err(_h(first), ref)
    _say("  rel", err)
    assert err <= TOL


@pytest.mark.parametrize("f16", [True, False])
def test_attention_wide_rows_sink_and_flat_tail(bh, dev, f16):
    """An early position that takes nearly all of a row's weight but holds a
    zero value, and a flat tail behind it, whose probabilities of 2^-15 to
    2^-19 are all rounded the same way.  In units of 2^-14 a probability p
    splits into two f16 with an error of 2^-25 at most: 2^-39 / p, 2^-20 of it
    at the smallest p here.  The ten tiles are 40 products, each of which
    rounds an f32 sum once: 2^-24 each at most; exponential, row sum and
    division are 8 more.  Scores are exact (multiples of 2^-8), the reference
    is in 64 bits."""
    import torch
    n, n_head, n_kv, hd = 320, 192, 32, 256
    rng = np.random.default_rng(5)
    delta = np.round(rng.uniform(15, 19, (n, n_head)) * np.log(2.0) * 256) / 256
    q = np.zeros((n, n_head, hd), np.float32)
    q[..., 0] = 16 * delta
    k = np.zeros((n, n_kv * hd), np.float32)
    k[0, ::hd] = 1.0
    vals = (1.0 + rng.integers(0, 1024, n_kv * hd) / 1024).astype(np.float32)
    v = np.tile(vals, (n, 1))
    v[0] = 0.0
    cache = (lambda a: torch.from_numpy(a).to(dev).to(torch.float16).view(torch.int16)) if f16 else \
        (lambda a: torch.from_numpy(a).to(dev))
    got = _h(bh.attention(_t(q, dev), 0, cache(k), cache(v), n_kv)).reshape(n, n_head, hd)
    p = np.exp(-delta)
    tail = np.arange(n)[:, None] * p  # row i sees i positions of the tail
    ref = (tail / (1.0 + tail))[..., None] * np.repeat(vals.reshape(n_kv, hd), n_head // n_kv, axis=0)
    rel = np.abs(got[1:] / ref[1:] - 1.0).max()
    _say("sink and tail", "f16" if f16 else "f32", rel)
    assert rel <= 2.0 ** -20 + 48 * 2.0 ** -24


def test_attention_wide_rows_large_values(bh, oracle, synth, dev):
    """Values within a factor of ten of the largest f32: a row's sum of p v is
    past it before the division, its result is not."""
    n, n_head, n_kv, hd = 320, 192, 32, 256
    q, kc, vc = _case(synth, n, 0, n_head, n_kv, hd, 91, qscale=1.0)
    vc = (np.float32(4e37) + vc * np.float32(1e36)).astype(np.float32)
    ref = oracle.attention(q, 0, kc, vc, n_kv)
    got = _run(bh, dev, q, 0, kc, vc, n_kv)
    assert np.isfinite(got).all()
    err = rel_err(got, ref)
    _say("wide rows, large values", err)
    assert err <= TOL


_SPLIT_CAPTURE_SCRIPT = r'''
import sys
import torch
sys.path.insert(0, sys.argv[1])
from conftest import load_bonsai
bh = load_bonsai()
dev = torch.device("cuda:0")
n_head, n_kv, hd, n = 8, 1, 256, 32 * 223
k, v = torch.randn((n, n_kv * hd), device=dev), torch.randn((n, n_kv * hd), device=dev)
qs = {t: torch.randn((t, n_head, hd), device=dev) for t in (2000, 120)}
s = torch.cuda.Stream(device=dev)
torch.cuda.synchronize()
bh.attention(qs[2000], n - 2000, k, v, n_kv, stream=s)
torch.cuda.synchronize()
out = torch.empty_like(qs[120])
g = torch.cuda.CUDAGraph()
with torch.cuda.graph(g, stream=s):
    bh.attention(qs[120], n - 120, k, v, n_kv, out=out, stream=s)
want = bh.attention(qs[120], n - 120, k, v, n_kv)
torch.cuda.synchronize()
for rep in range(3):
    out.fill_(float("nan"))
    torch.cuda.synchronize()
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want), rep
print("capture ok")
'''


def test_attention_split_scratch_of_fewer_queries(dev):
    """Over the same positions of an f32 cache, a call of 2000 queries (the
    32-row form's records) prepares the capture of 120 (the 16-row form's split
    halves, 223 tiles of one kv head: sizes whose rounding differs).  Runs in a
    fresh process so no earlier call has grown the scratch."""
    import subprocess
    import sys
    from pathlib import Path
    here = Path(__file__).resolve().parent
    res = subprocess.run([sys.executable, "-c", _SPLIT_CAPTURE_SCRIPT, str(here)], capture_output=True,
                         text=True, timeout=100)
    print(res.stdout[-2000:], res.stderr[-2000:])
    assert res.returncode == 0 and "capture ok" in res.stdout
