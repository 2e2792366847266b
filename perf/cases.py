"""The work that a program serving Ternary-Bonsai-27B has this library do.

Each case is one block of a forward pass on the model's own shapes (hidden
size 5120, feed-forward 17408, 24 query and 4 key/value heads of 256, a
gated-delta-net of 16 q/k and 48 v heads of 128, a vocabulary of 248320),
called through the Python binding with the buffers, weights and argument
blocks that such a program keeps between calls:

  embed  the first call of a pass: PQ2_0 rows gathered, first RMSNorm
  mlp    the feed-forward block: residual add + RMSNorm, gate and up
         products, SiLU gate, down product
  attn   the attention block: per-head norms + IMROPE + gate split, the KV
         cache append, attention over the cache (f32, f16, planar-quantized)
  gdn    the recurrent block: conv + SiLU + L2 norms + gates, the
         gated-delta-net recurrence, the output norm and gate
  head   the final RMSNorm, the vocabulary product, the sampler's softmax

Tokens `t` run from one (decode) over short ragged prompts and chunks to
2048-token prefill; caches from empty to 32768 positions.
"""
import importlib
import math

import numpy as np
import torch

bh = importlib.import_module("ternary-bonsai-inference_amd")

N_EMBD, N_FF, N_VOCAB, EPS = 5120, 17408, 248320, 1e-6
NQ, NKV, HD, N_ROT, SECTIONS, FREQ = 24, 4, 256, 64, (11, 11, 10, 0), 1e7
HK, HV, GS, CONV_K = 16, 48, 128, 4
QK_DIM, V_DIM = HK * GS, HV * GS
TEMP = 0.7


def listed():
    return [
        # the first call of every decoded token: one id
        {"name": "embed_decode", "kind": "embed", "t": 1},
        # the same call for a prompt
        {"name": "embed_prompt", "kind": "embed", "t": 2048},
        # 64 of these a decoded token: three weight matrices read for one column
        {"name": "mlp_decode", "kind": "mlp", "t": 1},
        # a short prompt, a draft being verified or a batch of decoders: ragged
        {"name": "mlp_short", "kind": "mlp", "t": 61},
        # a long prompt
        {"name": "mlp_prefill", "kind": "mlp", "t": 2048},
        # one token against a conversation, the default f32 cache
        {"name": "attn_decode_f32", "kind": "attn", "t": 1, "pos0": 8191, "kv": "f32"},
        # one token against a long document, 4-bit planar cache
        {"name": "attn_decode_planar4", "kind": "attn", "t": 1, "pos0": 30000, "kv": "planar4"},
        # a follow-up message in a conversation, f16 cache: ragged chunk
        {"name": "attn_chunk_f16", "kind": "attn", "t": 333, "pos0": 4000, "kv": "f16"},
        # a long prompt from an empty cache
        {"name": "attn_prefill_f32", "kind": "attn", "t": 2048, "pos0": 0, "kv": "f32"},
        # the recurrent layers of one decoded token
        {"name": "gdn_decode", "kind": "gdn", "t": 1},
        # and of a prompt, not a whole number of chunks
        {"name": "gdn_prefill", "kind": "gdn", "t": 2000},
        # the end of every decoded token: logits and sampling probabilities
        {"name": "head_decode", "kind": "head", "t": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["embed", "mlp", "mlp", "attn", "attn", "gdn", "head"])
    if kind == "embed":
        return {"kind": kind, "t": _log(rng, 1, 8192)}
    if kind == "mlp":
        return {"kind": kind, "t": _log(rng, 1, 2000)}
    if kind == "gdn":
        return {"kind": kind, "t": _log(rng, 1, 2048)}
    if kind == "head":  # one sequence, or the rows of a verified draft or a batch
        return {"kind": kind, "t": _log(rng, 1, 32)}
    t = rng.choice([1, _log(rng, 2, 2000)])
    most = min(32768 - t, 2000000 // t)
    pos0 = rng.choice([0, _log(rng, 1, most)]) if t > 1 else _log(rng, 16, most)
    kv = rng.choice(["f32", "f32", "f16", "planar4", "planar3", "planar8", "planar4k"])
    return {"kind": kind, "t": t, "pos0": pos0, "kv": kv}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, mean=0.0, std=1.0):
    return torch.randn(shape, device="cuda", generator=g) * std + mean


def _pq2(g, rows, ne0):
    """A PQ2_0 tensor: codes 0, 1, 2 (30/40/30 %), f16 block scales |N(0, 0.02)|."""
    nblk = ne0 // 128
    out = torch.empty((rows, nblk, 34), dtype=torch.uint8, device="cuda")
    for r in range(0, rows, 32768):
        n = min(32768, rows - r)
        u = torch.randint(0, 10, (n, nblk, 32, 4), dtype=torch.uint8, device="cuda", generator=g)
        c = (u >= 3).to(torch.uint8) + (u >= 7).to(torch.uint8)
        out[r:r + n, :, 2:] = c[..., 0] | (c[..., 1] << 2) | (c[..., 2] << 4) | (c[..., 3] << 6)
        sc = _randn(g, n, nblk, std=0.02).abs().to(torch.float16)
        out[r:r + n, :, :2] = sc.view(torch.uint8).view(n, nblk, 2)
    return out.view(-1)


def _planar(kv):
    """(bits, whether V is quantized too) of "planar4", "planar4k", ...; None otherwise."""
    return (int(kv[6]), not kv.endswith("k")) if kv.startswith("planar") else None


def _pack(idx, bits):
    """Centroid indices [..., 256] as one little-endian bitstream a row."""
    shifts = torch.arange(bits, device=idx.device)
    b = ((idx.to(torch.int64).unsqueeze(-1) >> shifts) & 1).flatten(-2)
    w = 1 << torch.arange(8, device=idx.device)
    return (b.view(*b.shape[:-1], -1, 8) * w).sum(-1).to(torch.uint8)


def _past_planar(g, n, bits):
    """A filled planar cache of n positions: indices of normal coordinates, norms about 16."""
    cent, _ = _codebook(bits)
    mid = torch.tensor((cent[1:] + cent[:-1]) / 2, dtype=torch.float32, device="cuda")
    idx = torch.bucketize(_randn(g, n, NKV, HD, std=1 / 16), mid)
    return idx, _randn(g, n, NKV, mean=16.0, std=0.7)


def _attn_inputs(case, g):
    t, pos0, kv = case["t"], case["pos0"], case["kv"]
    s = {"q": _randn(g, t, NQ, 2 * HD), "k": _randn(g, t, NKV, HD), "v": _randn(g, t, NKV * HD),
         "wq": _randn(g, HD, mean=1.0, std=0.1), "wk": _randn(g, HD, mean=1.0, std=0.1)}
    pl = _planar(kv)
    if pl is None:
        s["kpast"], s["vpast"] = _randn(g, pos0, NKV * HD), _randn(g, pos0, NKV * HD)
    else:
        s["kpast"] = _past_planar(g, pos0, pl[0])
        s["vpast"] = _past_planar(g, pos0, pl[0]) if pl[1] else _randn(g, pos0, NKV * HD)
    return s


def _gdn_inputs(case, g):
    t = case["t"]
    return {"qkv": [_randn(g, t, d) for d in (QK_DIM, QK_DIM, V_DIM)],
            "conv_w": [_randn(g, d, CONV_K, std=0.5) for d in (QK_DIM, QK_DIM, V_DIM)],
            "conv_state": [_randn(g, d, CONV_K - 1) for d in (QK_DIM, QK_DIM, V_DIM)],
            "z": _randn(g, t, V_DIM), "alpha": _randn(g, t, HV, std=0.5), "beta": _randn(g, t, HV),
            "dt_bias": _randn(g, HV, std=0.5),
            "ssm_a": -torch.exp(2 * torch.rand(HV, device="cuda", generator=g)) / 8,
            "state": _randn(g, HV, GS, GS, std=0.1), "w": _randn(g, GS, mean=1.0, std=0.1)}


def _inputs(case, seed):
    g, t, kind = _gen(seed), case["t"], case["kind"]
    if kind == "embed":
        ids = torch.randint(0, N_VOCAB, (t,), device="cuda", generator=g, dtype=torch.int32)
        return {"table": _pq2(g, N_VOCAB, N_EMBD), "ids": ids,
                "w": _randn(g, N_EMBD, mean=1.0, std=0.1)}
    if kind == "mlp":
        return {"x": _randn(g, t, N_EMBD), "r": _randn(g, t, N_EMBD, std=0.5),
                "w": _randn(g, N_EMBD, mean=1.0, std=0.1), "gate": _pq2(g, N_FF, N_EMBD),
                "up": _pq2(g, N_FF, N_EMBD), "down": _pq2(g, N_EMBD, N_FF)}
    if kind == "head":
        return {"x": _randn(g, t, N_EMBD), "w": _randn(g, N_EMBD, mean=1.0, std=0.1),
                "table": _pq2(g, N_VOCAB, N_EMBD)}
    return _attn_inputs(case, g) if kind == "attn" else _gdn_inputs(case, g)


def prepare(case, seed):
    s, t, kind = _inputs(case, seed), case["t"], case["kind"]
    s.update(case)
    s["stream"] = torch.cuda.current_stream()
    new = lambda *shape: torch.empty(shape, device="cuda")  # noqa: E731
    if kind == "embed":
        s["out"], s["out_norm"] = new(t, N_EMBD), new(t, N_EMBD)
    elif kind == "mlp":
        s["sum"], s["norm"], s["y"] = new(t, N_EMBD), new(t, N_EMBD), new(t, N_EMBD)
        s["g"], s["u"] = new(t, N_FF), new(t, N_FF)
        if t == 1:  # one column goes through the matrix-vector call
            for k in ("norm", "y", "g", "u"):
                s[k] = s[k].view(-1)
    elif kind == "head":
        s["norm"], s["logits"], s["probs"] = new(t, N_EMBD), new(t, N_VOCAB), new(t, N_VOCAB)
    elif kind == "attn":
        _prepare_attn(s, new)
    else:
        _prepare_gdn(s, new)
    return s


def _prepare_attn(s, new):
    t, pos0, pl = s["t"], s["pos0"], _planar(s["kv"])
    n = pos0 + t
    pos = torch.arange(pos0, n, device="cuda", dtype=torch.int32)
    s["pos"] = pos[:, None].repeat(1, 4).contiguous()
    s["qr"], s["kr"], s["gate"], s["out"] = (new(t, NQ, HD), new(t, NKV, HD), new(t, NQ, HD),
                                             new(t, NQ, HD))
    s["qk"] = bh.make_qk_args(s["q"], s["qr"], s["k"], s["kr"], s["wq"], s["wk"], s["pos"], t, NQ,
                              NKV, q_head_stride=2 * HD, gate_out=s["gate"])
    if pl is None:
        dt = torch.float32 if s["kv"] == "f32" else torch.float16
        for c, past in (("kc", "kpast"), ("vc", "vpast")):
            s[c] = torch.zeros((n, NKV * HD), device="cuda", dtype=dt)
            s[c][:pos0] = s.pop(past).to(dt)
        return

    def cache(past):
        idx, norm = past
        q = torch.zeros((n, NKV, 32 * pl[0]), device="cuda", dtype=torch.uint8)
        f = torch.zeros((n, NKV), device="cuda")
        for r in range(0, pos0, 8192):
            q[r:min(pos0, r + 8192)] = _pack(idx[r:r + 8192], pl[0])
        f[:pos0] = norm
        return q, f

    s["kq"], s["kn"] = cache(s.pop("kpast"))
    s["vq"] = s["vn"] = s["vf"] = None
    if pl[1]:
        s["vq"], s["vn"] = cache(s.pop("vpast"))
    else:
        s["vf"] = torch.zeros((n, NKV * HD), device="cuda")
        s["vf"][:pos0] = s.pop("vpast")


def _prepare_gdn(s, new):
    t = s["t"]
    s["g"], s["b"] = new(t, HV), new(t, HV)
    s["attn"], s["norm"], s["y"] = new(t, HV, GS), new(t * HV, GS), new(t, V_DIM)
    gates = dict(alpha_raw=s["alpha"], dt_bias=s["dt_bias"], ssm_a=s["ssm_a"], beta_raw=s["beta"],
                 gate_out=s["g"], beta_out=s["b"], n_v_head=HV)
    if t == 1:  # one row is whole: q, k and v are its parts
        s["conv_in"], s["conv_out"] = torch.cat(s["qkv"], 1), new(1, 2 * QK_DIM + V_DIM)
        s["w_all"], s["state_all"] = torch.cat(s["conv_w"]), torch.cat(s["conv_state"])
        s["prep"] = [bh.make_gdn_args(s["conv_in"], s["conv_out"], n_tok=t,
                                      conv_dim=2 * QK_DIM + V_DIM, l2_dim=2 * QK_DIM,
                                      conv_w=s["w_all"], conv_state=s["state_all"],
                                      conv_k=CONV_K, **gates)]
        parts = torch.split(s["conv_out"], [QK_DIM, QK_DIM, V_DIM], 1)
        s["conv_state"] = [s["state_all"]]
    else:  # q, k and v come from products of their own rows: one call for each
        parts = [new(t, d) for d in (QK_DIM, QK_DIM, V_DIM)]
        s["prep"] = [bh.make_gdn_args(s["qkv"][i], parts[i], n_tok=t, conv_dim=d,
                                      l2_dim=d if i < 2 else 0, conv_w=s["conv_w"][i],
                                      conv_state=s["conv_state"][i], conv_k=CONV_K,
                                      **(gates if i == 2 else {}))
                     for i, d in enumerate((QK_DIM, QK_DIM, V_DIM))]
    s["qc"], s["kc"], s["vc"] = (p.view(t, -1, GS) for p in parts)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(s):
    return {"embed": _run_embed, "mlp": _run_mlp, "head": _run_head, "attn": _run_attn,
            "gdn": _run_gdn}[s["kind"]](s, s["stream"])


def _run_embed(s, st):
    return bh.pq2_embed_gather(s["table"], N_EMBD, N_VOCAB, s["ids"], out=s["out"], w=s["w"],
                               out_norm=s["out_norm"], stream=st)


def _run_mlp(s, st):
    bh.add_rms_norm_rows(s["x"], s["r"], s["w"], sum_out=s["sum"], out=s["norm"], stream=st)
    bh.pq2_matmul_n(s["gate"], N_EMBD, N_FF, s["norm"], out=s["g"], stream=st)
    bh.pq2_matmul_n(s["up"], N_EMBD, N_FF, s["norm"], out=s["u"], stream=st)
    bh.unary(bh.BH_SILU_MUL, s["g"], s["u"], out=s["g"], stream=st)
    bh.pq2_matmul_n(s["down"], N_FF, N_EMBD, s["g"], out=s["y"], stream=st)
    return s["sum"], s["y"]


def _run_head(s, st):
    bh.rms_norm_rows(s["x"], s["w"], out=s["norm"], stream=st)
    one = s["t"] == 1
    bh.pq2_matmul_n(s["table"], N_EMBD, N_VOCAB, s["norm"].view(-1) if one else s["norm"],
                    out=s["logits"].view(-1) if one else s["logits"], stream=st)
    bh.softmax_rows(s["logits"], N_VOCAB, 1.0 / TEMP, out=s["probs"], stream=st)
    return s["logits"], s["probs"]


def _run_attn(s, st):
    bh.qk_norm_rope(s["qk"], stream=st)
    pl, t, pos0 = _planar(s["kv"]), s["t"], s["pos0"]
    if pl is None:
        bh.kv_store(s["kr"].view(t, -1), s["v"], s["kc"], s["vc"], pos0, stream=st)
        bh.attention(s["qr"], pos0, s["kc"], s["vc"], NKV, out=s["out"], stream=st)
        return s["out"], s["gate"], s["kc"], s["vc"]
    bh.kv_store_planar(s["kr"].view(t, -1), s["v"], pos0, NKV, pl[0], s["kq"], s["kn"], s["vq"],
                       s["vn"], s["vf"], stream=st)
    bh.attention_planar(s["qr"], pos0, s["kq"], s["kn"], NKV, pl[0], s["vq"], s["vn"], s["vf"],
                        out=s["out"], stream=st)
    return s["out"], s["gate"], s["kq"], s["kn"], *((s["vq"], s["vn"]) if pl[1] else (s["vf"],))


def _run_gdn(s, st):
    for a in s["prep"]:
        bh.gdn_prep_fused(a, stream=st)
    bh.gdn_step(s["qc"], s["kc"], s["vc"], s["g"], s["b"], s["state"], attn=s["attn"], stream=st)
    bh.rms_norm_rows(s["attn"].view(-1, GS), s["w"], out=s["norm"], stream=st)
    bh.unary(bh.BH_SILU_MUL, s["z"], s["norm"], out=s["y"], stream=st)
    return s["y"], s["state"], *s["conv_state"]


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how exact its results are
# ---------------------------------------------------------------------------

def work(case):
    t, kind, f = case["t"], case["kind"], 4
    row, ff, vocab = N_EMBD // 128 * 34, N_FF // 128 * 34, N_VOCAB
    if kind == "embed":
        return {"bytes": t * (4 + row + 2 * f * N_EMBD) + f * N_EMBD, "flops": 5 * t * N_EMBD}
    if kind == "mlp":
        return {"bytes": 2 * N_FF * row + N_EMBD * ff + 4 * t * f * N_EMBD + f * N_EMBD,
                "flops": 6 * t * N_FF * N_EMBD}
    if kind == "head":
        return {"bytes": vocab * row + t * f * (N_EMBD + 2 * vocab), "flops": 2 * t * vocab * N_EMBD}
    if kind == "attn":
        pos0, kv, n = case["pos0"], case["kv"], case["pos0"] + case["t"]
        pl, el = _planar(kv), NKV * HD
        kb = {"f32": 4 * el, "f16": 2 * el}.get(kv) or NKV * (32 * pl[0] + 4)
        vb = kb if pl is None or pl[1] else 4 * el
        pairs = t * pos0 + t * (t + 1) // 2
        return {"bytes": t * f * (4 * NQ * HD + 2 * el + 4) + n * (kb + vb),
                "flops": 4 * HD * NQ * pairs}
    state = 2 * f * (HV * GS * GS + (2 * QK_DIM + V_DIM) * (CONV_K - 1))
    per = f * (2 * QK_DIM + V_DIM + 2 * HV + 2 * V_DIM)
    return {"bytes": state + t * per + f * (2 * QK_DIM + V_DIM) * CONV_K,
            "flops": t * (HV * GS * GS * 7 + 2 * CONV_K * (2 * QK_DIM + V_DIM))}


def tolerance(case):
    """About four times what the kernels' 32-bit sums are off the 64-bit results below."""
    if case["kind"] == "embed":  # 5120 squares summed one after the other: 2.5e-6 .. 3.6e-6 off
        return {"rel": 1.5e-5}
    if case["kind"] == "attn" and case["kv"].startswith("planar"):
        # 3.3e-6 off; and a rounding at the edge of a quantizer cell may move an index of an
        # appended row, its neighbour's value then standing for one of its 256 coordinates
        return {"rel": 4e-5, "differ": 1e-4}
    return {"rel": 4e-6}  # mlp 8e-7, head 9e-7, attn 2e-7 .. 1e-6, gdn 2e-7 off


# ---------------------------------------------------------------------------
# the same passes in 64 bits
# ---------------------------------------------------------------------------

def _codebook(bits):
    """The 2^bits Lloyd-Max centroids of a normal coordinate of a unit vector
    of 256, and the rotation (cos, sin) of each coordinate pair (f32 values)."""
    n, sg = 1 << bits, 1 / 16
    erf_c = (1.061405429, -1.453152027, 1.421413741, -0.284496736, 0.254829592)

    def cdf(x):
        a = np.abs(x / (sg * math.sqrt(2)))
        u, y = 1 / (1 + 0.3275911 * a), 0.0
        for c in erf_c:
            y = (y + c) * u
        return 0.5 * (1 + np.sign(x) * (1 - y * np.exp(-a * a)))

    def pdf(x):
        return np.exp(-x * x / (2 * sg * sg)) / (sg * math.sqrt(2 * math.pi))

    c = -3.5 * sg + 7 * sg * (np.arange(n) + 0.5) / n
    for _ in range(300):
        e = np.concatenate([[-12 * sg], (c[1:] + c[:-1]) / 2, [12 * sg]])
        mass = cdf(e[1:]) - cdf(e[:-1])
        m1 = sg * sg * (pdf(e[:-1]) - pdf(e[1:]))
        nx = np.where(mass > 1e-15, m1 / np.where(mass > 1e-15, mass, 1.0), c)
        shift, c = np.max(np.abs(nx - c)), nx
        if shift < 1e-12:
            break
    st, ang = 42, []
    for _ in range(HD // 2):
        st = (st + 0x9E3779B97F4A7C15) % 2**64
        z = (st ^ (st >> 30)) * 0xBF58476D1CE4E5B9 % 2**64
        z = (z ^ (z >> 27)) * 0x94D049BB133111EB % 2**64
        ang.append(((z ^ (z >> 31)) >> 11) / 2**53 * 2 * math.pi)
    f = lambda a: np.asarray(a, np.float32).astype(np.float64)  # noqa: E731
    return f(c), (f(np.cos(ang)), f(np.sin(ang)))


def _weights(table, ne0, lo, hi):
    """Rows lo .. hi of a PQ2_0 tensor in 64 bits."""
    b = table.view(-1, ne0 // 128, 34)[lo:hi]
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    c = torch.stack([(b[:, :, 2:] >> (2 * k)) & 3 for k in range(4)], -1).view(*b.shape[:2], 128)
    return ((c.double() - 1) * d).view(-1, ne0)


def _product(table, ne0, x):
    rows = table.numel() // (ne0 // 128 * 34)
    return torch.cat([x @ _weights(table, ne0, r, min(rows, r + 8192)).T
                      for r in range(0, rows, 8192)], 1)


def _rms(x, w):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def exact(case, seed):
    s, kind, t = _inputs(case, seed), case["kind"], case["t"]
    if kind == "embed":
        tab = s["table"].view(N_VOCAB, -1)[s["ids"].long()].contiguous()
        e = _weights(tab, N_EMBD, 0, t)
        return e, _rms(e, s["w"].double())
    if kind == "mlp":
        x = s["x"].double() + s["r"].double()
        n = _rms(x, s["w"].double())
        g, u = _product(s["gate"], N_EMBD, n), _product(s["up"], N_EMBD, n)
        y = _product(s["down"], N_FF, g * torch.sigmoid(g) * u)
        return x, y.view(-1) if t == 1 else y
    if kind == "head":
        y = _product(s["table"], N_EMBD, _rms(s["x"].double(), s["w"].double()))
        return y, torch.softmax(y * float(np.float32(1.0 / TEMP)), -1)
    return _exact_attn(case, s) if kind == "attn" else _exact_gdn(case, s)


def _rope(x, pos0):
    """The rotation of the first N_ROT values of heads [t, h, HD], text positions."""
    t, half = x.shape[0], N_ROT // 2
    # an angle is defined by its chain of 32-bit products, p * scale * scale ..
    scale = np.float32(FREQ) ** np.float32(-2.0 / N_ROT)
    th = [np.arange(pos0, pos0 + t).astype(np.float32)]
    while len(th) < half:
        th.append(th[-1] * scale)
    th = torch.tensor(np.stack(th, -1), device="cuda").double()[:, None]
    a, b = x[..., :half], x[..., half:N_ROT]
    c, s = torch.cos(th), torch.sin(th)
    return torch.cat([a * c - b * s, a * s + b * c, x[..., N_ROT:]], -1)


def _exact_attn(case, s):
    t, pos0, pl = case["t"], case["pos0"], _planar(case["kv"])
    q = _rope(_rms(s["q"][..., :HD].double(), s["wq"].double()), pos0)
    gate = torch.sigmoid(s["q"][..., HD:].double())
    k = _rope(_rms(s["k"].double(), s["wk"].double()), pos0)
    v = s["v"].double().view(t, NKV, HD)
    if pl is None:
        half = case["kv"] == "f16"
        kept = (lambda a: a.half().double()) if half else (lambda a: a)
        kc, vc = (kept(torch.cat([s[p].double().view(pos0, NKV, HD), a]))
                  for p, a in (("kpast", k), ("vpast", v)))
        caches = [None, None] if half else [kc.view(-1, NKV * HD), vc.view(-1, NKV * HD)]
    else:
        cent, rot = _codebook(pl[0])
        cent, (co, si) = torch.tensor(cent, device="cuda"), (torch.tensor(a, device="cuda")
                                                             for a in rot)

        def turn(x, back=False):
            a, b, sn = x[..., ::2], x[..., 1::2], -si if back else si
            return torch.stack([co * a - sn * b, sn * a + co * b], -1).flatten(-2)

        def kept(past, x):  # what the cache holds: rotated rows of centroids, and norms
            norm = x.square().sum(-1).sqrt()
            idx = torch.bucketize(turn(x / norm[..., None]), (cent[1:] + cent[:-1]) / 2)
            n = torch.cat([past[1].double(), norm])
            return cent[torch.cat([past[0], idx])] * n[..., None], n

        q = turn(q)
        kc, kn = kept(s["kpast"], k)
        if pl[1]:
            vc, vn = kept(s["vpast"], v)
            caches = [None, kn, None, vn]
        else:
            vc = torch.cat([s["vpast"].double().view(pos0, NKV, HD), v])
            caches = [None, kn, vc.reshape(-1, NKV * HD)]
    out, rep = torch.empty((t, NQ, HD), device="cuda", dtype=torch.float64), NQ // NKV
    seen = torch.arange(pos0, pos0 + t, device="cuda")
    for h in range(NQ):
        for i in range(0, t, 512):
            n = min(t, i + 512) + pos0
            sc = q[i:i + 512, h] @ kc[:n, h // rep].T / math.sqrt(HD)
            sc.masked_fill_(torch.arange(n, device="cuda") > seen[i:i + 512, None], -math.inf)
            out[i:i + 512, h] = torch.softmax(sc, -1) @ vc[:n, h // rep]
    if pl is not None and pl[1]:
        out = turn(out, back=True)
    return (out, gate, *caches)


def _exact_gdn(case, s):
    t, done, states = case["t"], [], []
    for i, (x, w, st) in enumerate(zip(s["qkv"], s["conv_w"], s["conv_state"])):
        whole = torch.cat([st.double().T, x.double()])
        y = sum(whole[j:j + t] * w[:, j].double() for j in range(CONV_K))
        y = (y * torch.sigmoid(y)).view(t, -1, GS)
        if i < 2:
            y = y / y.square().sum(-1, keepdim=True).sqrt().clamp_min(EPS)
        done.append(y)
        states.append(whole[t:].T.contiguous())
    q, k, v = done
    q, k = q.repeat(1, HV // HK, 1), k.repeat(1, HV // HK, 1)
    a = torch.nn.functional.softplus(s["alpha"].double() + s["dt_bias"].double(), threshold=50)
    a, b = torch.exp(a * s["ssm_a"].double()), torch.sigmoid(s["beta"].double())
    m, attn = s["state"].double(), torch.empty((t, HV, GS), device="cuda", dtype=torch.float64)
    for i in range(t):
        m = m * a[i, :, None, None]
        d = (v[i] - (m * k[i, :, None]).sum(-1)) * b[i, :, None]
        m = m + d[..., None] * k[i, :, None]
        attn[i] = (m * q[i, :, None]).sum(-1) / math.sqrt(GS)
    z = s["z"].double()
    y = z * torch.sigmoid(z) * _rms(attn, s["w"].double()).view(t, -1)
    return (y, m, torch.cat(states)) if t == 1 else (y, m, *states)
