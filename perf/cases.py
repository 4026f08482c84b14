"""The workloads whose time counts for a user of cmf_amd, each through the
package's public entry points:

  gemv      y = W x on device pointers for 1..16 rows (cmf_gemv_dev_noalloc):
            one projection of a decode step, a verify batch or a serving loop
  ffn       cmf_amd.ffn on host rows: the SwiGLU seam call an engine makes per
            layer when it keeps its activations on the host
  moe       the routed-expert FFN of a verify batch on device pointers
            (cmf_moe_ffn_dev)
  prefill   Model.prefill of a prompt (dense and routed-expert models)
  generate  Model.decode from a prefilled prompt: plain or speculative,
            greedy, sampled, short and long contexts

Weights are random-init N(0, 0.02) quantized to the codec under test (q8 per
row, q4t 32-weight tiles, q4tp tiles on a 32-rung ladder), activations N(0, 1).
Shapes are those of the benchmark configurations (Qwen3-0.6B-arch decoder,
Qwen3-8B FFN matrices, the 128-expert 2048/768 MoE layer) and generic ones.
"""
import math

import numpy as np
import torch

import cmf_amd
from cmf_amd import model as cmf_model
from cmf_amd import moe as cmf_moe

DT = {"q8": cmf_amd.DT_Q8ROW, "q4t": cmf_amd.DT_Q4T, "q4tp": cmf_amd.DT_Q4TP}
EPS, THETA, HEAD = 1e-6, 1e6, 128

# the Qwen3-0.6B-arch decoder of the headline benchmark (q8 attention, q4t FFN)
QWEN06B = dict(layers=28, hidden=1024, heads=16, kv=8, inter=3072, vocab=151936, attn="q8", ffn="q4t", mtp=True,
               experts=0, top_k=0, moe_inter=0)
# a wider generic decoder, outside the shape of the fused decode blocks
WIDE = dict(layers=4, hidden=2048, heads=16, kv=8, inter=6144, vocab=32768, attn="q8", ffn="q4t", mtp=False,
            experts=0, top_k=0, moe_inter=0)
# a routed-expert block (128 experts of 2048/768, top 8) under a dense one,
# whose keys and values depend on every routed row
MOE2 = dict(layers=2, hidden=2048, heads=16, kv=8, inter=6144, vocab=32768, attn="q8", ffn="q4t", mtp=False,
            experts=128, top_k=8, moe_inter=768)


def listed():
    return [
        # a KV projection of a small decoder, one token: launch latency
        dict(name="gemv_q8_1024x1024_m1", kind="gemv", dtype="q8", rows=1024, cols=1024, m=1),
        # Qwen3-8B gate/up at one token: the memory roofline case
        dict(name="gemv_q4t_12288x4096_m1", kind="gemv", dtype="q4t", rows=12288, cols=4096, m=1),
        # the same for a K = 4 verify batch in the ladder codec
        dict(name="gemv_q4tp_12288x4096_m5", kind="gemv", dtype="q4tp", rows=12288, cols=4096, m=5),
        # the down projection for a batch of 13 sequences (odd batch, long rows)
        dict(name="gemv_q4t_4096x12288_m13", kind="gemv", dtype="q4t", rows=4096, cols=12288, m=13),
        # Qwen3-8B FFN of a verify batch from host rows
        dict(name="ffn_q4t_4096x12288_b5", kind="ffn", dtype="q4t", hidden=4096, inter=12288, b=5),
        # FFN of a prompt chunk from host rows, ladder codec, ragged batch
        dict(name="ffn_q4tp_2048x6144_b200", kind="ffn", dtype="q4tp", hidden=2048, inter=6144, b=200),
        # the routed layer of a K = 4 verify batch
        dict(name="moe_q4t_128x8_b5", kind="moe", dtype="q4t", experts=128, top_k=8, hidden=2048, inter=768, b=5),
        # a full 16-token batch over q8 experts
        dict(name="moe_q8_64x8_b16", kind="moe", dtype="q8", experts=64, top_k=8, hidden=1024, inter=512, b=16),
        # prompt processing of the headline model
        dict(name="prefill_qwen06b_2048", kind="prefill", n=2048, **QWEN06B),
        # prompt processing of a routed-expert model
        dict(name="prefill_moe_600", kind="prefill", n=600, **MOE2),
        # speculative decode of the headline model at context 2048
        dict(name="generate_qwen06b_spec_2048", kind="generate", ctx=2048, tokens=12, spec=4, temp=0.0, **QWEN06B),
        # plain decode at a long context
        dict(name="generate_wide_plain_12000", kind="generate", ctx=12000, tokens=12, spec=0, temp=0.0, **WIDE),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "ffn", "moe", "prefill", "prefill", "generate"])
    dt = rng.choice(["q8", "q4t", "q4tp"])
    if kind == "gemv":
        return dict(kind=kind, dtype=dt, rows=_log(rng, 512, 16384), cols=32 * _log(rng, 24, 384), m=rng.randint(1, 16))
    if kind == "ffn":
        return dict(kind=kind, dtype=dt, hidden=32 * _log(rng, 32, 128), inter=32 * _log(rng, 64, 384),
                    b=_log(rng, 1, 256))
    if kind == "moe":
        return dict(kind=kind, dtype=dt, experts=rng.choice([32, 64, 128]), top_k=rng.choice([2, 4, 8]),
                    hidden=128 * rng.randint(8, 16), inter=32 * rng.randint(12, 24), b=rng.randint(1, 16))
    hidden = rng.choice([512, 768, 1024, 2048])
    shape = dict(layers=rng.randint(2, 4), hidden=hidden, heads=hidden // HEAD, kv=hidden // (HEAD * rng.choice([1, 2])),
                 inter=hidden * 3, vocab=32768, attn=rng.choice(["q8", "q8", "q4t"]), ffn=dt, mtp=False, experts=0,
                 top_k=0, moe_inter=0)
    if kind == "prefill":
        if rng.random() < 0.3:
            shape.update(layers=2, experts=rng.choice([32, 64]), top_k=rng.choice([4, 8]), moe_inter=32 * rng.randint(8, 24))
        return dict(kind=kind, n=_log(rng, 16, 600 if shape["experts"] else 3000), **shape)
    if rng.random() < 0.4:
        shape.update(hidden=1024, heads=16, kv=8, inter=3072, attn="q8", ffn="q4t")
    spec = rng.choice([0, 2, 4])
    shape["mtp"] = spec > 0
    return dict(kind=kind, ctx=_log(rng, 64, 12000), tokens=rng.randint(6, 14), spec=spec,
                temp=rng.choice([0.0, 0.0, 0.8]), **shape)


# --------------------------------------------------------------------------
# inputs: random-init weights, quantized on the GPU into the upload formats
# --------------------------------------------------------------------------
class _Rng:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 17)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std

    def ids(self, n, vocab):
        return torch.randint(0, vocab, (n,), generator=self.g, device="cuda")


def _tiles(w, scale):
    """Nibble bytes [..., 16] of 32-weight tiles w [..., 32] over their scales."""
    n = (torch.round(w / scale.unsqueeze(-1)) + 8).clamp_(0, 15).to(torch.uint8)
    return n[..., 0::2] | (n[..., 1::2] << 4)


def _host(t):
    return t.cpu().numpy()


def quantize(dtype, w):
    """w [rows, cols] f32 (GPU) as the tensor dict the loader hands to Model."""
    rows, cols = w.shape
    out = dict(dtype=DT[dtype], rows=rows, cols=cols, q=None, row_scale=None, bytes=None)
    if dtype == "q8":
        s = (w.abs().amax(1) / 127).half().float().clamp_min(1e-7)
        out["q"] = _host(torch.round(w / s[:, None]).clamp_(-127, 127).to(torch.int8))
        out["row_scale"] = _host(s)
        return out
    g = w.view(rows, cols // 32, 32)
    amax = (g.abs().amax(2) / 7).clamp_min(1e-6)
    if dtype == "q4t":
        h = amax.half()
        p = torch.cat([h.view(torch.uint8).view(rows, cols // 32, 2), _tiles(g, h.float())], 2)
        out["bytes"] = _host(p.reshape(-1))
        return out
    lg = torch.log2(amax)
    lo = lg.amin(1).half()
    step = ((lg.amax(1) - lo.float()) / 31).clamp_min(1e-3).half()
    code = torch.round((lg - lo.float()[:, None]) / step.float()[:, None]).clamp_(0, 31).to(torch.int64)
    scale = torch.gather(_ladder(lo, step), 1, code)
    bits = (code.unsqueeze(-1) >> torch.arange(5, device=w.device)) & 1
    bits = bits.reshape(rows, -1)
    bits = torch.nn.functional.pad(bits, (0, -bits.shape[1] % 8)).view(rows, -1, 8)
    cb = (bits << torch.arange(8, device=w.device)).sum(2).to(torch.uint8)
    params = torch.stack([lo, step], 1).view(torch.uint8)
    out["bytes"] = _host(torch.cat([_tiles(g, scale).reshape(-1), params.reshape(-1), cb.reshape(-1)]))
    return out


def _ladder(lo, step):
    """The codec's 32 rungs t[0] = 2^lo, t[c] = t[c-1] * 2^step in f32."""
    r, t = torch.exp2(step.float()), [torch.exp2(lo.float())]
    for _ in range(31):
        t.append(t[-1] * r)
    return torch.stack(t, 1)


def dequant(t):
    """The f64 matrix a quantized tensor stands for."""
    rows, cols = t["rows"], t["cols"]
    if t["q"] is not None:
        return torch.from_numpy(t["q"]).cuda().double() * torch.from_numpy(t["row_scale"]).cuda().double()[:, None]
    b, gpr = torch.from_numpy(t["bytes"]).cuda(), cols // 32
    if t["dtype"] == DT["q4t"]:
        p = b.view(rows, gpr, 18)
        s, nib = p[:, :, :2].contiguous().view(torch.float16)[:, :, 0].double(), p[:, :, 2:]
    else:
        nn = rows * gpr * 16
        nib = b[:nn].view(rows, gpr, 16)
        par = b[nn:nn + 4 * rows].contiguous().view(torch.float16).view(rows, 2)
        cb = b[nn + 4 * rows:].view(rows, -1)
        bits = ((cb.unsqueeze(-1) >> torch.arange(8, device="cuda", dtype=torch.uint8)) & 1).view(rows, -1)
        code = (bits[:, :gpr * 5].view(rows, gpr, 5).long() << torch.arange(5, device="cuda")).sum(2)
        s = torch.gather(_ladder(par[:, 0], par[:, 1]), 1, code).double()
    w = torch.stack([(nib & 15).double() - 8, (nib >> 4).double() - 8], 3).reshape(rows, gpr, 32)
    return (w * s.unsqueeze(-1)).reshape(rows, cols)


def _weight(t):
    return cmf_amd.Weight(t["dtype"], t["rows"], t["cols"], payload=t["bytes"], q=t["q"], row_scale=t["row_scale"])


def _rows(whole, part, i):
    """Tensor i of `whole` = several equal matrices quantized together."""
    r, t = part, dict(whole, rows=part)
    if whole["q"] is not None:
        t.update(q=whole["q"][i * r:(i + 1) * r], row_scale=whole["row_scale"][i * r:(i + 1) * r])
        return t
    gpr = whole["cols"] // 32
    if whole["dtype"] == DT["q4t"]:
        t["bytes"] = whole["bytes"][i * r * gpr * 18:(i + 1) * r * gpr * 18]
        return t
    n, st = whole["rows"], (gpr * 5 + 7) // 8
    cut = lambda off, per: whole["bytes"][off + i * r * per:off + (i + 1) * r * per]  # noqa: E731
    t["bytes"] = np.concatenate([cut(0, gpr * 16), cut(n * gpr * 16, 4), cut(n * gpr * 16 + 4 * n, st)])
    return t


def _experts(dtype, r, ne, hidden, inter):
    gate, up = (quantize(dtype, r.normal(ne * inter, hidden, std=0.02)) for _ in range(2))
    down = quantize(dtype, r.normal(ne * hidden, inter, std=0.02))
    return [dict(gate=_rows(gate, inter, e), up=_rows(up, inter, e), down=_rows(down, hidden, e)) for e in range(ne)]


def _norm(r, n):
    return _host(1 + r.normal(n, std=0.1))


def _layer(c, r, moe):
    h, q, kv = c["hidden"], c["heads"] * HEAD, c["kv"] * HEAD
    w = lambda dt, rows, cols: quantize(dt, r.normal(rows, cols, std=0.02))  # noqa: E731
    d = dict(input_norm=_norm(r, h), post_norm=_norm(r, h), q_norm=_norm(r, HEAD), k_norm=_norm(r, HEAD),
             wq=w(c["attn"], q, h), wk=w(c["attn"], kv, h), wv=w(c["attn"], kv, h), wo=w(c["attn"], h, q))
    if moe:
        router = _host(r.normal(c["experts"], h, std=0.1).half())
        d["moe"] = dict(router=dict(dtype=1, rows=c["experts"], cols=h, q=None, row_scale=None,
                                    bytes=router.reshape(-1).view(np.uint8)),
                        top_k=c["top_k"], norm_topk=True, routed_scaling=1.0,
                        experts=_experts(c["ffn"], r, c["experts"], h, c["moe_inter"]))
    else:
        d.update(gate=w(c["ffn"], c["inter"], h), up=w(c["ffn"], c["inter"], h), down=w(c["ffn"], h, c["inter"]))
    return d


def _positions(c):
    return c["n"] if c["kind"] == "prefill" else c["ctx"]


def weights(c, seed):
    """The model a user has loaded, and a prompt."""
    r, h = _Rng(seed), c["hidden"]
    n = _positions(c)
    ids = _host(r.ids(n, c["vocab"])).astype(np.int32)
    room = 64 if c["kind"] == "prefill" else 64 + c["tokens"] * (c["spec"] + 1)
    cfg = dict(n_layers=c["layers"], hidden=h, n_heads=c["heads"], n_kv=c["kv"], head_dim=HEAD, inter=c["inter"],
               vocab=c["vocab"], max_seq=n + room, rope_theta=THETA, eps=EPS)
    sm = dict(cfg=cfg, layers=[_layer(c, r, c["experts"] > 0 and li == 0) for li in range(c["layers"])],
              lm_head=quantize("q8", r.normal(c["vocab"], h, std=0.02)), final_norm=_norm(r, h))
    if c["mtp"]:
        sm["mtp"] = dict(enorm=_norm(r, h), hnorm=_norm(r, h), eh_proj=quantize("q8", r.normal(h, 2 * h, std=0.02)),
                         layer=_layer(c, r, False), norm=_norm(r, h))
    return sm, ids


def _gemv_inputs(c, seed):
    r = _Rng(seed)
    return quantize(c["dtype"], r.normal(c["rows"], c["cols"], std=0.02)), r.normal(c["m"], c["cols"])


def _ffn_inputs(c, seed):
    r, h, i = _Rng(seed), c["hidden"], c["inter"]
    return [quantize(c["dtype"], r.normal(a, b, std=0.02)) for a, b in ((i, h), (i, h), (h, i))], r.normal(c["b"], h)


def _moe_inputs(c, seed):
    r = _Rng(seed)
    ex = _experts(c["dtype"], r, c["experts"], c["hidden"], c["inter"])
    return ex, r.normal(c["b"], c["hidden"]), r.normal(c["b"], c["experts"])


def prepare(case, seed):
    cmf_amd.init(0)
    k = case["kind"]
    if k == "gemv":
        t, x = _gemv_inputs(case, seed)
        return dict(case=case, w=_weight(t), x=x, y=torch.empty(case["m"], case["rows"], device="cuda"))
    if k == "ffn":
        ts, x = _ffn_inputs(case, seed)
        return dict(case=case, w=[_weight(t) for t in ts], x=_host(x), y=np.empty((case["b"], case["hidden"]), np.float32))
    if k == "moe":
        ex, x, lg = _moe_inputs(case, seed)
        return dict(case=case, x=x, lg=lg, y=torch.empty_like(x),
                    moe=cmf_moe.MoE(case["experts"], case["hidden"], case["inter"], case["top_k"], ex))
    sm, ids = weights(case, seed)
    m = cmf_model.Model(sm)
    if k == "generate":
        m.prefill(ids)
    return dict(case=case, m=m, ids=ids)


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------
def run(state):
    c, k = state["case"], state["case"]["kind"]
    if k == "gemv":
        cmf_amd.check(cmf_amd.lib().cmf_gemv_dev_noalloc(state["w"].h, state["x"].data_ptr(), c["cols"], c["m"],
                                                         state["y"].data_ptr(), c["rows"]))
        return state["y"]
    if k == "ffn":
        w1, w3, w2 = state["w"]
        if not cmf_amd.ffn(w1, w3, w2, state["x"], c["b"], c["hidden"], c["inter"], state["y"]):
            raise cmf_amd.CmfError("declined")
        return state["y"]
    if k == "moe":
        cmf_amd.check(cmf_amd.lib().cmf_moe_ffn_dev(state["moe"].h, state["x"].data_ptr(), state["lg"].data_ptr(),
                                                    c["b"], state["y"].data_ptr()))
        return state["y"]
    m, ids = state["m"], state["ids"]
    if k == "prefill":
        m.prefill(ids)
        # the prompt's last hidden row and the logits of a next token on top
        # of the prompt's keys and values
        hid = m.state()[1]
        return dict(hidden=hid, next=m.forward_batch(ids[:1], len(ids))[1])
    # another answer to the same prompt: back to its last token, then generate
    # (the hidden row is recomputed over the kept keys and values)
    n = len(ids)
    hid, lg = m.forward_batch(ids[n - 1:], n - 1)
    sampler = cmf_amd.SamplerConfig(temperature=c["temp"], repetition_penalty=1.0) if c["temp"] > 0 else None
    toks, _ = m.decode(c["tokens"], sampler=sampler, seed=7, spec=c["spec"] > 0, k=max(1, c["spec"]))
    return dict(hidden=hid, logits=lg, tokens=toks[:c["tokens"]], tip=m.state()[1])


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def _wbytes(dtype, rows, cols):
    g = cols // 32
    if dtype == "q8":
        return rows * (cols + 4)
    return rows * g * 18 if dtype == "q4t" else rows * (g * 16 + 4 + (g * 5 + 7) // 8)


def _layer_work(c, li, rows, kv_read, kv_pairs, distinct):
    """Bytes and flops of one block over `rows` rows that read kv_read cached
    positions and form kv_pairs (query, key) pairs."""
    h, q, kv = c["hidden"], c["heads"] * HEAD, c["kv"] * HEAD
    b = _wbytes(c["attn"], q + 2 * kv, h) + _wbytes(c["attn"], h, q) + 8 * kv * (kv_read + rows)
    f = 2.0 * rows * h * (2 * q + 2 * kv) + 4.0 * q * kv_pairs
    if c["experts"] and li == 0:
        i = c["moe_inter"]
        b += distinct * (2 * _wbytes(c["ffn"], i, h) + _wbytes(c["ffn"], h, i)) + 4 * c["experts"] * h
        f += rows * (6.0 * h * i * c["top_k"] + 2.0 * h * c["experts"])
    else:
        b += 2 * _wbytes(c["ffn"], c["inter"], h) + _wbytes(c["ffn"], h, c["inter"])
        f += 6.0 * rows * h * c["inter"]
    return b, f


def _distinct(ne, k, rows):
    """Experts that `rows` tokens are expected to reach."""
    return ne * (1 - (1 - k / ne) ** rows)


def work(case):
    c, k = case, case["kind"]
    if k == "gemv":
        return dict(bytes=_wbytes(c["dtype"], c["rows"], c["cols"]) + 4 * c["m"] * (c["rows"] + c["cols"]),
                    flops=2.0 * c["m"] * c["rows"] * c["cols"])
    if k == "ffn":
        h, i = c["hidden"], c["inter"]
        return dict(bytes=2 * _wbytes(c["dtype"], i, h) + _wbytes(c["dtype"], h, i) + 8 * c["b"] * h,
                    flops=6.0 * c["b"] * h * i)
    if k == "moe":
        h, i, b = c["hidden"], c["inter"], c["b"]
        e = _distinct(c["experts"], c["top_k"], b)
        return dict(bytes=e * (2 * _wbytes(c["dtype"], i, h) + _wbytes(c["dtype"], h, i)) + 4 * b * (2 * h + c["experts"]),
                    flops=6.0 * b * c["top_k"] * h * i)
    tot = [0.0, 0.0]

    def add(rows, pos0, times=1, layers=None, head=1):
        pairs = rows * pos0 + rows * (rows + 1) / 2
        for li in range(c["layers"] if layers is None else layers):
            b, f = _layer_work(c, li if layers is None else 1, rows, pos0, pairs, _distinct(c["experts"] or 1, c["top_k"], rows))
            tot[0] += times * b
            tot[1] += times * f
        tot[0] += times * head * _wbytes("q8", c["vocab"], c["hidden"])
        tot[1] += times * head * 2.0 * rows * c["vocab"] * c["hidden"]

    if k == "prefill":
        add(c["n"], 0, head=0)
        add(1, c["n"])
        if c["mtp"]:
            tot[0] += _wbytes("q8", c["hidden"], 2 * c["hidden"])
            tot[1] += 2.0 * c["n"] * c["hidden"] * (2 * c["hidden"] + (c["heads"] + 2 * c["kv"]) * HEAD)
        return dict(bytes=tot[0], flops=tot[1])
    add(1, c["ctx"] - 1)
    # random-init drafts are hardly ever accepted: a token a round
    add(1 + c["spec"], c["ctx"], times=c["tokens"])
    if c["spec"]:
        add(1, c["ctx"], times=c["tokens"] * c["spec"], layers=1)
    return dict(bytes=tot[0], flops=tot[1])


def tolerance(case):
    # measured against `exact` at the start, times about four: f32 sums over
    # 22-bit fixed-point operands (gemv, ffn, moe), and the same through the
    # layers of a model
    if case["kind"] == "gemv":
        return {"rel": 2e-6}
    if case["kind"] in ("ffn", "moe"):
        return {"rel": 6e-6}
    return {"rel": 2e-4, "max": 2e-3, "differ": 0.0}


# --------------------------------------------------------------------------
# the same in 64 bits
# --------------------------------------------------------------------------
def _silu(x):
    return x / (1 + torch.exp(-x))


def _moe64(x, logits, ex, top_k):
    p = torch.softmax(logits, 1)
    v, idx = torch.topk(p, top_k, dim=1)
    v = v / v.sum(1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(len(ex)):
        t, rank = torch.nonzero(idx == e, as_tuple=True)
        if len(t):
            g, u, d = (dequant(ex[e][n]) for n in ("gate", "up", "down"))
            y = (_silu(x[t] @ g.T) * (x[t] @ u.T)) @ d.T
            out.index_add_(0, t, y * v[t, rank][:, None])
    return out


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * torch.from_numpy(w).cuda().double()


def _rope(x, pos):
    # the model's angles are f32 products of the position and the frequency
    i = np.arange(HEAD // 2, dtype=np.float32)
    inv = np.float32(1) / np.power(np.float32(THETA), np.float32(2) * i / np.float32(HEAD), dtype=np.float32)
    ang = torch.from_numpy(pos.astype(np.float32)[:, None] * inv[None, :]).cuda().double()
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :HEAD // 2], x[..., HEAD // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


class _Exact:
    """The decoder's forward in f64 with its keys and values."""

    def __init__(self, c, sm):
        self.c, self.sm, self.kv = c, sm, [None] * c["layers"]
        self.big = c["layers"] > 8  # (the f64 weights of a deep model are made layer by layer)
        self.cache = {}

    def w(self, li, name):
        key = (li, name)
        if key not in self.cache:
            if self.big:
                self.cache.clear()
            self.cache[key] = dequant(self.sm["layers"][li][name])
        return self.cache[key]

    def rows(self, ids, pos0):
        c, lm = self.c, self.sm["lm_head"]
        at = np.asarray(ids)
        h = torch.from_numpy(lm["q"][at]).cuda().double() * torch.from_numpy(lm["row_scale"][at]).cuda().double()[:, None]
        n, pos = len(at), np.arange(pos0, pos0 + len(at))
        for li, l in enumerate(self.sm["layers"]):
            x = _rms(h, l["input_norm"])
            q, k, v = ((x @ self.w(li, m).T).view(n, -1, HEAD) for m in ("wq", "wk", "wv"))
            q, k = _rope(_rms(q, l["q_norm"]), pos), _rope(_rms(k, l["k_norm"]), pos)
            if self.kv[li] is not None and pos0:
                k, v = (torch.cat([o[:pos0], t]) for o, t in zip(self.kv[li], (k, v)))
            self.kv[li] = (k, v)
            mask = torch.arange(pos0 + n, device="cuda")[None, :] > torch.arange(pos0, pos0 + n, device="cuda")[:, None]
            a = torch.empty_like(q)
            for hd in range(c["heads"]):
                g = hd * c["kv"] // c["heads"]
                for r0 in range(0, n, 4096):
                    s = (q[r0:r0 + 4096, hd] @ k[:, g].T) / math.sqrt(HEAD)
                    s.masked_fill_(mask[r0:r0 + 4096], -math.inf)
                    a[r0:r0 + 4096, hd] = torch.softmax(s, 1) @ v[:, g]
            h = h + a.reshape(n, -1) @ self.w(li, "wo").T
            x = _rms(h, l["post_norm"])
            if "moe" in l:
                rt = l["moe"]["router"]
                rw = torch.from_numpy(rt["bytes"]).cuda().view(torch.float16).view(rt["rows"], rt["cols"]).double()
                h = h + _moe64(x, x @ rw.T, l["moe"]["experts"], l["moe"]["top_k"])
            else:
                h = h + (_silu(x @ self.w(li, "gate").T) * (x @ self.w(li, "up").T)) @ self.w(li, "down").T
        return h

    def logits(self, h):
        return _rms(h, self.sm["final_norm"]) @ dequant(self.sm["lm_head"]).T


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "gemv":
        t, x = _gemv_inputs(c, seed)
        return x.double() @ dequant(t).T
    if k == "ffn":
        (g, u, d), x = _ffn_inputs(c, seed)
        x = x.double()
        return ((_silu(x @ dequant(g).T) * (x @ dequant(u).T)) @ dequant(d).T).cpu().numpy()
    if k == "moe":
        ex, x, lg = _moe_inputs(c, seed)
        return _moe64(x.double(), lg.double(), ex, c["top_k"])
    sm, ids = weights(c, seed)
    m, n = _Exact(c, sm), len(ids)
    if k == "prefill":
        hid = m.rows(ids, 0)[-1]
        return dict(hidden=hid.cpu().numpy(), next=m.logits(m.rows(ids[:1], n)).cpu().numpy())
    hid = m.rows(ids, 0)[-1:]
    # (the tokens, and the tip they lead to, follow from greedy or seeded picks)
    return dict(hidden=hid.cpu().numpy(), logits=m.logits(hid).cpu().numpy(), tokens=None, tip=None)
