"""Timing cases: the work a program built on this package has it do.

Five kinds, each through the entry points such a program calls:

* ``proj``: one packed ternary projection (``PackedTernaryLinear``), with or
  without the input RMSNorm folded in; one token to a prefill chunk.
* ``moe``: one MoE block (``MapleSparseMoeBlock``) with its residual; one token
  to a prefill chunk, uniform or skewed routing.
* ``attn``: one layer's decode attention (``decode_attention``: QK-norm, RoPE,
  K/V write, GQA over the cache).
* ``head``: the 4-bit lm_head (``PackedRTN4Linear``) at a decode batch.
* ``step``: a whole decode step of a decoder (embedding, layers, head, greedy
  choice), as the decode-graph runner captures it.

Decode programs run their layers inside a captured graph, so decode-sized cases
(``graph: True``) are captured in ``prepare`` and ``run`` replays them; prefill
chunks and the single small call are ordinary eager calls.

Weights are random with the distributions of the repository's benchmark:
ternary codes uniform over {-1, 0, 1}, row scales in [0.01, 0.05] (bf16, or
float32 as a converted checkpoint keeps them), 4-bit codes uniform with
zero-centred groups, activations N(0, 1) in bf16.
"""

import math

import torch

import __graft_entry__

__graft_entry__.load_package()

from maple_amd import kernels, linear, moe  # noqa: E402
from maple_amd.decode_graph import Sampling, capture_decode_graph  # noqa: E402
from maple_amd.model import DecoderConfig, DecoderLayerWeights, KVCache, SyntheticDecoder, rope_tables  # noqa: E402
from maple_amd.synthetic import MoELayer  # noqa: E402

DEV = "cuda"
EPS = 1e-6
HIDDEN = 2048
TOP_K = 8
VOCAB = 151936
THETA = 10000.0
# (heads, kv_heads, head_dim), (experts, intermediate): the two decoders of the benchmark
HEADS = {"64": (32, 4, 64), "128": (16, 4, 128)}


def listed():
    return [
        # the smallest call: one token through one projection, outside a graph
        dict(name="proj_t1_call", kind="proj", tokens=1, rows=1536, k=2048, rms=False, alpha="bf16", graph=False),
        # prefill chunk through the QKV projection (input RMSNorm folded in)
        dict(name="proj_t2048_rms", kind="proj", tokens=2048, rows=2560, k=2048, rms=True, alpha="bf16", graph=False),
        # the ragged last chunk of a prompt through the output projection of a converted checkpoint
        dict(name="proj_t777", kind="proj", tokens=777, rows=2048, k=2048, rms=False, alpha="f32", graph=False),
        # batched decode, Zipf-like expert load
        dict(name="moe_t32_skew", kind="moe", tokens=32, experts=64, inter=768, skew=True, alpha="bf16", graph=True),
        # prefill chunk
        dict(name="moe_t2048", kind="moe", tokens=2048, experts=64, inter=768, skew=True, alpha="bf16", graph=False),
        # ragged prefill chunk at 256 small experts, float32 scales
        dict(name="moe_t509_e256", kind="moe", tokens=509, experts=256, inter=512, skew=False, alpha="f32", graph=False),
        # batched decode attention over a 4096-token context, rows at different lengths
        dict(name="attn_b32_l4096", kind="attn", batch=32, length=4096, heads="64", window=0, graph=True),
        # a few long-context rows
        dict(name="attn_b3_l32768", kind="attn", batch=3, length=32768, heads="128", window=0, graph=True),
        # head of a mid-sized decode batch in the converter's default groups of 64
        dict(name="head_b24_g64", kind="head", batch=24, vocab=VOCAB, group=64, graph=True),
        # head at the widest decode bucket
        dict(name="head_b256_g128", kind="head", batch=256, vocab=VOCAB, group=128, graph=True),
        # single-stream decode: 64 experts, 32/4 heads of 64, 4096-token context
        dict(name="step_b1_l4096", kind="step", batch=1, length=4096, layers=4, heads="64", experts=64, inter=768,
             group=128, mixed=False, alpha="bf16"),
        # batched decode at 256 experts, 16/4 heads of 128, three sliding layers to a full one, groups of 64
        dict(name="step_b32_e256", kind="step", batch=32, length=512, layers=4, heads="128", experts=256, inter=512,
             group=64, mixed=True, alpha="f32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["proj", "proj", "moe", "moe", "attn", "attn", "head", "head", "step"])
    if kind == "proj":
        tokens = _log_int(rng, 1, 2048)
        return dict(kind=kind, tokens=tokens, rows=8 * _log_int(rng, 128, 640), k=rng.choice([768, 1024, 2048, 3072, 4096]),
                    rms=rng.random() < 0.5, alpha=rng.choice(["bf16", "f32"]), graph=tokens <= 256)
    if kind == "moe":
        tokens = _log_int(rng, 1, 2048)
        experts, inter = rng.choice([(64, 768), (64, 768), (256, 512)])
        return dict(kind=kind, tokens=tokens, experts=experts, inter=inter, skew=rng.random() < 0.5,
                    alpha=rng.choice(["bf16", "f32"]), graph=tokens <= 256)
    if kind == "attn":
        length = _log_int(rng, 128, 32768)
        batch = min(_log_int(rng, 1, 64), max(1, 131072 // length))
        return dict(kind=kind, batch=batch, length=length, heads=rng.choice(["64", "128"]),
                    window=rng.choice([0, 0, 512]), graph=True)
    if kind == "head":
        return dict(kind=kind, batch=_log_int(rng, 1, 256), vocab=rng.choice([VOCAB, VOCAB, 100003, 32000]),
                    group=rng.choice([64, 128]), graph=True)
    heads, experts, inter, group, mixed = rng.choice([("64", 64, 768, 128, False), ("128", 256, 512, 64, True)])
    return dict(kind=kind, batch=_log_int(rng, 1, 32), length=_log_int(rng, 64, 4096), layers=4, heads=heads,
                experts=experts, inter=inter, group=group, mixed=mixed, alpha=rng.choice(["bf16", "f32"]))


# ---------------------------------------------------------------------------
# Inputs, from the seed alone (plain torch; exact() makes the same ones).
# ---------------------------------------------------------------------------
class _Make:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(1_000_003 * int(seed) + 17)

    def normal(self, *shape, std=1.0):
        return (torch.randn(shape, generator=self.g, device=DEV) * std).to(torch.bfloat16)

    def uniform(self, shape, lo, hi, dtype):
        return (torch.rand(shape, generator=self.g, device=DEV) * (hi - lo) + lo).to(dtype)

    def ternary(self, *shape):
        """uint32 [..., K/16] of uniform ternary codes {0, 1, 2}, 16 per word, LSB first."""
        *lead, k = shape
        rows = math.prod(lead)
        out = torch.empty(rows, k // 4, dtype=torch.uint8, device=DEV)
        for r in range(0, rows, 1 << 17):
            n = min(rows - r, 1 << 17)
            c = torch.randint(0, 3, (n, k // 4, 4), generator=self.g, device=DEV, dtype=torch.uint8)
            out[r:r + n] = c[..., 0] | (c[..., 1] << 2) | (c[..., 2] << 4) | (c[..., 3] << 6)
        return out.view(torch.int32).view(torch.uint32).reshape(*lead, k // 16)

    def alpha(self, kind, *shape):
        return self.uniform(shape, 0.01, 0.05, torch.bfloat16 if kind == "bf16" else torch.float32)

    def rtn4(self, rows, k, group, lo=0.003, hi=0.006):
        words = torch.randint(-2 ** 31, 2 ** 31, (rows, k // 8), generator=self.g, device=DEV, dtype=torch.int64)
        sc = self.uniform((rows, k // group), lo, hi, torch.bfloat16)
        return words.to(torch.int32).view(torch.uint32), sc, (-7.5 * sc.float()).to(torch.bfloat16)

    def moe(self, c):
        e, i = c["experts"], c["inter"]
        bias = None
        if c.get("skew"):  # log of Zipf(1.1) shares over a random order of the experts
            p = torch.arange(1, e + 1, device=DEV, dtype=torch.float64) ** -1.1
            bias = torch.log(p / p.sum())[torch.randperm(e, generator=self.g, device=DEV)].float()
        return dict(gate=self.normal(e, HIDDEN, std=0.02), up=self.ternary(e, 2 * i, HIDDEN),
                    up_a=self.alpha(c["alpha"], e, 2 * i), down=self.ternary(e, HIDDEN, i),
                    down_a=self.alpha(c["alpha"], e, HIDDEN), bias=bias)

    def lengths(self, batch, length):
        """Positions already in the cache per row: the longest row has ``length``."""
        if batch == 1:
            return torch.full((1,), length, device=DEV, dtype=torch.int64)
        n = torch.randint(length // 2, length + 1, (batch,), generator=self.g, device=DEV)
        n[0] = length
        return n


def _inputs(case, seed):
    m, c = _Make(seed), case
    if c["kind"] == "proj":
        return dict(w=m.ternary(c["rows"], c["k"]), a=m.alpha(c["alpha"], c["rows"]), x=m.normal(c["tokens"], c["k"]),
                    rms=m.uniform((c["k"],), 0.5, 1.5, torch.float32) if c["rms"] else None)
    if c["kind"] == "moe":
        return dict(layer=m.moe(c), x=m.normal(c["tokens"], HIDDEN), res=m.normal(c["tokens"], HIDDEN))
    if c["kind"] == "attn":
        nq, nkv, d = HEADS[c["heads"]]
        shape = (c["batch"], nkv, _max_len(c["length"]), d)
        return dict(qkv=m.normal(c["batch"], (nq + 2 * nkv) * d), qn=m.uniform((d,), 0.5, 1.5, torch.float32),
                    kn=m.uniform((d,), 0.5, 1.5, torch.float32), k=m.normal(*shape), v=m.normal(*shape),
                    seqlen=m.lengths(c["batch"], c["length"]))
    if c["kind"] == "head":
        return dict(table=m.rtn4(c["vocab"], HIDDEN, c["group"]), x=m.normal(c["batch"], HIDDEN))
    nq, nkv, d = HEADS[c["heads"]]
    layers = []
    for _ in range(c["layers"]):
        layers.append(dict(qkv=m.ternary((nq + 2 * nkv) * d, HIDDEN), qkv_a=m.alpha(c["alpha"], (nq + 2 * nkv) * d),
                           o=m.ternary(HIDDEN, nq * d), o_a=m.alpha(c["alpha"], HIDDEN),
                           ln=torch.ones(HIDDEN, device=DEV), hn=torch.ones(d, device=DEV), moe=m.moe(c)))
    shape = (c["batch"], nkv, _max_len(c["length"]), d)
    # embeddings larger than one layer's update, as a trained residual stream is: a random router's choice then
    # changes a row little where two correct results take the other of two nearly tied experts
    return dict(layers=layers, embed=m.rtn4(VOCAB, HIDDEN, c["group"], 0.6, 1.2), head=m.rtn4(VOCAB, HIDDEN, c["group"]),
                k=[m.normal(*shape) for _ in layers], v=[m.normal(*shape) for _ in layers],
                seqlen=m.lengths(c["batch"], c["length"]),
                ids=torch.randint(0, VOCAB, (c["batch"],), generator=m.g, device=DEV))


def _max_len(length):
    return length + 128


def _layer_kinds(case):
    return tuple(("sliding_attention", "sliding_attention", "sliding_attention", "full_attention")[i % 4]
                 for i in range(case["layers"])) if case["mixed"] else ()


# ---------------------------------------------------------------------------
# The program's own objects, and one pass.
# ---------------------------------------------------------------------------
def _moe_block(w, inter):
    return moe.MapleSparseMoeBlock(w["gate"], linear.PackedTernaryExperts(w["up"], w["up_a"]),
                                   linear.PackedTernaryExperts(w["down"], w["down_a"]), TOP_K, inter, w["bias"])


def _captured(call):
    """``call`` in a graph, after a warm-up on the capture's stream."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(2):
            call()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            out = call()
    torch.cuda.current_stream().wait_stream(stream)

    def replay():
        graph.replay()
        return out

    return replay


def prepare(case, seed):
    c, t = case, _inputs(case, seed)
    if c["kind"] == "step":
        return _prepare_step(c, t)
    if c["kind"] == "proj":
        layer = linear.PackedTernaryLinear(t["w"], t["a"])

        def call():
            return layer(t["x"], rms_weight=t["rms"], rms_eps=EPS)
    elif c["kind"] == "moe":
        block = _moe_block(t["layer"], c["inter"])

        def call():
            return block(t["x"], residual=t["res"])
    elif c["kind"] == "attn":
        nq, nkv, d = HEADS[c["heads"]]
        cos, sin = rope_tables(_max_len(c["length"]), d // 2, THETA, torch.device(DEV))
        ws = kernels.gqa_workspace(c["batch"], nkv, _max_len(c["length"]), torch.device(DEV), d)

        def call():
            out = kernels.decode_attention(
                t["qkv"], t["qn"], t["kn"], cos, sin, t["k"], t["v"], t["seqlen"], ws, num_heads=nq, num_kv_heads=nkv,
                head_dim=d, rotary_dim=d // 2, eps=EPS, scale=d ** -0.5, window=c["window"] or None)
            return out, t["k"], t["v"]
    else:
        head = linear.PackedRTN4Linear(*t["table"], group_size=c["group"])

        def call():
            return head(t["x"])

    return {"call": _captured(call) if c["graph"] else call, "keep": t}


def _prepare_step(c, t):
    dev = torch.device(DEV)
    nq, nkv, d = HEADS[c["heads"]]
    cfg = DecoderConfig(hidden=HIDDEN, layers=c["layers"], heads=nq, kv_heads=nkv, head_dim=d, experts=c["experts"],
                        inter=c["inter"], top_k=TOP_K, vocab=VOCAB, rtn_group=c["group"], rope_theta=THETA, eps=EPS,
                        layer_types=_layer_kinds(c), sliding_window=512, nope_on_global=c["mixed"])
    layers = [DecoderLayerWeights(w["qkv"], w["qkv_a"], w["o"], w["o_a"], w["ln"], w["ln"], w["hn"], w["hn"],
                                  MoELayer(w["moe"]["gate"], w["moe"]["up"], w["moe"]["up_a"], w["moe"]["down"],
                                           w["moe"]["down_a"])) for w in t["layers"]]
    model = SyntheticDecoder.from_weights(cfg, dev, layers, t["embed"], t["head"], torch.ones(HIDDEN, device=DEV),
                                          max_len=_max_len(c["length"]))
    ws = kernels.gqa_workspace(c["batch"], nkv, _max_len(c["length"]), dev, d)
    cache = KVCache(t["k"], t["v"], t["seqlen"].clone(), _max_len(c["length"]), ws)
    snap = cache.snapshot(steps=4)
    sampling = Sampling()
    graph = capture_decode_graph(model, cache, t["ids"].clone(), sampling, feed=False)
    cache.restore(snap)

    def call():
        cache.seqlen.copy_(t["seqlen"])  # the same position again: a program that regenerates from a snapshot
        graph.step(sampling)
        return graph.logits

    return {"call": call, "keep": (model, cache, t)}


def run(state):
    return state["call"]()


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how far two correct results may differ.
# ---------------------------------------------------------------------------
def _moe_work(tokens, experts, inter):
    hit = experts * (1.0 - (1.0 - TOP_K / experts) ** tokens)
    expert = 3 * inter * HIDDEN // 4 + (2 * inter + HIDDEN) * 2
    return hit * expert + experts * HIDDEN * 2, tokens * (6 * TOP_K * inter * HIDDEN + 2 * experts * HIDDEN)


def _attn_work(batch, length, heads, window):
    nq, nkv, d = HEADS[heads]
    mean = length if batch == 1 else (length + (batch - 1) * 0.75 * length) / batch
    span = min(mean, window) if window else mean
    return batch * (span * 2 * nkv * d * 2 + (2 * nq + 4 * nkv) * d * 2), batch * span * 4 * nq * d


def work(case):
    c = case
    if c["kind"] == "proj":
        a = 2 if c["alpha"] == "bf16" else 4
        return {"bytes": c["rows"] * (c["k"] // 4 + a) + c["tokens"] * (c["k"] + c["rows"]) * 2,
                "flops": 2 * c["tokens"] * c["rows"] * c["k"]}
    if c["kind"] == "moe":
        b, f = _moe_work(c["tokens"], c["experts"], c["inter"])
        return {"bytes": b + 3 * c["tokens"] * HIDDEN * 2, "flops": f}
    if c["kind"] == "attn":
        b, f = _attn_work(c["batch"], c["length"], c["heads"], c["window"])
        return {"bytes": b, "flops": f}
    table = lambda v: v * (HIDDEN // 2 + 4 * HIDDEN // c["group"])  # noqa: E731
    if c["kind"] == "head":
        return {"bytes": table(c["vocab"]) + c["batch"] * (HIDDEN + c["vocab"]) * 2,
                "flops": 2 * c["batch"] * c["vocab"] * HIDDEN}
    nq, nkv, d = HEADS[c["heads"]]
    b, f = table(VOCAB) + c["batch"] * VOCAB * 2, 2 * c["batch"] * VOCAB * HIDDEN
    kinds = _layer_kinds(c) or ("full_attention",) * c["layers"]
    for kind in kinds:
        mb, mf = _moe_work(c["batch"], c["experts"], c["inter"])
        ab, af = _attn_work(c["batch"], c["length"], c["heads"], 512 if kind == "sliding_attention" else 0)
        rows = (2 * nq + 2 * nkv) * d
        b, f = b + mb + ab + rows * HIDDEN // 4, f + mf + af + 2 * c["batch"] * rows * HIDDEN
    return {"bytes": b, "flops": f}


def tolerance(case):
    # four times what was measured against exact(): one bf16 rounding of the output (1.7e-3), with the bf16 inner values
    # of the MoE block (1.8e-3), with bf16 probabilities (2.8e-3); a step also carries the choice between nearly tied
    # experts (4e-3 to 9e-3, one row alone up to 2.8e-2)
    return {"proj": {"rel": 7e-3}, "head": {"rel": 7e-3}, "attn": {"rel": 1.1e-2}, "moe": {"rel": 8e-3},
            "step": {"rel": 5e-2}}[case["kind"]]


# ---------------------------------------------------------------------------
# The same values in 64 bits, without the package.
# ---------------------------------------------------------------------------
def _codes(words, bits):
    w = words.view(torch.int32)
    shifts = torch.arange(0, 32, bits, device=DEV, dtype=torch.int32)
    return ((w.unsqueeze(-1) >> shifts) & ((1 << bits) - 1)).flatten(-2)


def _ternary(words, alpha):
    return (_codes(words, 2) - 1).double() * alpha.double().unsqueeze(-1)


def _rms(x, weight):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _affine(table, rows, group):
    w, s, b = (t.view(torch.int32)[rows].view(torch.uint32) if t.dtype == torch.uint32 else t[rows] for t in table)
    q = _codes(w, 4).double()
    return (q.unflatten(-1, (-1, group)) * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).flatten(-2)


def _head(x, table, group):
    v = table[0].shape[0]
    return torch.cat([x.double() @ _affine(table, slice(r, min(v, r + 16384)), group).t() for r in range(0, v, 16384)], -1)


def _moe(x, w, inter, res):
    logits = x.double() @ w["gate"].double().t()
    if w["bias"] is not None:
        logits = logits + w["bias"].double()
    top, ids = torch.topk(torch.softmax(logits, -1), TOP_K, dim=-1)
    wt = top / (top.sum(-1, keepdim=True) + 1e-20)
    y = res.double().clone()
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        both = x[t].double() @ _ternary(w["up"][e], w["up_a"][e]).t()
        up, gate = both[:, :inter].clamp(-7.0, 7.0), both[:, inter:].clamp(max=7.0)
        h = up * gate * torch.sigmoid(gate)
        y.index_add_(0, t, (h @ _ternary(w["down"][e], w["down_a"][e]).t()) * wt[t, j].unsqueeze(-1))
    return y


def _rope(x, pos, rot):
    """Rotate-half over the first ``rot`` dims of ``x [B, heads, D]`` at ``pos [B]``, tables rounded to bf16."""
    cos, sin = rope_tables_plain(pos, rot)
    lo, hi = x[..., :rot // 2], x[..., rot // 2:rot]
    return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin, x[..., rot:]], -1)


def rope_tables_plain(pos, rot):
    inv = 1.0 / (THETA ** (torch.arange(0, rot, 2, device=DEV, dtype=torch.float32) / rot))
    f = (pos.float().unsqueeze(-1) * inv).unsqueeze(1)
    return f.cos().to(torch.bfloat16).double(), f.sin().to(torch.bfloat16).double()


def _attend(qkv, heads, qn, kn, k, v, seqlen, window, rope):
    """Attention of ``qkv [B, ...]`` over one layer's cache; returns it with the new K and V rows."""
    nq, nkv, d = HEADS[heads]
    b = qkv.shape[0]
    x = qkv.double().view(b, nq + 2 * nkv, d)
    q, nk, nv = _rms(x[:, :nq], qn), _rms(x[:, nq:nq + nkv], kn), x[:, nq + nkv:]
    if rope:
        q, nk = _rope(q, seqlen, d // 2), _rope(nk, seqlen, d // 2)
    out = torch.empty(b, nq, d, dtype=torch.float64, device=DEV)
    for i in range(b):
        n = int(seqlen[i])
        lo = max(0, n + 1 - window) if window else 0
        ki = torch.cat([k[i, :, lo:n].double(), nk[i].unsqueeze(1)], 1).repeat_interleave(nq // nkv, 0)
        vi = torch.cat([v[i, :, lo:n].double(), nv[i].unsqueeze(1)], 1).repeat_interleave(nq // nkv, 0)
        p = torch.softmax((ki @ q[i].unsqueeze(-1)).squeeze(-1) * d ** -0.5, -1)
        out[i] = (p.unsqueeze(1) @ vi).squeeze(1)
    return out, nk, nv


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    if c["kind"] == "proj":
        x = t["x"].double() if t["rms"] is None else _rms(t["x"], t["rms"])
        return x @ _ternary(t["w"], t["a"]).t()
    if c["kind"] == "moe":
        return _moe(t["x"], t["layer"], c["inter"], t["res"])
    if c["kind"] == "head":
        return _head(t["x"], t["table"], c["group"])
    if c["kind"] == "attn":
        out, nk, nv = _attend(t["qkv"], c["heads"], t["qn"], t["kn"], t["k"], t["v"], t["seqlen"], c["window"], True)
        k, v, rows = t["k"].double(), t["v"].double(), torch.arange(c["batch"], device=DEV)
        k[rows, :, t["seqlen"]], v[rows, :, t["seqlen"]] = nk, nv
        return out.unsqueeze(2), k, v
    h = _affine(t["embed"], t["ids"], c["group"])
    kinds = _layer_kinds(c) or ("full_attention",) * c["layers"]
    for i, w in enumerate(t["layers"]):
        full = kinds[i] == "full_attention"
        qkv = _rms(h, w["ln"]) @ _ternary(w["qkv"], w["qkv_a"]).t()
        a, _, _ = _attend(qkv, c["heads"], w["hn"], w["hn"], t["k"][i], t["v"][i], t["seqlen"], 0 if full else 512,
                          not (c["mixed"] and full))
        h = h + a.flatten(1) @ _ternary(w["o"], w["o_a"]).t()
        h = _moe(_rms(h, w["ln"]), w["moe"], c["inter"], h)
    return _head(_rms(h, torch.ones(HIDDEN, device=DEV)), t["head"], c["group"])
