"""The work that programs built on this package have it do, as cases whose time and results can be compared between
two builds of it.

A case is a dict of plain values; its "kind" says which entry point runs:

  linear       DecodeLinears.linear: one linear of a decode step, called by itself
  int8_linear  Int8Linear on bf16 activations (W8A8 with scales per token or per 64-channel group, or W8A16)
  lm_ffn       the feed-forward of one layer of a prompt pass: add_rmsnorm_q, w1|w3, silu_mul_q, w2 (W8A8)
  vision_ffn   the MLP of one vision-encoder layer: add_layernorm_q, fc1 + bias + GELU written as INT8, fc2 + bias
  decode       StaticDecoder: several tokens of a given continuation, one replayed graph per token
  prompt       StaticDecoder.prefill: a whole prompt in one pass

Sizes are the LFM2-1.2B language model's (hidden 2048, FFN 8192, 32 query and 8 KV heads of 64, vocabulary 65536)
and the vision encoder's (width 1152, FFN 4304). The StaticDecoder cases run all 16 layers or only the first 3 or 6:
these hold both layer types and are shallow enough for the logits of two correct builds to stay close.
"""

import math
import os
import pathlib
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, str(pathlib.Path.cwd() / "lfm2.5-vl-optimization_amd"))

from lfm2opt.decode import DecodeLinears, linear_path  # noqa: E402
from lfm2opt.int8 import Int8Linear, qbuf  # noqa: E402
from lfm2opt.kernels import int8_ext  # noqa: E402
from lfm2opt.runtime import StaticDecoder  # noqa: E402

DEV = "cuda"
BF16 = torch.bfloat16
H, FFN, HEADS, KV_HEADS, HEAD_DIM, VOCAB, CONV_LEN = 2048, 8192, 32, 8, 64, 65536, 3
LAYERS = "CCACCACCACACACAC"  # C: gated short convolution, A: attention
EPS = 1e-5
THETA = 1e6
V_DIM, V_FFN, V_PAD, V_EPS = 1152, 4304, 48, 1e-6  # the vision FFN is padded to a multiple of 64 for INT8 outputs
GROUP = 64
W4_GROUP = 128
# the decode linears of a layer and the head: [output rows, input channels]
LINEARS = {"qkv": ((HEADS + 2 * KV_HEADS) * HEAD_DIM, H), "o": (H, H), "in": (3 * H, H), "out": (H, H),
           "w13": (2 * FFN, H), "w2": (H, FFN), "head": (VOCAB, H)}


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # One small projection of a decode step called on its own: latency, launches and the host's share of a call.
        dict(name="linear_qkv_b1", kind="linear", layer="qkv", fmt="int8", batch=1),
        # The INT4 up-projection of a decode step at a small serving batch.
        dict(name="linear_w13_int4_b8", kind="linear", layer="w13", fmt="int4", batch=8),
        # The down-projection at a batch past the GEMV's: INT8 weights, bf16 activations.
        dict(name="linear_w2_b45", kind="linear", layer="w2", fmt="int8", batch=45),
        # An attention projection of a short prompt with an odd token count, activation scales per token.
        dict(name="int8_qkv_m333", kind="int8_linear", rows=333, cols=3072, inputs=2048, mode="token", bias=False,
             gelu=False),
        # A sensitive layer kept at bf16 activations over a prompt.
        dict(name="w8a16_m1500", kind="int8_linear", rows=1500, cols=2048, inputs=2048, mode="a16", bias=True,
             gelu=False),
        # The feed-forward of a layer over a long prompt: the largest matrix products of the language model.
        dict(name="lm_ffn_m4096", kind="lm_ffn", rows=4096, group=GROUP),
        # The MLP of a vision-encoder layer over a batch of image tiles (10 x 1024 patches).
        dict(name="vision_ffn_m10240", kind="vision_ffn", rows=10240),
        # A reply token by token at batch 1 on INT8 weights: the whole model, the usual interactive request.
        dict(name="decode_b1", kind="decode", layers=16, fmt="int8", batch=1, prompt=200, steps=16),
        # The same on INT4 weights behind a long conversation.
        dict(name="decode_int4_long", kind="decode", layers=3, fmt="int4", batch=1, prompt=3001, steps=8),
        # A batch of requests served together.
        dict(name="decode_b16", kind="decode", layers=3, fmt="int8", batch=16, prompt=300, steps=8),
        # An ordinary prompt in one pass on W8A8: many short kernels.
        dict(name="prompt_461", kind="prompt", layers=6, mode="int8", batch=1, tokens=461),
        # A long one, where the attention is part of the work.
        dict(name="prompt_2048", kind="prompt", layers=3, mode="int8", batch=1, tokens=2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "int8_linear", "int8_linear", "lm_ffn", "vision_ffn", "decode", "decode",
                       "prompt", "prompt"])
    if kind == "linear":
        return dict(kind=kind, layer=rng.choice(list(LINEARS)), fmt=rng.choice(["int8", "int8", "int4", "bf16"]),
                    batch=_log(rng, 1, 256))
    if kind == "int8_linear":
        mode = rng.choice(["token", "group", "a16"])
        cols, inputs = rng.choice([(3072, 2048), (6144, 2048), (2048, 2048), (3456, 1152), (1152, 1152)])
        return dict(kind=kind, rows=_log(rng, 1, 4096), cols=cols, inputs=inputs, mode=mode, bias=inputs == 1152,
                    gelu=inputs == 1152 and rng.random() < 0.3)
    if kind == "lm_ffn":
        return dict(kind=kind, rows=_log(rng, 8, 4096), group=GROUP)
    if kind == "vision_ffn":
        return dict(kind=kind, rows=_log(rng, 64, 10240))
    if kind == "decode":
        batch = _log(rng, 1, 64)
        return dict(kind=kind, layers=3, fmt=rng.choice(["int8", "int8", "int4", "bf16"]), batch=batch,
                    prompt=_log(rng, 16, max(32, min(4000, 16000 // batch))), steps=rng.randint(2, 12))
    batch = rng.choice([1, 1, 1, 2, 4])
    return dict(kind=kind, layers=3, mode=rng.choice(["int8", "int8", "bf16"]), batch=batch,
                tokens=_log(rng, 16, 2048 // batch))


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, std=1.0):
    return (torch.randn(*shape, device=DEV, generator=g) * std).to(BF16)


def _weight(g, rows, cols):
    return _normal(g, rows, cols, std=cols ** -0.5)


def _activations(g, rows, cols):
    """Unit-variance activations with a few outlier channels, as between the layers of a language model."""
    scale = torch.ones(cols, device=DEV)
    scale[torch.randperm(cols, device=DEV, generator=g)[:max(1, cols // 256)]] = 8.0
    return (torch.randn(rows, cols, device=DEV, generator=g) * scale).to(BF16)


class _Node(torch.nn.Module):
    """A module holding the children and weights it is given."""

    def __init__(self, weight=None, **children):
        super().__init__()
        self.bias = None
        if weight is not None:
            self.weight = torch.nn.Parameter(weight, requires_grad=False)
        for name, child in children.items():
            setattr(self, name, child)


def _model(g, n_layers):
    """A language model with the module and weight names StaticDecoder reads, random bf16 weights, tied head. The
    linears that write to the residual stream start at 1 / sqrt(2 layers) of the others' scale, as such models are
    initialised, so that the stream keeps its scale and no layer drowns the ones before it."""
    def lin(rows, cols, std=1.0):
        return _Node(_normal(g, rows, cols, std=std * cols ** -0.5))

    out = (2 * len(LAYERS)) ** -0.5

    def norm(n):
        return _Node((1.0 + 0.1 * torch.randn(n, device=DEV, generator=g)).to(BF16))

    layers = []
    for kind in LAYERS[:n_layers]:
        kv = KV_HEADS * HEAD_DIM
        if kind == "A":
            mixer = dict(self_attn=_Node(q_proj=lin(H, H), k_proj=lin(kv, H), v_proj=lin(kv, H),
                                         out_proj=lin(H, H, out), q_layernorm=norm(HEAD_DIM),
                                         k_layernorm=norm(HEAD_DIM)))
        else:
            mixer = dict(conv=_Node(in_proj=lin(3 * H, H), out_proj=lin(H, H, out),
                                    conv=_Node(_normal(g, H, 1, CONV_LEN, std=0.5))))
        layers.append(_Node(operator_norm=norm(H), ffn_norm=norm(H),
                            feed_forward=_Node(w1=lin(FFN, H), w3=lin(FFN, H), w2=lin(H, FFN, out)), **mixer))
    rotary = _Node()
    rotary.inv_freq = THETA ** (-torch.arange(0, HEAD_DIM, 2, device=DEV, dtype=torch.float32) / HEAD_DIM)
    rotary.attention_scaling = 1.0
    embed = _Node(_normal(g, VOCAB, H))
    lm = _Node(layers=torch.nn.ModuleList(layers), rotary_emb=rotary, embed_tokens=embed, embedding_norm=norm(H))
    lm.config = _Config(n_layers)
    net = _Node(model=lm, lm_head=_Node())
    net.lm_head.weight = embed.weight
    return net


class _Config:
    def __init__(self, n_layers):
        self.num_hidden_layers = n_layers
        self.layer_types = ["full_attention" if c == "A" else "conv" for c in LAYERS[:n_layers]]
        self.num_attention_heads, self.num_key_value_heads, self.head_dim = HEADS, KV_HEADS, HEAD_DIM
        self.hidden_size, self.vocab_size, self.conv_L_cache, self.norm_eps = H, VOCAB, CONV_LEN, EPS


class _Group:
    """LFM2_INT8_GROUP for the layers built inside (read when an Int8Linear is built)."""

    def __init__(self, group):
        self.group = group

    def __enter__(self):
        self.saved = os.environ.get("LFM2_INT8_GROUP")
        os.environ["LFM2_INT8_GROUP"] = str(self.group)

    def __exit__(self, *exc):
        if self.saved is None:
            del os.environ["LFM2_INT8_GROUP"]
        else:
            os.environ["LFM2_INT8_GROUP"] = self.saved


def _inputs(case, seed):
    """The tensors a case starts from: weights, activations, tokens."""
    g, kind = _gen(seed), case["kind"]
    if kind == "linear":
        rows, cols = LINEARS[case["layer"]]
        return dict(w=_weight(g, rows, cols), x=_activations(g, case["batch"], cols))
    if kind == "int8_linear":
        return dict(w=_weight(g, case["cols"], case["inputs"]),
                    b=_normal(g, case["cols"], std=0.5) if case["bias"] else None,
                    x=_activations(g, case["rows"], case["inputs"]))
    if kind == "lm_ffn":
        return dict(h=_activations(g, case["rows"], H), y=_normal(g, case["rows"], H),
                    norm=(1.0 + 0.1 * torch.randn(H, device=DEV, generator=g)).to(BF16),
                    w13=_weight(g, 2 * FFN, H), w2=_weight(g, H, FFN))
    if kind == "vision_ffn":
        return dict(h=_activations(g, case["rows"], V_DIM), y=_normal(g, case["rows"], V_DIM),
                    norm=(1.0 + 0.1 * torch.randn(V_DIM, device=DEV, generator=g)).to(BF16),
                    shift=_normal(g, V_DIM, std=0.1), w1=_weight(g, V_FFN, V_DIM), b1=_normal(g, V_FFN, std=0.1),
                    w2=_weight(g, V_DIM, V_FFN), b2=_normal(g, V_DIM, std=0.1))
    net = _model(g, case["layers"])
    n = case["prompt"] + case["steps"] if kind == "decode" else case["tokens"]
    return dict(net=net, ids=torch.randint(3, VOCAB, (case["batch"], n), device=DEV, generator=g))


# ------------------------------------------------------------------------------------------------ what is timed
def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    s["kind"] = kind
    if kind == "linear":
        key = (case["layer"], 0)
        s.update(key=key, lin=DecodeLinears({key: s.pop("w")}, gemv=case["fmt"]))
    elif kind == "int8_linear":
        with _Group(GROUP if case["mode"] == "group" else 0):
            s["layer"] = Int8Linear(s.pop("w"), s["b"], a8=case["mode"] != "a16")
        s["gelu"] = case["gelu"]
    elif kind == "lm_ffn":
        with _Group(case["group"]):
            s["w13"], s["w2"] = Int8Linear(s["w13"]), Int8Linear(s["w2"])
        s["res"] = torch.empty_like(s["h"])
    elif kind == "vision_ffn":
        with _Group(GROUP):
            s["fc1"] = Int8Linear(s.pop("w1"), s.pop("b1"), pad_n=V_PAD)
            s["fc2"] = Int8Linear(s.pop("w2"), s.pop("b2"), pad_k=V_PAD)
        s["res"] = torch.empty_like(s["h"])
    elif kind == "decode":
        P, n = case["prompt"], case["steps"]
        dec = StaticDecoder(s["net"], keep_logits=True, gemv=case["fmt"], fused_prefill=True)
        _, st = dec.prefill(s["ids"][:, :P], n + 1)  # the prompt's own next token, then n steps
        s.update(dec=dec, st=st, start=st.ctr.clone(), rings={i: c.clone() for i, c in st.conv.items()},
                 forced=s["ids"][:, P:].t().contiguous(),
                 logits=torch.empty(n, case["batch"], VOCAB, device=DEV, dtype=torch.float32))
    else:
        w8 = case["mode"] == "int8"
        with _Group(GROUP):
            dec = StaticDecoder(s["net"], keep_logits=True, gemv="int8" if w8 else "cublas", prefill_int8=w8,
                                fused_prefill=not w8)
        dec.state(case["batch"], case["tokens"] + 1, 1, graph=False)
        s.update(dec=dec)
    return s


def run(s):
    kind = s["kind"]
    if kind == "linear":
        return s["lin"].linear(s["x"], s["key"])
    if kind == "int8_linear":
        return s["layer"](s["x"], gelu=s["gelu"])
    if kind == "lm_ffn":
        K8, h = int8_ext(), s["res"].copy_(s["h"])
        rows = h.shape[0]
        xq = qbuf(rows, H, s["w13"].group, h.device)
        K8.add_rmsnorm_q(h, s["y"], s["norm"], *xq, EPS)
        g = s["w13"](xq)
        aq = qbuf(rows, FFN, s["w2"].group, h.device)
        K8.silu_mul_q(g, *aq)
        return h, s["w2"](aq)
    if kind == "vision_ffn":
        K8, h = int8_ext(), s["res"].copy_(s["h"])
        xq = qbuf(h.shape[0], V_DIM, s["fc1"].group, h.device)
        K8.add_layernorm_q(h, s["y"], s["norm"], s["shift"], *xq, V_EPS)
        return h, s["fc2"](s["fc1"](xq, gelu=True, quant_out=True))
    if kind == "decode":  # the prompt's state again, then the given tokens, one graph replay each
        st = s["st"]
        st.ctr.copy_(s["start"])
        for i, ring in s["rings"].items():
            st.conv[i].copy_(ring)
        for t, tok in enumerate(s["forced"]):
            st.tok.copy_(tok)
            st.graph.replay()
            s["logits"][t].copy_(st.logits)
        return s["logits"], list(st.k.values()), list(st.v.values()), list(st.conv.values())
    dec = s["dec"]
    _, st = dec.prefill(s["ids"], 1, graph=False)
    return dec.last_prefill_logits, list(st.k.values()), list(st.v.values()), list(st.conv.values())


# ------------------------------------------------------------------------------------------------ what it must cost
_WBYTES = {"int8": 1.0, "int4": 0.5 + 4.0 / W4_GROUP, "bf16": 2.0}


def _attention_layers(case):
    return LAYERS[:case["layers"]].count("A")


def _layer_params(case, head=True):
    n = 0
    for c in LAYERS[:case["layers"]]:
        for name in (("qkv", "o") if c == "A" else ("in", "out")) + ("w13", "w2"):
            n += LINEARS[name][0] * LINEARS[name][1]
    return n + (VOCAB * H if head else 0)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        N, K = LINEARS[case["layer"]]
        B = case["batch"]
        return dict(bytes=N * K * _WBYTES[case["fmt"]] + 2.0 * B * (N + K), flops=2.0 * B * N * K)
    if kind == "int8_linear":
        M, N, K = case["rows"], case["cols"], case["inputs"]
        return dict(bytes=N * K + 2.0 * M * (N + K), flops=2.0 * M * N * K)
    if kind == "lm_ffn":
        M = case["rows"]
        return dict(bytes=3.0 * H * FFN + 2.0 * M * H * 4, flops=2.0 * M * 3 * H * FFN)
    if kind == "vision_ffn":
        M = case["rows"]
        return dict(bytes=2.0 * V_DIM * V_FFN + 2.0 * M * V_DIM * 4, flops=2.0 * M * 2 * V_DIM * V_FFN)
    B = case["batch"]
    if kind == "decode":
        n, ctx, att = case["steps"], case["prompt"] + (case["steps"] + 1) / 2, _attention_layers(case)
        par = _layer_params(case)
        cache = att * B * ctx * 2 * KV_HEADS * HEAD_DIM * 2.0
        return dict(bytes=n * (par * _WBYTES[case["fmt"]] + cache + 4.0 * B * VOCAB),
                    flops=n * B * (2.0 * par + att * 4.0 * HEADS * HEAD_DIM * ctx))
    T, par = case["tokens"], _layer_params(case, head=False)
    att = _attention_layers(case) * B * 4.0 * HEADS * HEAD_DIM * T * (T + 1) / 2
    return dict(bytes=(par + VOCAB * H) * (1.0 if case["mode"] == "int8" else 2.0) + 2.0 * B * T * H,
                flops=2.0 * B * T * par + 2.0 * B * VOCAB * H + att)


# ------------------------------------------------------------------------------------------------ what it must give
def tolerance(case):
    """About four times what the same path gives with its attention in 32 bits, or its sums in another order. What
    differs first is the bf16 rounding of a layer's output (2^-9 of a value, 1e-3 of a tensor); each layer that reads
    it passes it on, and a W8A8 layer that rounds another way at a quantization step adds up to half such a step."""
    kind = case["kind"]
    if kind in ("linear", "int8_linear"):
        return dict(rel=5e-3)
    if kind in ("lm_ffn", "vision_ffn"):
        return dict(rel=1e-2)
    return dict(rel=1.5e-2 if case["layers"] <= 3 else 3e-2)


def _dq8(w):
    """The INT8 weights of w, one scale per output row (the package's format), in 64 bits."""
    wf = w.float()
    s = (wf.abs().amax(1) / 127).clamp_min(1e-12)
    return torch.round(wf / s[:, None]).clamp(-127, 127).double() * s.double()[:, None]


def _dq4(w):
    """Symmetric INT4 in groups of W4_GROUP inputs."""
    wg = w.float().view(w.shape[0], -1, W4_GROUP)
    s = wg.abs().amax(-1).clamp_min(1e-12) / 7
    return (torch.round(wg / s[..., None]).clamp(-8, 7).double() * s.double()[..., None]).view(w.shape)


_DQ = {"int8": _dq8, "int4": _dq4, "bf16": lambda w: w.double()}


def _decode_weight(case):
    """weight -> what a decode step at this batch multiplies in its place: its quantized form, or itself where the
    package's dispatch takes the kept bf16 copy."""
    def read(w, rows=None):
        N, K = rows or w.shape[0], w.shape[1]
        path = linear_path(case["fmt"], case["fmt"], case["batch"], N, K, case["fmt"] != "bf16")
        return w.double() if path == "linear" else _DQ[case["fmt"]](w)
    return read


def _fq(x, group):
    """x as the W8A8 layers see it: INT8 with a scale per row, or per row and group of columns."""
    xg = x.reshape(x.shape[0], -1, group or x.shape[1])
    s = xg.abs().amax(-1, keepdim=True).clamp_min(1e-8) / 127
    return (torch.round(xg / s).clamp(-127, 127) * s).view_as(x)


def _rms(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _rotate(x, pos):
    """Rotary embedding of x [B, T, heads, HEAD_DIM] at positions pos [T]."""
    freq = (THETA ** (-torch.arange(0, HEAD_DIM, 2, device=DEV, dtype=torch.float32) / HEAD_DIM)).double()
    ang = (pos.double()[:, None] * freq).repeat(1, 2)[:, None]
    a, b = x.chunk(2, -1)
    return x * ang.cos() + torch.cat((-b, a), -1) * ang.sin()


def _forward(net, ids, past, wt, quant, all_logits):
    """The model over ids [B, T] behind the cache `past` ({layer: (k, v) or conv inputs}), weights by wt and linear
    inputs by quant, in 64 bits; the cache is extended in place. Logits of every position or of the last."""
    lm = net.model
    B, T = ids.shape
    first = past.setdefault("n", 0)
    past["n"] = first + T
    pos = torch.arange(first, first + T, device=DEV)
    h = lm.embed_tokens.weight[ids].double()

    def lin(x, *ws):
        x2 = quant(x.reshape(B * T, -1))
        return torch.cat([x2 @ wt(w, sum(v.shape[0] for v in ws)).t() for w in ws], -1).view(B, T, -1)

    for i, layer in enumerate(lm.layers):
        x = _rms(h, layer.operator_norm.weight)
        if LAYERS[i] == "A":
            a = layer.self_attn
            qkv = lin(x, a.q_proj.weight, a.k_proj.weight, a.v_proj.weight).view(B, T, -1, HEAD_DIM)
            q, k, v = qkv.split((HEADS, KV_HEADS, KV_HEADS), 2)
            q, k = _rotate(_rms(q, a.q_layernorm.weight), pos), _rotate(_rms(k, a.k_layernorm.weight), pos)
            if i in past:
                k, v = torch.cat((past[i][0], k), 1), torch.cat((past[i][1], v), 1)
            past[i] = (k, v)
            seen = torch.arange(k.shape[1], device=DEV)[None] <= pos[:, None]
            o = torch.empty_like(q)
            for head in range(HEADS):
                kh, vh = (t[:, :, head * KV_HEADS // HEADS].contiguous() for t in (k, v))
                sc = q[:, :, head] @ kh.transpose(1, 2).contiguous() * HEAD_DIM ** -0.5
                o[:, :, head] = torch.softmax(sc.masked_fill(~seen, -math.inf), -1) @ vh
            h = h + lin(o.reshape(B, T, H), a.out_proj.weight)
        else:
            c = layer.conv
            b_, c_, x_ = lin(x, c.in_proj.weight).chunk(3, -1)
            u = torch.cat((past.get(i, b_.new_zeros(B, CONV_LEN, H)), b_ * x_), 1)
            past[i] = u[:, -CONV_LEN:]
            taps = c.conv.weight[:, 0].double()
            y = sum(u[:, j + 1:j + 1 + T] * taps[:, j] for j in range(CONV_LEN))
            h = h + lin(c_ * y, c.out_proj.weight)
        f = layer.feed_forward
        g, u = lin(_rms(h, layer.ffn_norm.weight), f.w1.weight, f.w3.weight).chunk(2, -1)
        h = h + lin(F.silu(g) * u, f.w2.weight)
    return h if all_logits else h[:, -1:]


def _caches(net, past, max_len):
    """The cache as the decoder lays it out: keys [B, kv, HEAD_DIM, max_len], values [B, kv, max_len, HEAD_DIM], the
    last conv inputs in a ring of CONV_LEN rows (position p in row p mod CONV_LEN)."""
    n, ks, vs, rings = past["n"], [], [], []
    for i in range(len(net.model.layers)):
        if LAYERS[i] == "A":
            k, v = past[i]
            pad = (0, 0, 0, 0, 0, max_len - n)
            ks.append(F.pad(k, pad).permute(0, 2, 3, 1).contiguous())
            vs.append(F.pad(v, pad).transpose(1, 2).contiguous())
        else:
            rings.append(torch.roll(past[i].transpose(0, 1), n % CONV_LEN, 0).contiguous())
    return ks, vs, rings


def _head(net, h, wt):
    return _rms(h, net.model.embedding_norm.weight) @ wt(net.lm_head.weight, VOCAB).t()


@torch.no_grad()
def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        return s["x"].double() @ _decode_weight(case)(s["w"]).t()
    if kind == "int8_linear":
        x = s["x"].double()
        if case["mode"] != "a16":
            x = _fq(x, GROUP if case["mode"] == "group" else 0)
        y = x @ _dq8(s["w"]).t()
        y = y if s["b"] is None else y + s["b"].double()
        return F.gelu(y, approximate="tanh") if case["gelu"] else y
    if kind == "lm_ffn":
        h = (s["h"].double() + s["y"].double())
        g, u = (_fq(_rms(h, s["norm"]), case["group"]) @ _dq8(s["w13"]).t()).chunk(2, -1)
        return h, _fq(F.silu(g) * u, GROUP) @ _dq8(s["w2"]).t()
    if kind == "vision_ffn":
        h = (s["h"].double() + s["y"].double())
        x = F.layer_norm(h, (V_DIM,), s["norm"].double(), s["shift"].double(), V_EPS)
        y = _fq(x, GROUP) @ _dq8(s["w1"]).t() + s["b1"].double()
        y = _fq(F.pad(F.gelu(y, approximate="tanh"), (0, V_PAD)), GROUP)[:, :V_FFN]
        return h, y @ _dq8(s["w2"]).t() + s["b2"].double()
    net, ids, past = s["net"], s["ids"], {}
    def plain(w, rows):
        return w.double()

    def int8(w, rows):
        return _dq8(w)

    if kind == "decode":
        P, n = case["prompt"], case["steps"]
        _forward(net, ids[:, :P], past, plain, lambda x: x, False)
        wt = _decode_weight(case)
        h = _forward(net, ids[:, P:], past, wt, lambda x: x, True)
        return (_head(net, h, wt).transpose(0, 1).contiguous(), *_caches(net, past, -(-(P + n + 1) // 256) * 256))
    w8 = case["mode"] == "int8"
    wt = int8 if w8 else plain
    h = _forward(net, ids, past, wt, (lambda x: _fq(x, GROUP)) if w8 else (lambda x: x), False)
    return (_head(net, h, wt)[:, 0], *_caches(net, past, -(-(case["tokens"] + 1) // 256) * 256))
