"""The calls whose speed counts: what an engine built on libhfmoe has it do.

Every case is one call through the C-ABI (hummingflight_amd.capi), as the
engine's generation loop makes it: the MoE block of a decoder layer at decode,
batched decode and prefill, a dense MLP layer, the LM head, the host contract
and a layer streamed from pinned host RAM.  The engine configures the library
once for its model, registers its layers and calls; weights, activations and
the output buffer sit in GPU memory (host memory for the host contract), and
all work goes to one stream of its own.

Layer shapes: "glm" is the GLM-5.2 MoE layer that the benchmark is quoted on,
"small" the repository's small configuration with flat top-8 routing, "mini"
the shape of the smoke run.  Router rows and activations are made together, so
that a token's experts win clearly, as under a trained router: which experts a
token goes to then does not hang on the last bits of its logits.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from hummingflight_amd import capi

SHAPES = {
    "glm": dict(hidden=6144, inter=2048, experts=256, k=8, groups=8, kept=4, max_tokens=4096),
    "small": dict(hidden=2048, inter=1024, experts=64, k=8, groups=1, kept=1, max_tokens=4096),
    "mini": dict(hidden=512, inter=256, experts=32, k=4, groups=4, kept=2, max_tokens=1024),
}
EPS = 1e-5
SCALE = 2.5
LOGIT_STD = 0.4  # spread of the logits of a token's other experts
VOCAB = {"glm": 154880, "small": 32000, "mini": 1003}
DENSE = {"glm": 12288, "small": 6144, "mini": 1536}


def listed():
    return [
        # The engine's moeLayer with host buffers on the small model: the
        # smallest call, all latency.
        dict(name="host_small_t1", kind="host", shape="small", tokens=1, x="fp32", popularity="uniform"),
        # One token through one small layer, activations on the GPU.
        dict(name="decode_small_t1", kind="moe", shape="small", tokens=1, x="fp32", popularity="uniform"),
        # Single-stream decode at the benchmark's layer: its headline number.
        dict(name="decode_glm_t1", kind="moe", shape="glm", tokens=1, x="fp32", popularity="uniform"),
        # A handful of concurrent requests: the whole MLP half of a decoder
        # layer (norm, MoE, residual), FP32 activations as the norm leaves them.
        dict(name="block_glm_t7", kind="block", shape="glm", tokens=7, x="fp32", popularity="uniform"),
        # Batched decode with skewed expert popularity, BF16-valued activations.
        dict(name="batched_glm_t64_zipf", kind="moe", shape="glm", tokens=64, x="bf16", popularity="zipf"),
        # A prompt chunk mixed into a serving batch, ragged, through the block.
        dict(name="block_glm_t509", kind="block", shape="glm", tokens=509, x="fp32", popularity="zipf"),
        # A full prefill chunk of an engine that keeps BF16 activations.
        dict(name="prefill_glm_t4096", kind="moe_bf16", shape="glm", tokens=4096, x="bf16", popularity="uniform"),
        # A ragged prompt with FP32 activations.
        dict(name="prefill_glm_t3001", kind="moe", shape="glm", tokens=3001, x="fp32", popularity="uniform"),
        # A dense layer (the model's first three) over a ragged prompt.
        dict(name="dense_glm_t777", kind="dense", shape="glm", tokens=777, x="fp32", rows=0),
        # The sampling step of single-stream decode: norm, logits, greedy token.
        dict(name="lm_head_glm_t1", kind="lm_head", shape="glm", tokens=1, x="fp32", rows=0),
        # The same for a batch of requests.
        dict(name="lm_head_glm_t24", kind="lm_head", shape="glm", tokens=24, x="fp32", rows=0),
        # Decode over experts in pinned host RAM: the selected ones cross PCIe.
        dict(name="streamed_small_t1", kind="streamed", shape="small", tokens=1, x="fp32", popularity="uniform"),
    ]


def draw(rng):
    def tokens(most):
        return max(1, min(most, int(round(math.exp(rng.uniform(0.0, math.log(most)))))))

    kind = rng.choice(["moe", "moe", "moe_bf16", "block", "block", "dense", "dense", "lm_head", "lm_head", "host"])
    shape = rng.choice(["glm", "glm", "small", "mini"])
    most = SHAPES[shape]["max_tokens"]
    if kind == "host":
        n = 1
    elif kind == "lm_head":
        n = tokens(128)
    else:
        n = tokens(most)
    x = "bf16" if kind == "moe_bf16" else "fp32" if kind == "block" else rng.choice(["fp32", "fp32", "bf16"])
    case = dict(kind=kind, shape=shape, tokens=n, x=x)
    if kind not in ("dense", "lm_head"):
        case["popularity"] = rng.choice(["uniform", "zipf"])
    else:
        # Dense and LM-head tables are not tied to the MoE shape: a ragged one too.
        case["rows"] = rng.choice([0, 0, 1]) * 64
    return case


# ---------------------------------------------------------------- inputs

_stream = None


def _use_stream():
    """The engine's one stream, torch's current one from here on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
        torch.cuda.set_stream(_stream)
    return _stream


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _bf16(gen, std, *size, mean=0.0):
    """N(mean, std) in BF16, filled in pieces of at most 2^30 values."""
    t = torch.empty(size, dtype=torch.bfloat16, device="cuda")
    flat = t.view(-1)
    for i in range(0, flat.numel(), 1 << 30):
        flat[i:i + (1 << 30)].normal_(mean, std, generator=gen)
    return t


def _plan(case, seed):
    """Experts [T, k] that the tokens go to, on the host."""
    s = SHAPES[case["shape"]]
    T, E, G = case["tokens"], s["experts"], s["groups"]
    r = np.random.RandomState((int(seed) * 1000003 + 17) % (1 << 32))
    p = np.ones(E)
    if case["popularity"] == "zipf":
        p = np.arange(1, E + 1.0) ** -1.1
    p = r.permutation(p)
    # Kept groups, then as many experts of each, by weighted draws without
    # replacement (Gumbel top-k).
    g = np.log(p.reshape(G, -1).sum(1)) + r.gumbel(size=(T, G))
    kept = np.argsort(-g, axis=1)[:, :s["kept"]]
    e = np.log(p).reshape(G, -1)[None] + r.gumbel(size=(T, G, E // G))
    best = np.argsort(-e, axis=2)[:, :, :s["k"] // s["kept"]] + (np.arange(G) * (E // G))[None, :, None]
    return np.take_along_axis(best, kept[:, :, None], axis=1).reshape(T, -1)


def _tokens(case, gen, seed, router):
    """Activations [T, hidden] FP32 (BF16-valued with x = "bf16")."""
    s = SHAPES[case["shape"]]
    T, d = case["tokens"], s["hidden"]
    x = torch.randn(T, d, generator=gen, device="cuda")
    if router is not None:
        idx = torch.from_numpy(_plan(case, seed)).cuda()
        up = torch.rand(T, s["k"], generator=gen, device="cuda") * 2.1 + 2.4  # logits of the token's experts
        mix = torch.zeros(T, s["experts"], device="cuda").scatter_(1, idx, up / LOGIT_STD ** 2)
        x += mix @ router.float()
    return x.bfloat16().float() if case["x"] == "bf16" else x


def _tables(case, seed):
    """Weights and activations of a case, from its seed alone."""
    s = SHAPES[case["shape"]]
    d, I, E = s["hidden"], s["inter"], s["experts"]
    std = 1.57 / math.sqrt(d)  # 0.02 at hidden 6144
    kind = case["kind"]
    if kind == "lm_head":  # the model's one table; a state's own are its tokens
        gen = _generator(VOCAB[case["shape"]] + case["rows"])
        t = dict(head=_bf16(gen, std, VOCAB[case["shape"]] + case["rows"], d), norm=_bf16(gen, 0.05, d, mean=1.0))
        t["x"] = _tokens(case, _generator(seed), seed, None)
        return t
    gen = _generator(seed)
    if kind == "dense":
        n = DENSE[case["shape"]] + case["rows"]
        t = dict(gate=_bf16(gen, std, n, d), up=_bf16(gen, std, n, d), down=_bf16(gen, std, d, n))
        t["x"] = _tokens(case, gen, seed, None)
        return t
    t = dict(router=_bf16(gen, LOGIT_STD / math.sqrt(d), E, d), norm=_bf16(gen, 0.05, d, mean=1.0),
             bias=torch.randn(E, generator=gen, device="cuda") * 0.01,
             experts=_bf16(gen, std, E, 3, I * d), shared=_bf16(gen, std, 3, I * d))
    t["x"] = _tokens(case, gen, seed, t["router"])
    if kind == "block":
        t["x"] *= 3.0  # a residual stream, not yet normalised
    return t


# ---------------------------------------------------------------- the library

_configured = None
_next_layer = 0


def _configure(case):
    """The engine's start-up: one model per process at a time."""
    global _configured, _next_layer
    if _configured == case["shape"]:
        return
    s = SHAPES[case["shape"]]
    torch.cuda.synchronize()
    capi.call("hfmoe_init", torch.cuda.current_device())
    capi.call("hfmoe_configure", ctypes.byref(capi.Config(
        s["hidden"], s["inter"], s["experts"], s["k"], s["groups"], s["kept"], 1, 1, SCALE, EPS, 0, s["max_tokens"], 0)))
    _configured, _next_layer = case["shape"], 0


_head = {}  # the registered LM head's tables


def prepare(case, seed):
    global _next_layer
    stream = _use_stream().cuda_stream
    _configure(case)
    s, kind, T = SHAPES[case["shape"]], case["kind"], case["tokens"]
    d, I, E = s["hidden"], s["inter"], s["experts"]
    layer, _next_layer = _next_layer, _next_layer + 2
    if kind == "lm_head":
        key = (case["shape"], VOCAB[case["shape"]] + case["rows"])
        if _head.get("key") != key:
            _head.clear()
            t = _tables(case, seed)
            _head.update(key=key, head=t["head"], norm=t["norm"])
            x = t["x"]
        else:
            x = _tokens(case, _generator(seed), seed, None)
        capi.call("hfmoe_register_lm_head", _head["head"].data_ptr(), _head["norm"].data_ptr(), key[1])
        return dict(call="hfmoe_lm_head", x=x, out=torch.empty(T, key[1], device="cuda"),
                    token=torch.empty(T, dtype=torch.int32, device="cuda"), T=T, stream=stream)
    _head.clear()
    t = _tables(case, seed)
    if kind == "dense":
        w = capi.DenseWeights(t["gate"].data_ptr(), t["up"].data_ptr(), t["down"].data_ptr(), None, t["gate"].shape[0], 0)
        capi.call("hfmoe_register_dense_layer", layer, ctypes.byref(w))
        return dict(call="hfmoe_dense_mlp_forward", tables=t, layer=layer, x=t["x"], out=torch.empty(T, d, device="cuda"),
                    T=T, stream=stream)
    if kind == "streamed":
        host = torch.empty(t["experts"].shape, dtype=torch.bfloat16, pin_memory=True)
        host.copy_(t["experts"])
        t["experts"] = host
    base, size = t["experts"].data_ptr(), I * d * 2
    table = (ctypes.c_void_p * (3 * E))(*[base + i * size for i in range(3 * E)])
    sh = t["shared"].data_ptr()
    w = capi.LayerWeights(t["router"].data_ptr(), t["bias"].data_ptr(), sh, sh + size, sh + 2 * size,
                          ctypes.cast(table, ctypes.c_void_p), t["norm"].data_ptr(),
                          capi.EXPERTS_HOST_PINNED if kind == "streamed" else capi.EXPERTS_DEVICE, 0)
    torch.cuda.synchronize()
    capi.call("hfmoe_register_layer", layer, ctypes.byref(w))
    st = dict(tables=t, layer=layer, T=T, stream=stream, x=t["x"])
    if kind == "host":
        st.update(call="hfmoe_moe_layer", x=t["x"][0].cpu().numpy(), out=np.empty(d, np.float32))
    elif kind == "block":
        st.update(call="hfmoe_mlp_block", out=torch.empty(T, d, device="cuda"))
    elif kind == "moe_bf16":
        st.update(call="hfmoe_moe_forward_bf16", x=t["x"].bfloat16(), out=torch.empty(T, d, device="cuda"))
    else:
        st.update(call="hfmoe_moe_forward", out=torch.empty(T, d, device="cuda"))
    return st


def run(st):
    call = st["call"]
    if call == "hfmoe_moe_layer":
        capi.call(call, st["layer"], st["x"].ctypes.data, st["out"].ctypes.data)
        return st["out"]
    if call == "hfmoe_mlp_block":  # updates the residual stream, which attention has just written
        st["out"].copy_(st["x"])
        capi.call(call, st["layer"], st["out"].data_ptr(), st["T"], st["stream"])
        return st["out"]
    if call == "hfmoe_lm_head":
        capi.call(call, st["x"].data_ptr(), st["T"], st["out"].data_ptr(), st["token"].data_ptr(), st["stream"])
        return {"logits": st["out"], "token": st["token"]}
    capi.call(call, st["layer"], st["x"].data_ptr(), st["T"], st["out"].data_ptr(), st["stream"])
    return st["out"]


# ---------------------------------------------------------------- what a pass needs


def work(case):
    s, kind, T = SHAPES[case["shape"]], case["kind"], case["tokens"]
    d, I, E = s["hidden"], s["inter"], s["experts"]
    if kind == "lm_head":
        V = VOCAB[case["shape"]] + case["rows"]
        return {"bytes": 2 * V * d + 4 * T * (d + V), "flops": 2 * T * V * d}
    if kind == "dense":
        n = DENSE[case["shape"]] + case["rows"]
        return {"bytes": 6 * n * d + 8 * T * d, "flops": 6 * T * n * d}
    hit = len(np.unique(_plan(case, 1)))
    x_bytes = 2 if kind == "moe_bf16" else 4
    return {"bytes": 6 * d * I * (hit + 1) + 2 * E * d + (x_bytes + 4) * T * d,
            "flops": 6 * d * I * T * (s["k"] + 1) + 2 * T * E * d}


def tolerance(case):
    # One token is summed in FP32 throughout (2e-7 to 3.2e-7 off the 64-bit
    # result); a batch's FP32 values go through the matrix cores as two BF16
    # halves, about 16 bits (2.3e-6 to 4.4e-6 off).  About four times that.
    t = {"rel": 2e-6 if case["tokens"] == 1 else 2e-5}
    if case["kind"] == "lm_head":
        t["differ"] = 0.01
    return t


# ---------------------------------------------------------------- the same in 64 bits


def _silu_mul(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def _rms_norm(h, w):
    return h * torch.rsqrt((h * h).mean(1, keepdim=True) + EPS) * w.double()


def _swiglu(x, gate, up, down):
    """x [n, d] in 64 bits through one expert, a slice of its rows at a time."""
    out = torch.zeros_like(x)
    for i in range(0, gate.shape[0], 4096):
        h = _silu_mul(x @ gate[i:i + 4096].double().t(), x @ up[i:i + 4096].double().t())
        out += h @ down[:, i:i + 4096].double().t()
    return out


def exact(case, seed):
    _use_stream()
    s, kind = SHAPES[case["shape"]], case["kind"]
    d, I, E, k = s["hidden"], s["inter"], s["experts"], s["k"]
    t = _tables(case, seed)
    x = t["x"].double()
    if kind == "lm_head":
        xn = _rms_norm(x, t["norm"])
        w = t["head"]
        logits = torch.cat([xn @ w[i:i + 8192].double().t() for i in range(0, w.shape[0], 8192)], 1)
        return {"logits": logits, "token": None}
    if kind == "dense":
        return _swiglu(x, t["gate"], t["up"], t["down"])
    h, x = x, _rms_norm(x, t["norm"]) if kind == "block" else x
    score = torch.sigmoid(x @ t["router"].double().t())
    key = score + t["bias"].double()
    if s["groups"] > 1:
        g = key.view(len(x), s["groups"], -1)
        best = g.topk(2, 2).values.sum(2).topk(s["kept"], 1).indices
        keep = torch.zeros(len(x), s["groups"], dtype=torch.bool, device="cuda").scatter_(1, best, True)
        key = g.masked_fill(~keep[:, :, None], -math.inf).view(len(x), E)
    idx = key.topk(k, 1).indices
    wt = score.gather(1, idx)
    wt = SCALE * wt / wt.sum(1, keepdim=True)
    out = _swiglu(x, t["shared"][0].view(I, d), t["shared"][1].view(I, d), t["shared"][2].view(d, I))
    for e in idx.unique().tolist():
        row, rank = (idx == e).nonzero(as_tuple=True)
        we = t["experts"][e]
        out[row] += wt[row, rank, None] * _swiglu(x[row], we[0].view(I, d), we[1].view(I, d), we[2].view(d, I))
    if kind == "host":
        return out[0]
    return h + out if kind == "block" else out
