"""The measured work of this backend: what an inference host has it do, call by
call, through the C-ABI entry points of infer_hip.

Four kinds of case, over the ranges that the supported models span:

- linear: one Linear of `rows` activation rows (1 row: a decode step; 2..16:
  several sequences decoded together; up to 1024: a prompt chunk) over a
  weight of any block or float type, in the CPU's arithmetic (mode q8) or the
  float one (mode f32);
- attention: the causal attention of `rows` new rows over a cache, decode and
  prompt, with or without a window and sinks, float or half-float keys;
- experts: the routed experts of one token, as the layer operations are
  enqueued one by one (route, gate, up, SwiGLU, down, combine);
- model: a decoder of a few layers of a family (moe: Qwen3-30B-A3B's layers,
  dense: Qwen3-0.6B's, delta: Qwen3.5's Gated DeltaNet and gated attention),
  a prompt chunk or decode steps through its context.

Weights are GGUF blocks of random codes with scales of trained weights' spread
(sigma about 0.02), activations are normal with a few larger channels.
"""
import json
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "mormot2-ai_amd"))

import infer_hip as H  # noqa: E402

TYPES = {"Q8_0": H.Q8_0, "Q4_0": H.Q4_0, "Q5_0": H.Q5_0, "Q5_1": H.Q5_1, "Q4_K": H.Q4_K,
         "Q6_K": H.Q6_K, "MXFP4": H.MXFP4, "F32": H.F32, "F16": H.F16, "BF16": H.BF16}
K_QUANTS = ("Q4_K", "Q6_K")
FLOATS = ("F32", "F16", "BF16")

# layer shapes of the supported families (infer_hip.models)
FAMILIES = {
    "moe": dict(hidden=2048, heads=32, kv_heads=4, head_dim=128, experts=128, experts_used=8,
                expert_ffn=768, ffn=0, theta=1e6, eps=1e-6),
    "dense": dict(hidden=1024, heads=16, kv_heads=8, head_dim=128, experts=0, experts_used=0,
                  expert_ffn=0, ffn=3072, theta=1e6, eps=1e-6),
    "delta": dict(hidden=1024, heads=8, kv_heads=2, head_dim=256, experts=0, experts_used=0,
                  expert_ffn=0, ffn=3584, theta=1e7, eps=1e-6, rope_dims=64, lin_heads=16,
                  lin_dim=128, conv=4),
}
VOCAB = 4096


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a token's 8 of 128 experts, the layer operations enqueued one by one
        dict(name="experts-token", kind="experts", type="Q4_K", experts=128, used=8, hidden=2048,
             ffn=768),
        # a decode step's attention of a layer after a 1151-token context
        dict(name="attention-decode", kind="attention", rows=1, past=1151, heads=32, kv_heads=4,
             head_dim=128, window=0, sinks=False, half=True),
        # the output head of a decode step: the largest one-row product
        dict(name="linear-head", kind="linear", type="Q6_K", rows=1, cols=2048, out=151936,
             mode="q8"),
        # eight sequences decoded together
        dict(name="linear-batch8", kind="linear", type="Q4_K", rows=8, cols=2048, out=6144,
             mode="q8"),
        # a projection of a 512-token prompt chunk
        dict(name="linear-prompt", kind="linear", type="Q4_K", rows=512, cols=2048, out=6144,
             mode="q8"),
        # a feed-forward down projection of a short prompt, a ragged row count
        dict(name="linear-ragged", kind="linear", type="Q8_0", rows=301, cols=3072, out=1024,
             mode="q8"),
        # a BF16 query projection of a full prompt chunk (gpt-oss-20b's)
        dict(name="linear-bf16", kind="linear", type="BF16", rows=1024, cols=2880, out=4096,
             mode="q8"),
        # prompt attention, causal from an empty cache
        dict(name="attention-prompt", kind="attention", rows=1024, past=0, heads=32, kv_heads=4,
             head_dim=128, window=0, sinks=False, half=True),
        # a later prompt chunk of a sliding-window layer with sinks
        dict(name="attention-window", kind="attention", rows=1000, past=1048, heads=64, kv_heads=8,
             head_dim=64, window=128, sinks=True, half=True),
        # prompt and decode of mixture-of-experts layers
        dict(name="prefill-moe", kind="model", family="moe", layers=2, past=0, rows=1024, steps=0),
        dict(name="decode-moe", kind="model", family="moe", layers=2, past=1024, rows=0, steps=16),
        # a prompt through a Gated DeltaNet layer and a gated attention layer
        dict(name="prefill-delta", kind="model", family="delta", layers=2, past=0, rows=512,
             steps=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("linear", "attention", "experts", "model"), (10, 6, 2, 3))[0]
    if kind == "linear":
        t = rng.choice(list(TYPES))
        mode = "f32" if rng.random() < 0.15 else "q8"
        rows = _log(rng, 1, 64 if mode == "f32" else 1024)
        unit = 256 if t in K_QUANTS else 32
        cols = unit * max(1, round(_log(rng, 256, 4096) / unit))
        out = _log(rng, 64, 16384)
        out = max(64, min(out, int(12e9 / (rows * cols))))
        return dict(kind=kind, type=t, rows=rows, cols=cols, out=out, mode=mode)
    if kind == "attention":
        heads, kv, hd = rng.choice(((32, 4, 128), (16, 8, 128), (64, 8, 64), (8, 2, 256),
                                    (16, 8, 256), (14, 2, 64)))
        windowed = rng.random() < 0.35
        rows = _log(rng, 1, 1024)
        return dict(kind=kind, rows=rows, past=rng.choice((0, _log(rng, 1, 2048))), heads=heads,
                    kv_heads=kv, head_dim=hd, window=rng.choice((128, 1024)) if windowed else 0,
                    sinks=windowed and hd == 64, half=rng.random() < 0.8)
    if kind == "experts":
        return dict(kind=kind, type=rng.choice(("Q4_K", "Q6_K", "MXFP4", "Q8_0")),
                    experts=rng.choice((8, 16, 32, 64)), used=rng.choice((1, 2, 4, 6, 8)),
                    hidden=256 * rng.randint(2, 8), ffn=256 * rng.randint(1, 8))
    family = rng.choice(("moe", "dense", "delta"))
    steps = 0 if family == "delta" or rng.random() < 0.5 else rng.randint(1, 16)
    past = 0 if family == "delta" else _log(rng, 1, 1024) if steps or rng.random() < 0.3 else 0
    rows = 0 if steps else _log(rng, 2, 512 if past else 1024)
    return dict(kind="model", family=family, layers=rng.randint(1, 2), past=past, rows=rows,
                steps=steps)


# ------------------------------------------------------- GGUF blocks, dequant
def _halfs(rng, shape, base):
    return (rng.uniform(0.8, 1.2, shape) * base).astype(np.float16)[..., None].view(np.uint8)


def blocks(rng, name, rows, cols):
    """A [rows, cols] weight of the type as GGUF bytes."""
    if name in FLOATS:
        a = rng.standard_normal((rows, cols), np.float32) * np.float32(0.02)
        if name == "F32":
            return a
        if name == "F16":
            return a.astype(np.float16)
        u = a.view(np.uint32)
        return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)
    bv, bs = H.BLOCK[TYPES[name]]
    nb = cols // bv
    b = rng.integers(0, 256, (rows, nb, bs), dtype=np.uint8)
    n = (rows, nb)
    if name == "Q8_0":
        b[..., 0:2] = _halfs(rng, n, 0.02 / 73)
    elif name == "Q4_0":
        b[..., 0:2] = _halfs(rng, n, 0.02 / 4.6)
    elif name == "Q5_0":
        b[..., 0:2] = _halfs(rng, n, 0.02 / 9.2)
    elif name == "Q5_1":
        b[..., 0:2] = _halfs(rng, n, 0.02 / 9.2)
        b[..., 2:4] = _halfs(rng, n, -0.02 / 9.2 * 15.5)
    elif name == "MXFP4":
        b[..., 0] = rng.integers(119, 122, n)
    elif name == "Q4_K":
        # the minimum of a sub-block follows its scale
        b[..., 0:2] = _halfs(rng, n, 0.02 / 150)
        b[..., 2:4] = _halfs(rng, n, 0.02 / 150 * 7.5)
        b[..., 8:12] = b[..., 4:8]
        b[..., 12:16] = (b[..., 12:16] & 15) * 17
    elif name == "Q6_K":
        b[..., 208:210] = _halfs(rng, n, 0.02 / 1400)
    return b


_MX = torch.tensor([0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12], dtype=torch.float64)


def dense(a, name, rows, cols):
    """The weight's values in 64 bits on the GPU."""
    if name == "F32" or name == "F16":
        return torch.from_numpy(a.reshape(rows, cols)).cuda().double()
    if name == "BF16":
        u = torch.from_numpy(a.astype(np.int32).reshape(rows, cols)).cuda() << 16
        return u.view(torch.float32).double()
    bv, bs = H.BLOCK[TYPES[name]]
    t = torch.from_numpy(a.reshape(rows, cols // bv, bs)).cuda()

    def half(i):
        return t[..., i:i + 2].contiguous().view(torch.float16).double()

    def nibbles(i):
        q = t[..., i:i + 16]
        return torch.cat([q & 15, q >> 4], -1).double()

    def fifth(i):
        w = t[..., i:i + 4].int()
        v = torch.arange(32, device=t.device)
        return ((w[..., v // 8] >> (v % 8)) & 1).double() * 16

    if name == "Q8_0":
        v = half(0) * t[..., 2:].contiguous().view(torch.int8).double()
    elif name == "Q4_0":
        v = half(0) * (nibbles(2) - 8)
    elif name == "Q5_0":
        v = half(0) * (nibbles(6) + fifth(2) - 16)
    elif name == "Q5_1":
        v = half(0) * (nibbles(8) + fifth(4)) + half(2)
    elif name == "MXFP4":
        q = nibbles(1).long()
        v = torch.exp2(t[..., 0:1].double() - 128) * _MX.cuda()[q]
    elif name == "Q4_K":
        s = t[..., 4:16].int()
        lo, mid, hi = s[..., 0:4], s[..., 4:8], s[..., 8:12]
        sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], -1).double()
        mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], -1).double()
        q = t[..., 16:].reshape(rows, -1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], -2).reshape(rows, -1, 8, 32).double()
        v = (half(0) * sc)[..., None] * q - (half(2) * mn)[..., None]
    else:
        ql = t[..., 0:128].reshape(rows, -1, 2, 2, 32)
        ql = torch.cat([ql & 15, ql >> 4], -2).int()
        sh = torch.arange(0, 8, 2, device=t.device, dtype=torch.int32)[:, None]
        qh = (t[..., 128:192].reshape(rows, -1, 2, 1, 32).int() >> sh) & 3
        q = (ql | (qh << 4)).reshape(rows, -1, 16, 16).double() - 32
        sc = t[..., 192:208].contiguous().view(torch.int8).double()
        v = (half(208) * sc)[..., None] * q
    return v.reshape(rows, cols)


def quantized(x, name):
    """The activation rows as the CPU's quantizers of the type hold them."""
    x = x.float()
    if name in FLOATS:
        return x.double()
    if name in K_QUANTS:
        b = x.reshape(x.shape[0], -1, 256)
        top = b.gather(-1, b.abs().argmax(-1, keepdim=True))
        inv = (-127.0 / top.double()).float()  # (a single quotient, rounded once)
        q = torch.round(inv * b).clamp(max=127)
        d = (1.0 / inv.double()).float().double()
    else:
        b = x.reshape(x.shape[0], -1, 32)
        s = (b.abs().amax(-1, keepdim=True).double() / 127.0).float()
        q = torch.round(b * (1.0 / s.double()).float())
        d = s.half().double()
    return torch.nan_to_num(q.double() * d).reshape(x.shape)


def linear64(x, a, name, out, cols, mode="q8"):
    xq = quantized(x, name) if mode == "q8" else x.double()
    y = torch.empty((x.shape[0], out), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 28) // cols)
    a = a.reshape(out, -1) if name in FLOATS else a.reshape(out, -1, a.shape[-1])
    for o in range(0, out, step):
        n = min(step, out - o)
        y[:, o:o + n] = xq @ dense(a[o:o + n], name, n, cols).T
    return y


def attention64(q, k, v, c):
    """q [rows, heads, hd] at the end of k, v [total, kv_heads, hd]."""
    rows, heads, hd = q.shape
    total, kvh = k.shape[0], k.shape[1]
    past = total - rows
    pos = torch.arange(total, device="cuda")
    at = past + torch.arange(rows, device="cuda")[:, None]
    seen = pos[None] <= at
    if c.get("window"):
        seen &= pos[None] > at - c["window"]
    y = torch.empty((rows, heads, hd), dtype=torch.float64, device="cuda")
    for h in range(heads):
        g = h // (heads // kvh)
        s = (q[:, h].double() @ k[:, g].double().T) * hd ** -0.5
        s = s.masked_fill(~seen, -math.inf)
        if c.get("sinks") is not None and c["sinks"] is not False:
            s = torch.cat([s, c["sinks"][h].double().expand(rows, 1)], 1)
        y[:, h] = torch.softmax(s, -1)[:, :total] @ v[:, g].double()
    return y


def silu64(x):
    x = x.double()
    return x / (1 + torch.exp(-x))


# ------------------------------------------------------------------- prepare
_ctx = None


def ctx():
    global _ctx
    if _ctx is None:
        _ctx = H.Context(0)
    return _ctx


_loaded = set()


def _load(s):
    """The first call of a kind of case loads its kernels. The lookups that miss
    on the way are left as HIP's last error, which torch would take for its
    own at its next launch: read here, once per kind of case."""
    key = json.dumps({k: v for k, v in s.case.items() if k != "name"}, sort_keys=True)
    if key in _loaded:
        return
    _loaded.add(key)
    run(s)
    try:
        torch.zeros(1, device="cuda")
    except RuntimeError:
        pass
    torch.cuda.synchronize()


class State:
    """What a program has in hand: device inputs and outputs, and the weights'
    device copies, dropped with it."""

    def __init__(self):
        self.host = []

    def weight(self, a, name, out, cols, count=1):
        d = H.C.c_uint64()
        H.check(H.lib().ihip_weight(ctx().h, a.ctypes.data, TYPES[name], out, cols, count,
                                    H.C.byref(d)), "weight")
        self.host.append(a)
        return d.value

    def __del__(self):
        for a in self.host:
            H.lib().ihip_forget_weights(ctx().h, a.ctypes.data, a.ctypes.data + a.nbytes)


def _rows(rng, rows, cols):
    """Activation rows: normal, every 97th channel larger."""
    x = rng.standard_normal((rows, cols), np.float32)
    x[:, ::97] *= 6
    return x


def _linear_inputs(c, seed):
    rng = np.random.default_rng([seed, 1])
    return _rows(rng, c["rows"], c["cols"]), blocks(rng, c["type"], c["out"], c["cols"])


def _attention_inputs(c, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    total, hd = c["past"] + c["rows"], c["head_dim"]

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda")

    q = normal(c["rows"], c["heads"], hd)
    k, v = normal(total, c["kv_heads"], hd), normal(total, c["kv_heads"], hd)
    if c["half"]:
        k, v = k.half(), v.half()
    return q, k, v, normal(c["heads"]) if c["sinks"] else None


def _experts_inputs(c, seed):
    rng = np.random.default_rng([seed, 2])
    e, h, f = c["experts"], c["hidden"], c["ffn"]
    return (_rows(rng, 1, h), rng.standard_normal(e, np.float32),
            blocks(rng, c["type"], e * f, h), blocks(rng, c["type"], e * f, h),
            blocks(rng, c["type"], e * h, f))


class Decoder:
    """The tensors of a few layers of a family and the model on the device."""

    def __init__(self, c):
        f = FAMILIES[c["family"]]
        self.f, self.layers_n = f, c["layers"]
        self.keep, self.t = [], {}
        self.rng = np.random.default_rng([5, c["layers"], len(c["family"])])
        self.vocab = VOCAB
        h, hd = f["hidden"], f["head_dim"]
        qw, kvw = f["heads"] * hd, f["kv_heads"] * hd
        delta = c["family"] == "delta"
        d = H.ModelDesc()
        d.vocab, d.hidden, d.layers = VOCAB, h, c["layers"]
        d.heads, d.kv_heads, d.head_dim, d.ffn = f["heads"], f["kv_heads"], hd, f["ffn"]
        d.experts, d.experts_used = f["experts"], f["experts_used"]
        d.expert_ffn, d.norm_topk = f["expert_ffn"], int(f["experts"] > 0)
        d.max_positions, d.rms_eps, d.swiglu_alpha = 1 << 20, f["eps"], 1.0
        d.rope_theta, d.rope_dims = f["theta"], f.get("rope_dims", 0)
        if delta:
            d.lin_key_heads = d.lin_value_heads = f["lin_heads"]
            d.lin_key_dim = d.lin_value_dim = f["lin_dim"]
            d.lin_conv = f["conv"]
        base = "Q8_0" if delta else "Q4_K"
        more = "Q8_0" if delta else "Q6_K"
        d.embed = self.mat("embed", more, VOCAB, h)
        d.final_norm = self.norm("final_norm", h)
        ls = (H.LayerDesc * c["layers"])()
        for i in range(c["layers"]):
            L = ls[i]
            L.input_norm = self.norm((i, "input_norm"), h)
            L.post_norm = self.norm((i, "post_norm"), h)
            if delta and i % 2 == 0:
                n, dim = f["lin_heads"], f["lin_dim"]
                vd, cd = n * dim, 3 * n * dim
                L.mixer = H.MIXER_DELTANET
                L.lin_qkv = self.mat((i, "lin_qkv"), base, cd, h)
                L.lin_z = self.mat((i, "lin_z"), base, vd, h)
                L.lin_b = self.mat((i, "lin_b"), base, n, h)
                L.lin_a = self.mat((i, "lin_a"), base, n, h)
                L.lin_out = self.mat((i, "lin_out"), base, h, vd)
                L.lin_conv = self.vec((i, "conv"), self.rng.standard_normal((cd, f["conv"])) * 0.3)
                L.lin_dt_bias = self.vec((i, "dt"), self.rng.standard_normal(n) * 0.5)
                L.lin_neg_a = self.vec((i, "neg_a"), -np.exp(self.rng.standard_normal(n) * 0.5))
                L.lin_norm = self.norm((i, "lin_norm"), dim)
            else:
                L.output_gate = int(delta)
                L.q = self.mat((i, "q"), base, qw * (2 if delta else 1), h)
                L.k = self.mat((i, "k"), base, kvw, h)
                L.v = self.mat((i, "v"), more, kvw, h)
                L.o = self.mat((i, "o"), base, h, qw)
                L.q_norm, L.k_norm = self.norm((i, "q_norm"), hd), self.norm((i, "k_norm"), hd)
            if f["experts"]:
                e, fi = f["experts"], f["expert_ffn"]
                L.moe = H.FFN_MOE
                L.router = self.mat((i, "router"), "F32", e, h)
                L.exp_gate = self.mat((i, "gate"), base, e * fi, h)
                L.exp_up = self.mat((i, "up"), base, e * fi, h)
                L.exp_down = self.mat((i, "down"), more, e * h, fi)
            else:
                L.gate = self.mat((i, "gate"), base, f["ffn"], h)
                L.up = self.mat((i, "up"), base, f["ffn"], h)
                L.down = self.mat((i, "down"), more, h, f["ffn"])
        self.ls = ls
        d.layer = H.C.cast(ls, H.C.POINTER(H.LayerDesc))
        self.struct = d

    def mat(self, key, name, rows, cols):
        a = blocks(self.rng, name, rows, cols)
        self.t[key] = (a, name, rows, cols)
        return H.Tensor(a.ctypes.data, TYPES[name], 0)

    def vec(self, key, a):
        a = np.ascontiguousarray(a, np.float32)
        self.t[key] = a
        return H.Tensor(a.ctypes.data, H.F32, 0)

    def norm(self, key, n):
        return self.vec(key, 1 + 0.1 * self.rng.standard_normal(n))


_model = {}


def _decoder(c):
    """The model of the case's layers, loaded once and kept, as a host does."""
    key = json.dumps([c["family"], c["layers"]])
    if key not in _model:
        _model.clear()
        d = Decoder(c)
        _model[key] = (d, H.Model(ctx(), d, mode=H.MODE_Q8, kv_f16=True, max_tokens=64))
    return _model[key]


def _tokens(c, seed):
    rng = np.random.default_rng([seed, 3])
    return (rng.integers(0, VOCAB, c["past"], dtype=np.int32),
            rng.integers(0, VOCAB, max(c["rows"], 1), dtype=np.int32))


def prepare(case, seed):
    c, s = case, State()
    s.case = c
    if c["kind"] == "linear":
        x, w = _linear_inputs(c, seed)
        s.w = s.weight(w, c["type"], c["out"], c["cols"])
        s.x = torch.from_numpy(x).cuda()
        s.y = torch.zeros((c["rows"], c["out"]), device="cuda")
    elif c["kind"] == "attention":
        s.q, s.k, s.v, s.sinks = _attention_inputs(c, seed)
        s.y = torch.zeros_like(s.q)
    elif c["kind"] == "experts":
        x, lg, wg, wu, wd = _experts_inputs(c, seed)
        e, h, f, k = c["experts"], c["hidden"], c["ffn"], c["used"]
        s.wg, s.wu = (s.weight(a, c["type"], f, h, e) for a in (wg, wu))
        s.wd = s.weight(wd, c["type"], h, f, e)
        s.x, s.lg = torch.from_numpy(x).cuda(), torch.from_numpy(lg).cuda()
        s.ids = torch.zeros(k, dtype=torch.int32, device="cuda")
        s.rw = torch.zeros(k, device="cuda")
        s.g, s.u = torch.zeros((k, f), device="cuda"), torch.zeros((k, f), device="cuda")
        s.d, s.y = torch.zeros((k, h), device="cuda"), torch.zeros(h, device="cuda")
    else:
        _, s.model = _decoder(c)
        past, s.ids = _tokens(c, seed)
        s.ctx = s.model.new_context()
        if c["past"]:
            s.ctx.forward(past)
    torch.cuda.synchronize()
    _load(s)
    return s


def run(s):
    c, L, h = s.case, H.lib(), ctx().h
    if c["kind"] == "linear":
        mode = H.MODE_Q8 if c["mode"] == "q8" else H.MODE_F32
        H.check(L.ihip_enqueue_linear_at(h, s.x.data_ptr(), c["rows"], c["cols"], TYPES[c["type"]],
                                         s.w, c["out"], s.y.data_ptr(), 0, mode), "linear")
        return s.y
    if c["kind"] == "attention":
        H.check(L.ihip_enqueue_attention(h, s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(),
                                         s.y.data_ptr(), c["rows"], c["heads"], c["kv_heads"],
                                         c["head_dim"], c["past"], c["window"],
                                         s.sinks.data_ptr() if c["sinks"] else 0, 0.0,
                                         int(c["half"])), "attention")
        return s.y
    if c["kind"] == "experts":
        e, k, hid, f, t = c["experts"], c["used"], c["hidden"], c["ffn"], TYPES[c["type"]]
        gs, ds = f * H.row_bytes(t, hid), hid * H.row_bytes(t, f)
        ids = s.ids.data_ptr()
        H.check(L.ihip_enqueue_route(h, s.lg.data_ptr(), e, k, 1, ids, s.rw.data_ptr(), 0))
        H.check(L.ihip_enqueue_linear_ids(h, s.x.data_ptr(), hid, t, s.wg, gs, f, ids, k, 0,
                                          s.g.data_ptr(), 0, H.MODE_Q8))
        H.check(L.ihip_enqueue_linear_ids(h, s.x.data_ptr(), hid, t, s.wu, gs, f, ids, k, 0,
                                          s.u.data_ptr(), 0, H.MODE_Q8))
        H.check(L.ihip_enqueue_swiglu(h, s.g.data_ptr(), s.u.data_ptr(), k * f, 1.0, 0.0))
        H.check(L.ihip_enqueue_linear_ids(h, s.g.data_ptr(), f, t, s.wd, ds, hid, ids, k, 1,
                                          s.d.data_ptr(), 0, H.MODE_Q8))
        H.check(L.ihip_enqueue_moecombine(h, s.d.data_ptr(), s.rw.data_ptr(), s.y.data_ptr(), k,
                                          hid))
        return {"ids": s.ids, "weights": s.rw, "gated": s.g, "y": s.y}
    s.ctx.truncate(c["past"])
    if not c["steps"]:
        return {"logits": s.ctx.forward(s.ids)}
    toks = s.ctx.decode(s.ids[0], c["steps"])
    return {"tokens": toks, "logits": s.ctx.forward(toks[-1:])}


# -------------------------------------------------------------- work, tolerance
def work(case):
    c = case
    if c["kind"] == "linear":
        r, k, o = c["rows"], c["cols"], c["out"]
        return {"bytes": o * H.row_bytes(TYPES[c["type"]], k) + 4 * r * (k + o),
                "flops": 2.0 * r * k * o}
    if c["kind"] == "attention":
        r, hd = c["rows"], c["head_dim"]
        first = [c["past"] + i + 1 for i in range(r)]
        if c["window"]:
            first = [min(n, c["window"]) for n in first]
        keys = min(c["past"] + r, c["window"] + r - 1) if c["window"] else c["past"] + r
        kv = 2 * keys * c["kv_heads"] * hd * (2 if c["half"] else 4)
        return {"bytes": kv + 8 * r * c["heads"] * hd, "flops": 4.0 * sum(first) * c["heads"] * hd}
    if c["kind"] == "experts":
        k, h, f, t = c["used"], c["hidden"], c["ffn"], TYPES[c["type"]]
        return {"bytes": k * (2 * f * H.row_bytes(t, h) + h * H.row_bytes(t, f)) +
                4 * (c["experts"] + 2 * h + k * f), "flops": 6.0 * k * h * f}
    f, n, delta = FAMILIES[c["family"]], c["layers"], c["family"] == "delta"
    h, hd = f["hidden"], f["head_dim"]
    qw, kvw = f["heads"] * hd, f["kv_heads"] * hd
    base, more = (H.Q8_0, H.Q8_0) if delta else (H.Q4_K, H.Q6_K)
    steps = c["steps"] + 1 if c["steps"] else 1
    rows = 1 if c["steps"] else c["rows"]
    mats = []  # (type, out, in, of the rows: how many rows use it, copies read)
    for i in range(n):
        if delta and i % 2 == 0:
            d = f["lin_heads"] * f["lin_dim"]
            mats += [(base, 3 * d, h, rows, 1), (base, d, h, rows, 1), (base, h, d, rows, 1),
                     (base, 2 * f["lin_heads"], h, rows, 1)]
        else:
            mats += [(base, qw * (2 if delta else 1), h, rows, 1), (base, kvw, h, rows, 1),
                     (more, kvw, h, rows, 1), (base, h, qw, rows, 1)]
        if f["experts"]:
            k, fi = f["experts_used"], f["expert_ffn"]
            hit = min(f["experts"], rows * k)
            mats += [(H.F32, f["experts"], h, rows, 1), (base, 2 * fi, h, rows * k, hit),
                     (more, h, fi, rows * k, hit)]
        else:
            mats += [(base, 2 * f["ffn"], h, rows, 1), (more, h, f["ffn"], rows, 1)]
    nb = sum(m * o * H.row_bytes(t, k) for t, o, k, _, m in mats) + VOCAB * H.row_bytes(more, h)
    fl = sum(2.0 * o * k * r for _, o, k, r, _ in mats) + 2.0 * VOCAB * h
    if delta:
        fl += 8.0 * rows * f["lin_heads"] * f["lin_dim"] ** 2 * ((n + 1) // 2)
    attn = n // 2 if delta else n
    keys = c["past"] + (rows + 1) / 2 if not c["steps"] else c["past"] + steps / 2
    fl += attn * 4.0 * rows * keys * qw
    nb += attn * 4 * kvw * (c["past"] + rows)
    return {"bytes": steps * nb, "flops": steps * fl}


def tolerance(case):
    c = case
    if c["kind"] == "linear":
        # one rounding to single of an exact or double sum; the float mode
        # sums in single
        return {"rel": 2e-7} if c["mode"] == "q8" else {"rel": 2e-6}
    if c["kind"] == "attention":
        return {"rel": 3e-7}
    if c["kind"] == "experts":
        # a gated value at the edge of two activation codes of the down
        # projection moves one code
        return {"rel": 2e-3, "max": 2e-2}
    # a single rounding that moves one activation code moves about 1% of the
    # codes of the products after it: 0.8% to 1.6% of the logits between two
    # correct CPU implementations (sums in 64 bits, 512 rows of one or two
    # layers), 1e-7 where no code moves; a token of a near tie
    return {"rel": 0.03, "max": 0.5, "differ": 0.01}


# ---------------------------------------------------------------------- exact
def _rms(x, w, eps):
    x = x.double()
    n = (x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)).float()
    return n * torch.from_numpy(w).cuda()


def _rope(x, first, theta, dims):
    half = dims // 2
    e = torch.arange(half, device="cuda", dtype=torch.float64) * 2 / dims
    freq = 1.0 / torch.exp(math.log(theta) * e.float().double()).float()
    at = torch.arange(first, first + x.shape[0], device="cuda").float()
    ang = (at[:, None] * freq[None]).double()
    cos, sin = ang.cos().float().double()[:, None], ang.sin().float().double()[:, None]
    a, b = x[..., :half].double(), x[..., half:dims].double()
    return torch.cat([(a * cos - b * sin).float(), (b * cos + a * sin).float(), x[..., dims:]], -1)


class Exact:
    """The decoder's forward in 64 bits, rounded to single where a layer's
    operations meet, with its cached keys and values."""

    def __init__(self, d):
        self.d, self.n, self.kv = d, 0, {}

    def lin(self, x, key):
        a, name, out, cols = self.d.t[key]
        return linear64(x, a, name, out, cols).float()

    def w(self, key):
        return torch.from_numpy(self.d.t[key]).cuda()

    def attention(self, x, i):
        f, n = self.d.f, x.shape[0]
        hd, hs, kvh = f["head_dim"], f["heads"], f["kv_heads"]
        q, gate = self.lin(x, (i, "q")), None
        if "rope_dims" in f:
            q = q.reshape(n, hs, 2, hd)
            q, gate = q[:, :, 0], q[:, :, 1].reshape(n, -1)
        q = _rms(q.reshape(n, hs, hd), self.d.t[i, "q_norm"], f["eps"])
        k = _rms(self.lin(x, (i, "k")).reshape(n, kvh, hd), self.d.t[i, "k_norm"], f["eps"])
        v = self.lin(x, (i, "v")).reshape(n, kvh, hd).half()
        dims = f.get("rope_dims", hd)
        q, k = _rope(q, self.n, f["theta"], dims), _rope(k, self.n, f["theta"], dims).half()
        if i in self.kv:
            k, v = torch.cat([self.kv[i][0], k]), torch.cat([self.kv[i][1], v])
        self.kv[i] = (k, v)
        y = attention64(q, k, v, {}).float().reshape(n, -1)
        if gate is not None:
            y = y * torch.sigmoid(gate.double()).float()
        return self.lin(y, (i, "o"))

    def delta(self, x, i):
        f, n = self.d.f, x.shape[0]
        hs, dim, kw = f["lin_heads"], f["lin_dim"], f["conv"]
        qkv = self.lin(x, (i, "lin_qkv")).double()
        conv = self.w((i, "conv")).double()
        pad = torch.cat([qkv.new_zeros(kw - 1, qkv.shape[1]), qkv])
        y = sum(pad[j:j + n] * conv[:, j] for j in range(kw)).float()
        q, k, v = silu64(y).float().reshape(n, 3, hs, dim).unbind(1)

        def l2(t):
            t = t.double()
            return (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)).float()

        q, k, v = (l2(q) * dim ** -0.5).double(), l2(k).double(), v.double()
        beta = torch.sigmoid(self.lin(x, (i, "lin_b")).double())
        a = (self.lin(x, (i, "lin_a")) + self.w((i, "dt"))).double()
        decay = torch.exp(self.w((i, "neg_a")).double() * torch.nn.functional.softplus(a))
        z = silu64(self.lin(x, (i, "lin_z"))).float()
        st = qkv.new_zeros(hs, dim, dim)  # [head, value, key]
        out = qkv.new_empty(n, hs, dim)
        for t in range(n):
            st = st * decay[t][:, None, None]
            seen = (st @ k[t][:, :, None])[..., 0]
            st = st + ((v[t] - seen) * beta[t][:, None])[:, :, None] * k[t][:, None]
            out[t] = (st @ q[t][:, :, None])[..., 0]
        out = _rms(out.float(), self.d.t[i, "lin_norm"], f["eps"]).reshape(n, -1) * z
        return self.lin(out, (i, "lin_out"))

    def moe(self, x, i):
        f = self.d.f
        e, k, fi, h = f["experts"], f["experts_used"], f["expert_ffn"], f["hidden"]
        p = torch.softmax(self.lin(x, (i, "router")).double(), -1)
        pw, ids = p.topk(k)
        pw = pw.float()
        pw = (pw.double() / pw.double().sum(-1, keepdim=True)).float()
        y = torch.zeros_like(x)
        w = {n: self.d.t[i, n] for n in ("gate", "up", "down")}
        part = {n: w[n][0].reshape(e, -1, *w[n][0].shape[1:]) for n in w}
        for x_id in ids.unique().tolist():
            r, j = (ids == x_id).nonzero().unbind(1)
            g, u = (linear64(x[r], part[n][x_id], w[n][1], fi, h).float() for n in ("gate", "up"))
            o = linear64(silu64(g).float() * u, part["down"][x_id], w["down"][1], h, fi).float()
            y[r] += pw[r, j][:, None] * o
        return y

    def forward(self, ids):
        d, f = self.d, self.d.f
        a, name, _, cols = d.t["embed"]
        x = dense(a[np.asarray(ids)], name, len(ids), cols).float()
        for i in range(d.layers_n):
            hh = _rms(x, d.t[i, "input_norm"], f["eps"])
            x = x + (self.delta(hh, i) if (i, "lin_qkv") in d.t else self.attention(hh, i))
            hh = _rms(x, d.t[i, "post_norm"], f["eps"])
            if f["experts"]:
                x = x + self.moe(hh, i)
            else:
                g, u = self.lin(hh, (i, "gate")), self.lin(hh, (i, "up"))
                x = x + self.lin(silu64(g).float() * u, (i, "down"))
        self.n += len(ids)
        hh = _rms(x[-1:], d.t["final_norm"], f["eps"])
        return linear64(hh, a, name, VOCAB, cols)[0]


def exact(case, seed):
    c = case
    if c["kind"] == "linear":
        x, w = _linear_inputs(c, seed)
        return linear64(torch.from_numpy(x).cuda(), w, c["type"], c["out"], c["cols"], c["mode"])
    if c["kind"] == "attention":
        q, k, v, sinks = _attention_inputs(c, seed)
        return attention64(q, k, v, {"window": c["window"], "sinks": sinks})
    if c["kind"] == "experts":
        x, lg, wg, wu, wd = _experts_inputs(c, seed)
        e, k, h, f, t = c["experts"], c["used"], c["hidden"], c["ffn"], c["type"]
        x = torch.from_numpy(x).cuda()
        p, ids = torch.softmax(torch.from_numpy(lg).cuda().double(), -1).topk(k)
        ids, order = ids.sort()
        p = p[order].float().double()
        p = p / p.sum()

        def part(a, i, n):
            return a.reshape(e, n, *a.shape[1:])[i]

        y, gated = torch.zeros(h, dtype=torch.float64, device="cuda"), []
        for j, i in enumerate(ids.tolist()):
            g = linear64(x, part(wg, i, f), t, f, h).float()
            u = linear64(x, part(wu, i, f), t, f, h).float()
            gated.append(silu64(g) * u)
            y += p[j] * linear64(gated[-1].float(), part(wd, i, h), t, h, f)[0]
        return {"ids": ids.int(), "weights": p, "gated": torch.cat(gated), "y": y}
    past, ids = _tokens(c, seed)
    m = Exact(_decoder(c)[0])
    if c["past"]:
        m.forward(past)
    if not c["steps"]:
        return {"logits": m.forward(ids)}
    toks, at = [], ids[0]
    for _ in range(c["steps"]):
        at = int(m.forward([at]).argmax())
        toks.append(at)
    return {"tokens": np.array(toks, np.int32), "logits": m.forward(toks[-1:])}
