"""Representative calls of the framework for timing: what a diffusion-transformer step and a token of text generation
ask of it, each through the public entry point that a program calls, with inputs drawn from a seed.

A case is a dict with a "kind" (attention, linear, w4a8, w4a4, norm, block, decode, logits) and its sizes. `listed()`
holds the cases that are quoted; `draw(rng)` gives more of the same ranges. `prepare` builds on the GPU what a program
has in hand, `run` is one pass, `exact` the same values in 64 bits with the quantizers' and norms' defined rounding
points kept (they are part of what the calls compute).
"""
import math
import sys
import types

import torch

import __graft_entry__

__graft_entry__.load_package()
from comfyui_rdna2_attention_amd import attention, hip_attention, int8_gemm, int8_gemv, rms_norm  # noqa: E402

DEV = "cuda"
HEAD = 128


# ------------------------------------------------------------------------------------------------------------ the cases

def listed():
    return [
        # One self-attention of the DiT over 4096 latent tokens (the configuration bench.py quotes).
        dict(name="attention-4096", kind="attention", batch=1, heads=24, kv_heads=24, q_len=4096, k_len=4096, int8_qk=False),
        # The same layer at 512 x 512: 1024 image tokens and 77 text tokens in one ragged sequence.
        dict(name="attention-1101", kind="attention", batch=1, heads=24, kv_heads=24, q_len=1101, k_len=1101, int8_qk=False),
        # The longest sequence (1536 x 1536 and text) with int8 scores and grouped KV heads.
        dict(name="attention-i8-9293", kind="attention", batch=1, heads=24, kv_heads=8, q_len=9293, k_len=9293, int8_qk=True),
        # A projection of the DiT at hidden 3072: ConvRot, per-token int8, int8 GEMM.
        dict(name="linear-4096", kind="linear", rows=4096, k=3072, n=3072, act="rotate", group=256, bias=False, tokens=0),
        # The fewest rows the hooks send to the int8 kernels (a prompt's tokens), with a bias.
        dict(name="linear-512", kind="linear", rows=512, k=3072, n=3072, act="rotate", group=256, bias=True, tokens=0),
        # The MLP's down projection at 512 x 512 and text: SwiGLU before the rotation, gated residual after the GEMM.
        dict(name="mlp-down-1101", kind="linear", rows=1101, k=8192, n=3072, act="swiglu", group=256, bias=False, tokens=1101),
        # W4A8 with group scales: the widening projection of an MLP.
        dict(name="w4a8-4096", kind="w4a8", rows=4096, k=3072, n=12288, bias=False),
        # W4A4 as the int4 loader's hook runs it, two images at 512 x 512 and text.
        dict(name="w4a4-2202", kind="w4a4", rows=2202, k=3072, n=8192),
        # The fused RMSNorm of the DiT's smallest sequence: the smallest call, bound by its launch.
        dict(name="norm-1101", kind="norm", batch=1, tokens=1101, dim=3072, heads=0),
        # A whole fused Krea 2 block, the unit a diffusion step repeats.
        dict(name="block-4096", kind="block", tokens=4096, heads=24, hidden=8192, int8_qk=False),
        # One token through one text-encoder layer (seven int8 linears and decode attention), replayed from a graph as
        # the generation loop does.
        dict(name="decode-layer-2048", kind="decode", dim=4096, heads=32, kv_heads=8, hidden=12288, cache=2048, length=2048),
        # The logits of a token against the bf16 embedding table.
        dict(name="logits-131072", kind="logits", n=131072, k=4096),
    ]


def _log(rng, lo, hi, multiple=1):
    """A size spread over the logarithm of [lo, hi], in whole multiples."""
    return max(-(-lo // multiple), min(hi // multiple, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / multiple))) * multiple


def draw(rng):
    kind = rng.choice(["attention", "attention", "linear", "linear", "linear", "w4a8", "w4a4", "norm", "block", "decode", "logits"])
    if kind == "attention":
        kv = rng.choice([1, 2, 4, 8, 24])
        heads = 24 if kv == 24 else kv * rng.choice([1, 2, 3, 4])
        q_len = _log(rng, 256, 9000)
        batch = 2 if q_len < 2500 and rng.random() < 0.4 else 1  # 2: a classifier-free-guidance pair
        k_len = q_len if rng.random() < 0.75 else _log(rng, 64, 2000)  # otherwise: text that the image attends to
        return dict(kind=kind, batch=batch, heads=heads, kv_heads=kv, q_len=q_len, k_len=k_len, int8_qk=rng.random() < 0.4)
    if kind == "linear":
        act = rng.choice(["rotate", "rotate", "none", "swiglu", "gate"])
        rows = _log(rng, 64, 8192)
        return dict(kind=kind, rows=rows, k=_log(rng, 1024, 12288, 256), n=_log(rng, 512, 12288 if rows < 4096 else 6144, 64), act=act,
                    group=rng.choice([256, 256, 128]), bias=rng.random() < 0.3, tokens=rows if rng.random() < 0.3 else 0)
    if kind == "w4a8":
        rows = _log(rng, 64, 6000)
        return dict(kind=kind, rows=rows, k=_log(rng, 1024, 12288, 256), n=_log(rng, 512, 12288 if rows < 3000 else 4096, 128), bias=rng.random() < 0.3)
    if kind == "w4a4":
        return dict(kind=kind, rows=_log(rng, 512, 6000), k=_log(rng, 1024, 8192, 256), n=_log(rng, 512, 8192, 64))
    if kind == "norm":
        heads = rng.choice([0, 0, 8, 24])  # 0: rows of the hidden size; otherwise QK-norm and RoPE over heads of 128
        return dict(kind=kind, batch=rng.choice([1, 1, 2]), tokens=_log(rng, 64, 9000), dim=heads * HEAD or _log(rng, 512, 8192, 8), heads=heads)
    if kind == "block":
        heads = rng.choice([8, 12, 16, 24])
        return dict(kind=kind, tokens=_log(rng, 512, 4096), heads=heads, hidden=_log(rng, heads * HEAD, 8192, 256), int8_qk=rng.random() < 0.5)
    if kind == "decode":
        kv = rng.choice([2, 4, 8])
        cache = _log(rng, 256, 8192, 64)
        return dict(kind=kind, dim=rng.choice([1024, 2048, 2560, 4096, 5120]), heads=kv * 4, kv_heads=kv, hidden=_log(rng, 3072, 13824, 512), cache=cache,
                    length=rng.randint(cache // 4, cache))
    return dict(kind=kind, n=_log(rng, 32000, 152064, 16), k=_log(rng, 1024, 4096, 256))


# ---------------------------------------------------------------------------------------------- inputs, from a seed alone

class _Draws:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device=DEV) * std).to(dtype)

    def activations(self, rows, k):
        """fp16 ~N(0, 1) with eight outlier channels x 30, as the activations of these models have."""
        x = self.normal(rows, k)
        x[:, torch.randperm(k, generator=self.g, device=DEV)[:8]] *= 30
        return x.half()

    def codes(self, n, k):
        return torch.randint(-127, 128, (n, k), generator=self.g, device=DEV, dtype=torch.int8)

    def packed(self, n, k):
        return torch.randint(0, 256, (n, k // 2), generator=self.g, device=DEV, dtype=torch.uint8)

    def scales(self, n, typical):
        return (0.5 + torch.rand(n, generator=self.g, device=DEV)) * typical


def _freqs(d, tokens):
    ang = d.normal(1, 1, tokens, 64)
    return torch.stack([torch.cos(ang), -torch.sin(ang), torch.sin(ang), torch.cos(ang)], -1).reshape(1, 1, tokens, 64, 2, 2).contiguous()


def _attention(c, d):
    B, H, Hkv = c["batch"], c["heads"], c["kv_heads"]
    if H == Hkv:  # what a model's projections give the backend: (B, L, H 128)
        return [d.normal(B, c[n], H * HEAD, dtype=torch.float16) for n in ("q_len", "k_len", "k_len")]
    # grouped KV heads: head views of the projections, as the block passes them
    return [d.normal(B, c[n], h, HEAD, dtype=torch.float16).transpose(1, 2) for n, h in (("q_len", H), ("k_len", Hkv), ("k_len", Hkv))]


def _linear(c, d):
    M, K, N = c["rows"], c["k"], c["n"]
    s = dict(x=d.activations(M, K), up=None, gate=None, w=d.codes(N, K), ws=d.scales(N, 1 / (73 * K ** 0.5)), bias=None, res=None)
    if c["act"] == "swiglu":
        s["x"], s["up"] = d.normal(M, K, dtype=torch.float16), d.normal(M, K, dtype=torch.float16)
    elif c["act"] == "gate":
        s["gate"] = d.normal(M, K, dtype=torch.float16)
    if c["bias"]:
        s["bias"] = d.normal(N, std=0.1, dtype=torch.float16)
    if c["tokens"]:
        B = M // c["tokens"]
        s["res"] = d.normal(B, c["tokens"], N, dtype=torch.float16), d.normal(B, N, std=0.3, dtype=torch.float16)
    return s


def _w4a8(c, d):
    M, K, N = c["rows"], c["k"], c["n"]
    return dict(x=d.activations(M, K), w=d.packed(N, K), gs=d.scales(N * K // 128, 1 / (4.6 * K ** 0.5)).reshape(N, K // 128).half(),
                bias=d.normal(N, std=0.1, dtype=torch.float16) if c["bias"] else None)


def _w4a4(c, d):
    M, K, N = c["rows"], c["k"], c["n"]
    return dict(x=d.activations(M, K), w=d.packed(N, K), ws=d.scales(N, 1 / (4.6 * K ** 0.5)))


class _Norm:
    def __init__(self, scale, eps=1e-6):
        self.scale, self.eps = scale, eps


def _norm(c, d):
    D = HEAD if c["heads"] else c["dim"]
    return dict(x=d.normal(c["batch"], c["tokens"], c["dim"], dtype=torch.float16), norm=_Norm(d.normal(D, std=0.1)),
                freqs=_freqs(d, c["tokens"]) if c["heads"] else None)


# ------------------------------------------------ the int8 layers of the plugin that the block's hooks are installed into

class _Int8Linear:
    """An int8 ConvRot layer: its forward rotates, then calls the plugin's int8 linear; both are looked up at call time,
    so that the framework's hooks take effect."""
    _is_quantized = _use_convrot = True
    _convrot_groupsize = 256
    bias = None
    lora_patches = ()

    def __init__(self, w, ws):
        self.weight, self.weight_scale = w, ws
        self.out_features, self.in_features = w.shape

    def forward(self, x):
        x = sys.modules["perf_plugin.convrot"].rotate_activation(x, None, self._convrot_groupsize)
        return sys.modules["perf_plugin.int8_quant"].triton_int8_linear(x, self.weight, self.weight_scale, self.bias, torch.float16)

    def __call__(self, x):
        return self.forward(x)


def _plugin():
    """The modules of a program with the int8 plugin loaded, and the framework's hooks installed into them."""
    if "perf_plugin.int8_quant" in sys.modules:
        return
    quant, convrot, ops = types.ModuleType("perf_plugin.int8_quant"), types.ModuleType("perf_plugin.convrot"), types.ModuleType("comfy.ops")

    def missing(*args, **kwargs):
        raise RuntimeError("a hooked call reached the plugin's own function")

    quant.triton_int8_linear = quant.triton_int8_linear_per_row = missing
    quant._TRITON_AVAILABLE = True
    quant.Int8TensorwiseOps = types.SimpleNamespace(Linear=_Int8Linear)
    convrot.rotate_activation = convrot.build_hadamard = ops.linear_input_act = ops._eager_input_act = missing
    sys.modules["perf_plugin.int8_quant"], sys.modules["perf_plugin.convrot"] = quant, convrot
    cast = types.SimpleNamespace(cast_to=lambda t, dtype=None, device=None: t.to(dtype=dtype, device=device))
    int8_gemm.comfy = rms_norm.comfy = types.SimpleNamespace(ops=ops, model_management=cast)
    int8_gemm.enable(True)


def _block(c, d):
    D, F, L = c["heads"] * HEAD, c["hidden"], c["tokens"]
    layer = lambda k, n: _Int8Linear(d.codes(n, k), d.scales(n, 1 / (73 * k ** 0.5)))  # noqa: E731
    norm = lambda n: _Norm(d.normal(n, std=0.1))  # noqa: E731
    attn = types.SimpleNamespace(heads=c["heads"], kvheads=c["heads"], headdim=HEAD, wq=layer(D, D), wk=layer(D, D), wv=layer(D, D), gate=layer(D, D),
                                 wo=layer(D, D), qknorm=types.SimpleNamespace(qnorm=norm(HEAD), knorm=norm(HEAD)))
    mlp = types.SimpleNamespace(gate=layer(D, F), up=layer(D, F), down=layer(F, D))
    mods = tuple(d.normal(1, 1, D, std=0.2, dtype=torch.float16) for _ in range(6))
    module = types.SimpleNamespace(attn=attn, mlp=mlp, prenorm=norm(D), postnorm=norm(D), mod=lambda vec: mods)
    return dict(module=module, mods=mods, x=d.normal(1, L, D, dtype=torch.float16), freqs=_freqs(d, L))


# --------------------------------------------------------------------------------------- a text-generation layer, one token

class _Weight:
    def __init__(self, w, s):
        self._qdata, self._params = w, types.SimpleNamespace(scale=s)


class _Layer:
    weight_function = bias_function = ()

    def __init__(self, w, s):
        self.value = _Weight(w, s)


class _Cast:
    """The program's weight context: a layer's weight is on the GPU already."""

    def __init__(self, module, **kwargs):
        self.module = module

    def __enter__(self):
        return self.module.value, None

    def __exit__(self, *exc):
        return False


def _decode_shapes(c):
    D, F, q, kv = c["dim"], c["hidden"], c["heads"] * HEAD, c["kv_heads"] * HEAD
    return {"q": (q, D), "k": (kv, D), "v": (kv, D), "o": (D, q), "gate": (F, D), "up": (F, D), "down": (D, F)}


def _decode_inputs(c, d):
    shapes = _decode_shapes(c)
    s = {n: (d.codes(*nk), d.scales(nk[0], 1 / (73 * nk[1] ** 0.5))) for n, nk in shapes.items()}
    cache = lambda: d.normal(1, c["cache"], c["kv_heads"], HEAD)  # noqa: E731
    return dict(weights=s, k=cache(), v=cache(), x=d.normal(1, 1, c["dim"]), lengths=torch.tensor([c["length"]], dtype=torch.int32, device=DEV))


def _decode_step(c, s):
    """The int8 linears and the attention of one layer, as the patched forwards run them (the layer's own norms, rope and
    element-wise ops are torch's and are left out)."""
    shapes, mods, x = _decode_shapes(c), s["mods"], s["x"]
    lin = lambda name, inp: int8_gemv.linear_forward(mods[name], *shapes[name], torch.int8, 256, inp)  # noqa: E731
    q, k, v = lin("q", x), lin("k", x), lin("v", x)
    o = int8_gemv.attention_decode(q.view(1, 1, c["heads"], HEAD), s["k"], s["v"], s["lengths"])
    h = lin("o", o.view(1, 1, -1))
    gate, up = lin("gate", h), lin("up", h)
    return [q, k, v, o, h, gate, up, lin("down", gate)]


def _decode(c, d):
    int8_gemv.comfy = types.SimpleNamespace(ops=types.SimpleNamespace(CastBiasWeightContext=_Cast))
    s, shapes = _decode_inputs(c, d), _decode_shapes(c)
    s["mods"] = {n: _Layer(*ws) for n, ws in s.pop("weights").items()}
    for names in (("q", "k", "v"), ("gate", "up")):
        if c["dim"] <= int8_gemv.MULTI_MAX_K:
            int8_gemv.register_siblings([(s["mods"][n], *shapes[n], torch.int8, 256) for n in names])
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        _decode_step(c, s)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"], stream=stream):
            s["out"] = _decode_step(c, s)
    torch.cuda.current_stream().wait_stream(stream)
    return s


def _logits(c, d):
    return dict(x=d.normal(1, 1, c["k"]), w=d.normal(c["n"], c["k"], std=c["k"] ** -0.5, dtype=torch.bfloat16))


MAKE = dict(attention=_attention, linear=_linear, w4a8=_w4a8, w4a4=_w4a4, norm=_norm, block=_block, decode=_decode, logits=_logits)


def prepare(case, seed):
    if case["kind"] == "block":
        _plugin()
    return case, MAKE[case["kind"]](case, _Draws(seed))


# ------------------------------------------------------------------------------------------------------------- one pass

def run(state):
    c, s = state
    kind = c["kind"]
    if kind == "attention":
        if c["heads"] == c["kv_heads"]:
            return (attention.attention_hip_int8 if c["int8_qk"] else attention.attention_hip)(*s, c["heads"])
        out = torch.empty(c["batch"], c["q_len"], c["heads"], HEAD, dtype=torch.float16, device=DEV).transpose(1, 2)
        hip_attention.attention(*s, out, HEAD ** -0.5, c["int8_qk"])
        return out
    if kind == "linear":
        return int8_gemm.linear(s["x"], s["w"], s["ws"], s["bias"], rotate=c["act"] == "rotate", up=s["up"], gate=s["gate"], res=s["res"], group=c["group"])
    if kind == "w4a8":
        return int8_gemm.linear_w4a8(s["x"], s["w"], s["gs"], s["bias"])
    if kind == "w4a4":
        k = int8_gemm.get_kernels()
        return int8_gemm.run(k.rot_quant_pack_a_i4, k.gemm_i4, s["x"], s["w"], s["ws"], None, c["k"])
    if kind == "norm":
        if c["heads"]:
            return rms_norm.rms_norm_rope(s["x"], c["heads"], s["norm"], s["freqs"])
        return rms_norm.rms_norm(s["x"], s["norm"].scale, s["norm"].eps)
    if kind == "block":
        return int8_gemm.block_forward(s["module"], c["int8_qk"], s["x"], None, s["freqs"])
    if kind == "decode":
        s["graph"].replay()
        return s["out"]
    return int8_gemv.logits_gemv(s["x"], s["w"])


# ------------------------------------------------------------------------------------------- what a pass cannot do without

def _product(M, N, K, weight_bytes):
    return 2.0 * M * N * K, M * K * 2 + weight_bytes + M * N * 2


def work(case):
    c, kind = case, case["kind"]
    if kind == "attention":
        B, H, q, k = c["batch"], c["heads"], c["q_len"], c["k_len"]
        return {"bytes": 2 * HEAD * B * (2 * H * q + 2 * c["kv_heads"] * k), "flops": 4.0 * B * H * q * k * HEAD}
    if kind in ("linear", "w4a8", "w4a4"):
        M, K, N = c["rows"], c["k"], c["n"]
        flops, nbytes = _product(M, N, K, {"linear": N * K + 4 * N, "w4a8": N * K // 2 + N * K // 64, "w4a4": N * K // 2 + 4 * N}[kind])
        if kind == "linear":
            nbytes += (M * K * 2 if c["act"] in ("swiglu", "gate") else 0) + (M * N * 2 if c["tokens"] else 0)
        return {"bytes": nbytes, "flops": flops}
    if kind == "norm":
        return {"bytes": 4 * c["batch"] * c["tokens"] * c["dim"] + (c["tokens"] * 1024 if c["heads"] else 4 * c["dim"]), "flops": 0}
    if kind == "block":
        L, D, F = c["tokens"], c["heads"] * HEAD, c["hidden"]
        return {"bytes": 4 * L * D + 5 * D * D + 3 * D * F + L * 1024, "flops": 2.0 * L * D * (5 * D + 3 * F) + 4.0 * L * L * D}
    if kind == "decode":
        params = sum(n * k for n, k in _decode_shapes(c).values())
        cache = 2 * c["length"] * c["kv_heads"] * HEAD
        return {"bytes": params + 4 * cache, "flops": 2.0 * params + 8.0 * cache}
    return {"bytes": 2 * c["n"] * c["k"] + 4 * c["n"], "flops": 2.0 * c["n"] * c["k"]}


# Largest relative errors: about four times what `run` differs from `exact` by. fp16 results differ by their rounding
# (attention: P's as well); int4 activations (steps of a seventh of the row's largest value) and whole blocks by the codes
# that a last-bit difference ahead of a quantizer moves by one; decode and logits are fp32 sums and results.
TOLERANCE = dict(attention=1.6e-3, linear=1e-3, w4a8=1e-3, w4a4=8e-3, norm=1.2e-3, block=8e-3, decode=4e-6, logits=1e-6)


def tolerance(case):
    return {"rel": TOLERANCE[case["kind"]]}


# ----------------------------------------------------------------------------------------------------- the same in 64 bits

def _h(x):
    """One of the defined roundings to fp16."""
    return x.half().double()


def _hadamard(group):
    h4 = torch.ones(4, 4, dtype=torch.float64, device=DEV) - 2 * torch.eye(4, dtype=torch.float64, device=DEV).flip(0)
    h, n = torch.ones(1, 1, dtype=torch.float64, device=DEV), group
    while n >= 4:
        h, n = torch.kron(h4, h), n // 4
    if n == 2:
        h = torch.kron(torch.tensor([[1.0, 1.0], [1.0, -1.0]], dtype=torch.float64, device=DEV), h)
    return h / group ** 0.5


def _rotate(x, group):
    return (x.reshape(-1, group) @ _hadamard(group).T).reshape(x.shape)


def _quant(x, group=0, int4=False):
    """Codes and scales of rows x (64 bits): rotated and rounded to fp16 where group is given."""
    if group:
        x = _h(_rotate(x, group))
    top = x.abs().amax(1, keepdim=True)
    if int4:
        s = top.clamp(min=1e-10) / 7
        return torch.round(x / s).clamp(-7, 7), s
    s = (top / 127).clamp(min=1e-30)
    return torch.floor(x / s + 0.5).clamp(-128, 127), s


def _act(x, act, other):
    if act == "swiglu":
        x = x.double()
        return _h(_h(x * torch.sigmoid(x)) * other.double())
    if act == "gate":
        return _h(x.double() * _h(torch.sigmoid(other.double())))
    return x.double()


def _int8_out(codes, s, w, ws, bias=None, res=None):
    y = (codes @ w.double().T) * s * ws.double()
    if bias is not None:
        y = y + bias.double()
    if res is None:
        return y
    r, g = res[0].double().reshape(y.shape), res[1].double()
    return r + _h(g.reshape(-1, 1, y.shape[1]) * _h(y).reshape(g.reshape(-1, y.shape[1]).shape[0], -1, y.shape[1])).reshape(y.shape)


def _softmax_rows(q, k, v, scale):
    """softmax(q k^T scale) v of one head, some rows at a time."""
    return torch.cat([torch.softmax((p @ k.T) * scale, -1) @ v for p in q.split(2048)])


def _heads(q, k, v, int8_qk):
    """Attention of (B, H, L, 128) tensors; int8_qk: q and k rounded per row to 127 steps of their largest value."""
    if int8_qk:
        step = lambda t: (t.double().abs().amax(-1, keepdim=True) / 127).clamp(min=1e-30)  # noqa: E731
        q, k = (torch.round(t.double() / step(t)) * step(t) for t in (q, k))
    rep = q.shape[1] // k.shape[1]
    out = [[_softmax_rows(q[b, h].double(), k[b, h // rep].double(), v[b, h // rep].double(), HEAD ** -0.5) for h in range(q.shape[1])]
           for b in range(q.shape[0])]
    return torch.stack([torch.stack(o) for o in out])


def _rms(x, w, eps):
    x = x.double()
    return _h(x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * (w.double() + 1))


def _rope(x, freqs):
    """x (B, H, L, 128); freqs (1, 1, L, 64, 2, 2)."""
    p, f = x.reshape(*x.shape[:-1], 64, 2), freqs.double()
    return torch.stack([(f[..., i, :] * p).sum(-1) for i in range(2)], -1).reshape(x.shape)


def _exact_block(c, s):
    m, x = s["module"], s["x"][0].double()
    a, p, L = m.attn, m.mlp, c["tokens"]
    pre_s, pre_t, pre_g, post_s, post_t, post_g = (t.reshape(-1) for t in s["mods"])

    def mod(rows, norm, scale, shift):
        return _quant(_h(_h(_rms(rows, norm.scale, norm.eps) * (1 + scale).double()) + shift.double()), 256)

    def lin(q, layer, res=None):
        return _h(_int8_out(*q, layer.weight, layer.weight_scale, res=res))

    q8 = mod(x, m.prenorm, pre_s, pre_t)
    q, k, v = (lin(q8, layer).reshape(1, L, c["heads"], HEAD).transpose(1, 2) for layer in (a.wq, a.wk, a.wv))
    gate = lin(q8, a.gate)
    q, k = (_h(_rope(_rms(t, n.scale, n.eps), s["freqs"])) for t, n in ((q, a.qknorm.qnorm), (k, a.qknorm.knorm)))
    o = _h(_heads(q, k, v, c["int8_qk"])).transpose(1, 2).reshape(L, -1)
    x = lin(_quant(_act(o, "gate", gate), 256), a.wo, (x, pre_g))
    q8 = mod(x, m.postnorm, post_s, post_t)
    return lin(_quant(_act(lin(q8, p.gate), "swiglu", lin(q8, p.up)), 256), p.down, (x, post_g))[None]


def _exact_decode(c, s):
    def lin(name, x):
        w, ws = s["weights"][name]
        return (_rotate(x.reshape(1, -1), 256) @ w.double().T * ws.double()).reshape(1, 1, -1)

    x, n = s["x"].double(), c["length"]
    q, k, v = lin("q", x), lin("k", x), lin("v", x)
    kc, vc = (t[:, :n].transpose(1, 2) for t in (s["k"], s["v"]))
    o = _heads(q.view(1, 1, c["heads"], HEAD).transpose(1, 2), kc, vc, False).transpose(1, 2)
    h = lin("o", o)
    gate, up = lin("gate", h), lin("up", h)
    return [q, k, v, o, h, gate, up, lin("down", gate)]


def exact(case, seed):
    c, d, kind = case, _Draws(seed), case["kind"]
    if kind == "decode":
        return _exact_decode(c, _decode_inputs(c, d))
    s = MAKE[kind](c, d)
    if kind == "attention":
        if c["heads"] == c["kv_heads"]:
            o = _heads(*(t.reshape(c["batch"], -1, c["heads"], HEAD).transpose(1, 2) for t in s), c["int8_qk"])
            return o.transpose(1, 2).reshape(c["batch"], c["q_len"], -1)
        return _heads(*s, c["int8_qk"])
    if kind == "linear":
        x = _act(s["x"], c["act"], s["up"] if c["act"] == "swiglu" else s["gate"])
        return _int8_out(*_quant(x, 0 if c["act"] == "none" else c["group"]), s["w"], s["ws"], s["bias"], s["res"])
    if kind in ("w4a8", "w4a4"):
        # signed nibbles, the low one first
        w = torch.stack([s["w"] & 15, s["w"] >> 4], -1).reshape(c["n"], c["k"]).to(torch.int8)
        w = torch.where(w > 7, w - 16, w)
        if kind == "w4a4":
            return _int8_out(*_quant(s["x"].double(), 256, int4=True), w, s["ws"])
        codes, scale = _quant(s["x"].double(), 256)
        y = (codes @ (w.double().reshape(c["n"], -1, 128) * s["gs"].double()[..., None]).reshape(c["n"], -1).T) * scale
        return y if s["bias"] is None else y + s["bias"].double()
    if kind == "norm":
        if not c["heads"]:
            x = s["x"].double()
            return x / torch.sqrt(x.square().mean(-1, keepdim=True) + s["norm"].eps) * (s["norm"].scale.double() + 1)
        x = s["x"].reshape(c["batch"], c["tokens"], c["heads"], HEAD).transpose(1, 2)
        return _rope(_rms(x, s["norm"].scale, s["norm"].eps), s["freqs"])
    if kind == "block":
        return _exact_block(c, s)
    return (s["w"].double() @ s["x"].double().reshape(-1)).reshape(1, 1, -1)
