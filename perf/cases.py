"""The workloads this framework is timed on: the NF4 + LoRA blocks of a decoder layer.

Every case goes through an entry point that a program calls: `Linear4bit` and `LoraLinear4bit`
modules, the attention's `project_qkv` with the rotation that follows it, the `MLP` module,
`unpack_nf4` and `quantize_4bit`.  Shapes are the Qwen2.5-1.5B projections (hidden 1536,
intermediate 8960, 12 query and 2 key/value heads of 128) and the other widths the tests use
(intermediate 6144, 11008, 14336; hidden 4096).  Token counts run from one generated token to
8192 packed training tokens; a training pass is one forward and one backward with the gradients
of the input and of every LoRA weight.
"""

import math
import types

import torch

import mindxsoup_amd
from mindxsoup_amd import attention, linear4bit, mlp, nf4, quant, rope

# The package's own modules are used, so there is no transformers model to patch.
mindxsoup_amd.FEATURES.update(mlp_fp16=False, attention_fp16=False)
mindxsoup_amd.apply()

HEAD = 128
SCALING = 2.0  # lora_alpha / r


def listed():
    return [
        # one token of greedy generation through a frozen q_proj (no adapter on this layer)
        dict(name="linear_decode_1", kind="linear", tokens=1, k=1536, n=1536, bias=True,
             train=False),
        # a generation step of a small batch through an MLP with its adapters attached
        dict(name="mlp_decode_4", kind="mlp", tokens=4, hidden=1536, inter=8960, r=16,
             drop=0.0, train=False),
        # evaluation or prefill of one short prompt
        dict(name="mlp_prefill_300", kind="mlp", tokens=300, hidden=1536, inter=8960, r=16,
             drop=0.0, train=False),
        # the training step's attention projections at the benchmark's 1024 packed tokens
        dict(name="qkv_train_1024", kind="qkv", tokens=1024, seqs=1, hidden=1536, heads=12,
             kv_heads=2, r=16, drop=0.05, train=True),
        # o_proj of a ragged micro-batch
        dict(name="o_train_830", kind="lora", tokens=830, k=1536, n=1536, bias=False, r=16,
             drop=0.05, train=True),
        # the training step's MLP at the benchmark's 1024 packed tokens
        dict(name="mlp_train_1024", kind="mlp", tokens=1024, hidden=1536, inter=8960, r=16,
             drop=0.05, train=True),
        # a ragged packed batch
        dict(name="mlp_train_3001", kind="mlp", tokens=3001, hidden=1536, inter=8960, r=16,
             drop=0.05, train=True),
        # adapters on the attention only: a frozen MLP weight still passes gradients through
        dict(name="frozen_train_2048", kind="linear", tokens=2048, k=1536, n=8960, bias=False,
             train=True),
        # long packed batches, as a card with much memory is fed
        dict(name="qkv_train_8192", kind="qkv", tokens=8192, seqs=4, hidden=1536, heads=12,
             kv_heads=2, r=16, drop=0.05, train=True),
        dict(name="mlp_train_8192", kind="mlp", tokens=8192, hidden=1536, inter=8960, r=16,
             drop=0.05, train=True),
        # a dense copy of one weight (merging adapters, exporting a layer)
        dict(name="unpack_gate", kind="unpack", n=8960, k=1536, dtype="float16"),
        # a checkpoint's weight brought onto the path at load time
        dict(name="quantize_down", kind="quantize", n=1536, k=8960),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "lora", "lora", "qkv", "qkv", "mlp", "mlp", "mlp",
                       "unpack", "quantize"])
    rank = rng.choice([16, 16, 16, 32, 64])
    drop = rng.choice([0.0, 0.05, 0.05, 0.1])
    shapes = [(1536, 1536), (256, 1536), (8960, 1536), (1536, 8960), (6144, 1536), (4096, 4096),
              (11008, 4096), (4096, 14336)]
    train = rng.random() < 0.65
    if kind in ("linear", "lora"):
        n, k = rng.choice(shapes)
        tokens = _log_int(rng, 8, 4096) if train else _log_int(rng, 1, 1024)
        case = dict(kind=kind, tokens=tokens, k=k, n=n, bias=rng.random() < 0.5, train=train)
        if kind == "lora":
            case.update(r=rank, drop=drop if train else 0.0)
    elif kind == "qkv":
        hidden, heads, kv = rng.choice([(1536, 12, 2), (1536, 12, 2), (2048, 16, 2),
                                        (4096, 32, 8)])
        seqs = rng.choice([1, 1, 2, 4])
        t = max(1, (_log_int(rng, 16, 4096) if train else _log_int(rng, 1, 1024)) // seqs)
        case = dict(kind=kind, tokens=t * seqs, seqs=seqs, hidden=hidden, heads=heads,
                    kv_heads=kv, r=rank, drop=drop if train else 0.0, train=train)
    elif kind == "mlp":
        hidden, inter = rng.choice([(1536, 8960), (1536, 8960), (1536, 6144), (4096, 11008)])
        most = (8192 if rank == 16 else 4096) if hidden == 1536 else 2048
        tokens = _log_int(rng, 16, most) if train else _log_int(rng, 1, 1024)
        case = dict(kind=kind, tokens=tokens, hidden=hidden, inter=inter, r=rank,
                    drop=drop if train else 0.0, train=train)
    elif kind == "unpack":
        n, k = rng.choice(shapes + [(100, 64), (1111, 1472)])
        case = dict(kind=kind, n=n, k=k, dtype=rng.choice(["float16", "float16", "float32"]))
    else:
        n, k = rng.choice(shapes + [(100, 64), (1111, 1472)])
        case = dict(kind=kind, n=n, k=k)
    return case


# ---- inputs --------------------------------------------------------------------------------

class _Rng:
    """Normal and uniform draws on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float16):
        return (torch.randn(shape, device="cuda", generator=self.g) * std).to(dtype)

    def uniform(self, *shape):
        return torch.rand(shape, device="cuda", generator=self.g)


def _layer(g, n, k, bias):
    """A Linear4bit quantized from an N(0, 0.02) weight."""
    return linear4bit.Linear4bit.from_weight(g.normal(n, k, std=0.02),
                                             g.normal(n, std=0.1) if bias else None)


def _lora(g, n, k, case, bias=False):
    """A LoRA layer (fp32 adapter weights, as peft keeps them) over a Linear4bit, with a trained
    (nonzero) B and, for a training pass with dropout, its keep mask."""
    layer = linear4bit.LoraLinear4bit(_layer(g, n, k, bias), r=case["r"],
                                      lora_alpha=SCALING * case["r"],
                                      lora_dropout=case["drop"])
    a, b = layer.lora_A["default"].weight, layer.lora_B["default"].weight
    a.data = (g.uniform(case["r"], k) * 2 - 1) / math.sqrt(k)
    b.data = g.normal(n, case["r"], std=0.01, dtype=torch.float32)
    layer.train(case["train"])
    keep = None
    if case["train"] and case["drop"] > 0:
        keep = (g.uniform(case["tokens"], k) >= case["drop"]).to(torch.uint8)
    return layer, keep


def _params(layers):
    return [p for lyr in layers
            for p in (lyr.lora_A["default"].weight, lyr.lora_B["default"].weight)]


def prepare(case, seed):
    g = _Rng(seed)
    kind = case["kind"]
    s = types.SimpleNamespace(case=case)
    if kind in ("unpack", "quantize"):
        w = g.normal(case["n"], case["k"], std=0.02)
        if kind == "quantize":
            s.w = w
        else:
            s.packed, s.state = quant.quantize_4bit(w)
            s.dtype = getattr(torch, case["dtype"])
        return s
    m, train = case["tokens"], case["train"]
    dtype = torch.float16
    if kind == "linear":
        s.layers, s.keeps = [_layer(g, case["n"], case["k"], case["bias"])], []
        width, outs = case["k"], [case["n"]]
    elif kind == "lora":
        made = [_lora(g, case["n"], case["k"], case, case["bias"])]
        width, outs = case["k"], [case["n"]]
    elif kind == "qkv":
        h = case["hidden"]
        outs = [case["heads"] * HEAD, case["kv_heads"] * HEAD, case["kv_heads"] * HEAD]
        made = [_lora(g, n, h, case, True) for n in outs]
        width = h
    else:
        h, i = case["hidden"], case["inter"]
        made = [_lora(g, i, h, case), _lora(g, i, h, case), _lora(g, h, i, case)]
        width, outs = h, [h]
        if train:
            dtype = torch.float32  # the residual stream of a training step
    if kind != "linear":
        s.layers, s.keeps = [x[0] for x in made], [x[1] for x in made]
    if kind == "qkv":
        seqs = case["seqs"]
        t = m // seqs
        s.attn = types.SimpleNamespace(q_proj=s.layers[0], k_proj=s.layers[1],
                                       v_proj=s.layers[2])
        freq = 1e6 ** (-torch.arange(0, HEAD, 2, device="cuda").float() / HEAD)
        ang = torch.arange(t, device="cuda").float()[:, None] * freq
        ang = torch.cat((ang, ang), -1)[None]
        s.cos, s.sin = ang.cos(), ang.sin()
        shape = (seqs, t)
        # attention's gradients: fp16 [B, heads, T, 128] views of [B, T, heads, 128] memory
        s.dys = [g.normal(seqs, t, n // HEAD, HEAD, std=1e-3).transpose(1, 2) for n in outs]
    else:
        shape = (1, m) if kind == "mlp" else (m,)
        s.dys = [g.normal(*shape, n, std=1e-3, dtype=dtype) for n in outs]
    if kind == "mlp":
        s.module = mlp.MLP(*s.layers).train(train)
    s.x = g.normal(*shape, width, dtype=dtype)
    if train:
        s.x.requires_grad_(True)
        s.wants = [s.x] + (_params(s.layers) if kind != "linear" else [])
    return s


# ---- one pass ------------------------------------------------------------------------------

def _forward(s):
    kind = s.case["kind"]
    for layer, keep in zip(s.layers, s.keeps):
        layer.next_keep = keep
    if kind in ("linear", "lora"):
        return [s.layers[0](s.x)]
    if kind == "mlp":
        return [s.module(s.x)]
    (q, k, v), rotated = attention.project_qkv(s.attn, s.x, (s.cos, s.sin))
    n_q, n_kv = s.case["heads"], s.case["kv_heads"]
    if rotated:
        query, key = rope.rotated_heads(q, k, s.cos, s.sin, n_q, n_kv)
        value = rope.as_heads(v, n_kv)
    else:
        query, key, value = rope.qkv_rope(q, None, k, v, None, s.cos, s.sin, n_q, n_kv)
    return [query, key, value]


def run(s):
    kind = s.case["kind"]
    if kind == "unpack":
        st = s.state
        return nf4.unpack_nf4(s.packed, st.shape, st.state2.absmax, st.blocksize, s.dtype,
                              absmax_8bit=st.absmax, code=st.state2.code, offset=st.offset)
    if kind == "quantize":
        packed, st = quant.quantize_4bit(s.w)
        return [packed, st.absmax, st.state2.absmax, st.offset]
    if not s.case["train"]:
        with torch.no_grad():
            return _forward(s)
    ys = _forward(s)
    grads = torch.autograd.grad(ys, s.wants, s.dys)
    return [y.detach() for y in ys] + list(grads)


# ---- what a pass cannot do without -----------------------------------------------------------

def _linears(case):
    """(N, K) of the case's projections."""
    kind = case["kind"]
    if kind == "qkv":
        h = case["hidden"]
        return [(case["heads"] * HEAD, h)] + [(case["kv_heads"] * HEAD, h)] * 2
    if kind == "mlp":
        h, i = case["hidden"], case["inter"]
        return [(i, h), (i, h), (h, i)]
    return [(case["n"], case["k"])]


def _nf4_bytes(n, k):
    return n * k / 2 + n * k / 64 + n * k / 64 / 256 * 4 + 1028


def work(case):
    kind = case["kind"]
    if kind == "unpack":
        n, k = case["n"], case["k"]
        return {"bytes": _nf4_bytes(n, k) + n * k * (2 if case["dtype"] == "float16" else 4),
                "flops": n * k}
    if kind == "quantize":
        n, k = case["n"], case["k"]
        return {"bytes": 2 * n * k + _nf4_bytes(n, k), "flops": 16 * n * k}
    m, train, r = case["tokens"], case["train"], case.get("r", 0)
    flops = nbytes = 0
    for n, k in _linears(case):
        main, low = 2 * m * n * k, 2 * m * r * (n + k)
        flops += (2 if train else 1) * main + (3 if train else 1) * low
        nbytes += _nf4_bytes(n, k) + 4 * r * (n + k) * (2 if train else 1)
        if train and case.get("drop", 0) > 0:
            nbytes += m * k  # the byte keep mask
    width = case.get("hidden", case.get("k"))
    outs = [width] if kind == "mlp" else [n for n, _ in _linears(case)]
    item = 4 if kind == "mlp" and train else 2
    nbytes += item * m * (width + sum(outs)) * (2 if train else 1)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("unpack", "quantize"):
        return "exact"
    # fp16 outputs of fp32 sums, the LoRA terms through an fp16 [tokens, r] operand: at most
    # 3.6e-4 from the 64-bit result; the MLP, through three fp16 [tokens, intermediate]
    # activations, 4.9e-4.  Four times that.
    return {"rel": 2e-3 if kind == "mlp" else 1.4e-3}


# ---- 64-bit reference --------------------------------------------------------------------------

_NF4 = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453,
        -0.28444138169288635, -0.18477343022823334, -0.09105003625154495, 0.0,
        0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
        0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0]


def _dense(packed, state, rounded=True):
    """The weight's values in fp64: decoded from the format; rounded to the fp16 values it
    stands for, or before that rounding."""
    b = packed.reshape(-1).to(torch.int64)
    codes = torch.stack((b >> 4, b & 15), -1).reshape(-1)
    table = torch.tensor(_NF4, dtype=torch.float64, device=b.device)
    blocks = state.absmax.numel()
    scale = state.state2.code.double()[state.absmax.reshape(-1).long()]
    scale = scale * state.state2.absmax.double().repeat_interleave(256)[:blocks]
    scale = (scale + state.offset.double()).float().double()
    w = table[codes].view(-1, 64) * scale[:, None]
    w = w.view(tuple(state.shape))
    return w.float().half().double() if rounded else w


def _rotate(y, cos, sin, heads):
    b, t = y.shape[:2]
    y = y.view(b, t, heads, HEAD).transpose(1, 2)
    c, sn = cos.double()[:, None], sin.double()[:, None]
    half = torch.cat((-y[..., HEAD // 2:], y[..., :HEAD // 2]), -1)
    return y * c + half * sn


def exact(case, seed):
    kind = case["kind"]
    if kind == "quantize":
        return None  # codes, not computed numbers
    s = prepare(case, seed)
    if kind == "unpack":
        return _dense(s.packed, s.state, rounded=False)
    train = case["train"]
    x = s.x.detach().half().double().requires_grad_(train)
    params = []

    def project(i, inp):
        layer = s.layers[i]
        base = layer if kind == "linear" else layer.base_layer
        y = inp @ _dense(base.weight.data, base.weight.quant_state).t()
        if base.bias is not None:
            y = y + base.bias.double()
        if kind == "linear":
            return y
        a, b = (p.detach().half().double().requires_grad_(train) for p in _params([layer]))
        params.extend((a, b))
        h = inp
        if s.keeps[i] is not None:
            h = inp * s.keeps[i].view(inp.shape).double() / (1.0 - case["drop"])
        return y + (h @ a.t() @ b.t()) * SCALING

    with torch.set_grad_enabled(train):
        if kind == "mlp":
            ys = [project(2, torch.nn.functional.silu(project(0, x)) * project(1, x))]
        elif kind == "qkv":
            q, k, v = (project(i, x) for i in range(3))
            ys = [_rotate(q, s.cos, s.sin, case["heads"]),
                  _rotate(k, s.cos, s.sin, case["kv_heads"]),
                  v.view(*v.shape[:2], case["kv_heads"], HEAD).transpose(1, 2)]
        else:
            ys = [project(0, x)]
        if not train:
            return ys
        grads = torch.autograd.grad(ys, [x] + params, [d.half().double() for d in s.dys])
    return [y.detach() for y in ys] + list(grads)
