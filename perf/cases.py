"""The work that is measured: what a program built on libtinygiant_hip.so has
it do, through the C ABI (include/tinygiant_hip.h) and the package's wrappers.

  matmul     tg_hip_matmul_dev: quantized matrix x k rows held on the device
  head       tg_hip_head_argmax_dev: output norm, q6_K head and greedy argmax
  attention  tg_hip_attention_dev: one decode step of a layer's attention
  engine     moe_forward_rows_v2: the host-buffer call of the unchanged engine,
             its experts registered with tg_mlock
  layer      tg_hip_moe_plan_run: one planned MoE layer on device rows
  step       tg_hip_decode_run: all MoE layers of a decode step, a verify pass
             or a prefill chunk, from the rows' embeddings on

The shapes are those of the two models the package names (tinygiant_amd/
synth.py): Qwen3-30B-A3B (q4_K gate/up, q6_K down) and gpt-oss-120b (MXFP4,
biases, clamped SwiGLU); routing is a Zipf(1.1) popularity over a permutation
of the experts, as there.  Weights are drawn block by block in their formats,
with the spread that keeps activations near one, as trained weights do.

exact() computes the same function with torch in 64 bits.  Inputs that the
caller gives are rounded to q8 as the formats define it (32-bit arithmetic on
given values, so the codes are the same everywhere); values that the path
computes itself (normed rows, hidden rows, attention outputs) are left as
they are: their own q8 rounding depends on the last bit of a sum, and it is
most of the error that the outputs behind it show.
"""

import ctypes
import math

import numpy as np
import torch

import tinygiant_amd as tg

Q4K, F16, Q6K, MXFP4, Q80 = tg.FMT_Q4K, tg.FMT_F16, tg.FMT_Q6K, tg.FMT_MXFP4, tg.FMT_Q80
FORMATS = {"q4_k": Q4K, "float16": F16, "q6_k": Q6K, "mxfp4": MXFP4, "q8_0": Q80}
BLOCK = {Q4K: (256, 144), Q6K: (256, 210), MXFP4: (32, 17), Q80: (32, 34), F16: (1, 2)}   # values, bytes

MODELS = {
    "qwen3": dict(D=2048, I=768, E=128, top=8, L=48, gate=Q4K, down=Q6K, act=tg.ACT_SILU, bias=False, eps=1e-6),
    "gptoss": dict(D=2880, I=2880, E=128, top=4, L=36, gate=MXFP4, down=MXFP4, act=tg.ACT_GPTOSS, bias=True, eps=1e-5),
}
ATTENTION = {
    "qwen3": dict(D=2048, nh=32, nkv=4, hd=128, fmts=(Q4K, Q4K, Q6K, Q4K), norm=True, bias=False, sinks=False),
    "gptoss": dict(D=2880, nh=64, nkv=8, hd=64, fmts=(Q80, Q80, Q80, Q80), norm=False, bias=True, sinks=True),
}
VOCAB, HEAD_COLS = 151936, 2048


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # a lone projection of one token, the smallest call there is: latency
        dict(name="matmul q4_k one row", kind="matmul", fmt="q4_k", rows=768, cols=2048, k=1, bias=False),
        # the next token of a plain decode
        dict(name="head one row", kind="head", vocab=VOCAB, k=1),
        # the targets of a speculative round of eight drafts
        dict(name="head verify", kind="head", vocab=VOCAB, k=9),
        # a decode step in a conversation of a few thousand tokens
        dict(name="attention qwen3", kind="attention", model="qwen3", kv=4000, kv_max=4096, window=0),
        # a full-attention layer in a long document
        dict(name="attention gptoss long", kind="attention", model="gptoss", kv=30001, kv_max=32768, window=0),
        # the engine decoding token by token over host buffers
        dict(name="engine qwen3 one row", kind="engine", model="qwen3", k=1),
        # the verify batch's MoE layer
        dict(name="layer qwen3 verify", kind="layer", model="qwen3", k=5),
        # prompts: an ordinary one, and a long one in one piece
        dict(name="layer gptoss prompt", kind="layer", model="gptoss", k=64),
        dict(name="layer qwen3 long prompt", kind="layer", model="qwen3", k=509),
        # one token through every layer of either model
        dict(name="step qwen3", kind="step", model="qwen3", layers=48, k=1),
        dict(name="step gptoss", kind="step", model="gptoss", layers=36, k=1),
        # the verify pass of eight drafts through every layer
        dict(name="step qwen3 verify", kind="step", model="qwen3", layers=48, k=9),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))


def draw(rng):
    kind = rng.choice(["matmul", "matmul", "head", "attention", "attention", "engine", "layer", "layer", "layer", "step"])
    if kind == "matmul":
        fmt = rng.choice(list(FORMATS))
        unit = BLOCK[FORMATS[fmt]][0] if FORMATS[fmt] != F16 else 32
        cols = unit * _log_int(rng, max(1, 256 // unit), 8192 // unit)
        return dict(kind=kind, fmt=fmt, rows=_log_int(rng, 100, 12000), cols=cols, k=_log_int(rng, 1, 16),
                    bias=rng.random() < 0.5)
    if kind == "head":
        return dict(kind=kind, vocab=rng.choice([VOCAB, _log_int(rng, 30000, VOCAB)]), k=_log_int(rng, 1, 16))
    if kind == "attention":
        model = rng.choice(list(ATTENTION))
        kv = _log_int(rng, 16, 32000)
        window = 128 if model == "gptoss" and rng.random() < 0.5 else 0   # every other layer slides
        return dict(kind=kind, model=model, kv=kv, kv_max=1024 * (kv // 1024 + 1), window=window)
    model = rng.choice(list(MODELS))
    if kind == "engine":
        return dict(kind=kind, model=model, k=_log_int(rng, 1, 9 if model == "qwen3" else 4))
    if kind == "layer":
        return dict(kind=kind, model=model, k=_log_int(rng, 1, 512 if model == "qwen3" else 200))
    if model == "gptoss":
        return dict(kind=kind, model=model, layers=_log_int(rng, 9, 36), k=1)
    k = rng.choice([1, 1, _log_int(rng, 2, 9)])
    return dict(kind=kind, model=model, layers=_log_int(rng, 12, 48), k=k)


# ------------------------------------------------------------------ inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * scale


def _bytes(g, n):
    words = torch.randint(-2 ** 31, 2 ** 31, ((n + 3) // 4,), generator=g, device="cuda", dtype=torch.int32)
    return words.view(torch.uint8)[:n]


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def _row_bytes(fmt, cols):
    vals, size = BLOCK[fmt]
    return cols // vals * size


def _weights(g, fmt, n, cols):
    """n rows of `cols` weights of zero mean and a spread of about cols ** -0.5, in the format's blocks."""
    if fmt == F16:
        return _f16_bytes(_normal(g, n, cols, scale=cols ** -0.5)).reshape(-1)
    vals, size = BLOCK[fmt]
    nb = n * cols // vals
    b = _bytes(g, nb * size).view(nb, size)
    s = cols ** -0.5 * torch.empty(nb, device="cuda").uniform_(0.8, 1.25, generator=g)
    if fmt == Q4K:      # scales 32..63, mins beside them, so that 0..15 is centred
        sc = torch.randint(32, 64, (nb, 8), generator=g, device="cuda", dtype=torch.uint8)
        mn = (sc ^ (b[:, 16:24] & 3))
        b[:, 0:2] = _f16_bytes(s / (4.6 * 47.5))
        b[:, 2:4] = _f16_bytes(s / (4.6 * 47.5) * 7.5)
        b[:, 4:8] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
        b[:, 8:12] = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
        b[:, 12:16] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    elif fmt == Q6K:    # 6-bit codes under signed scales of size 32..127
        sc = torch.randint(32, 128, (nb, 16), generator=g, device="cuda", dtype=torch.int16)
        b[:, 192:208] = torch.where(b[:, :16] > 127, -sc, sc).to(torch.int8).view(torch.uint8)
        b[:, 208:210] = _f16_bytes(s / (18.5 * 84))
    elif fmt == MXFP4:  # e2m1 codes (spread 2.9) under a power of two
        b[:, 0] = (torch.log2(s / 2.9).round() + 127).to(torch.uint8)
    else:
        b[:, 0:2] = _f16_bytes(s / 73.6)
    return b.view(-1)


def _routing(seed, k, n_experts, top):
    """The experts that k tokens choose, in order, and the weights [experts][k] of the rows."""
    rng = np.random.default_rng(seed)
    perm = rng.permutation(n_experts)
    keys = -1.1 * np.log(np.arange(1, n_experts + 1)) + rng.gumbel(size=(k, n_experts))
    chosen = perm[np.argsort(-keys, axis=1)[:, :top]]
    w = np.exp(rng.standard_normal((k, top)))
    w /= w.sum(axis=1, keepdims=True)
    full = np.zeros((n_experts, k), np.float32)
    full[chosen, np.arange(k)[:, None]] = w
    experts = np.flatnonzero((full != 0).any(axis=1))
    return experts, np.ascontiguousarray(full[experts])


class Layer:
    """One MoE layer's active experts (weights as one buffer a matrix kind), biases and routing."""

    def __init__(self, g, m, k, seed):
        self.m, self.k = m, k
        self.experts, self.rw = _routing(seed, k, m["E"], m["top"])
        self.n = n = len(self.experts)
        self.gate = _weights(g, m["gate"], n * m["I"], m["D"])
        self.up = _weights(g, m["gate"], n * m["I"], m["D"])
        self.down = _weights(g, m["down"], n * m["D"], m["I"])
        self.bias = None
        if m["bias"]:
            self.bias = [_normal(g, n, c, scale=0.05) for c in (m["I"], m["I"], m["D"])]

    def plan(self):
        m, n, vp = self.m, self.n, ctypes.c_void_p
        mats = [(vp * n)(*[t.data_ptr() + e * (t.numel() // n) for e in range(n)]) for t in (self.gate, self.up, self.down)]
        bias = [(vp * n)(*[t[e].data_ptr() for e in range(n)]) for t in self.bias] if self.bias else [None] * 3
        fmts = np.full(n, m["down"], np.int32)
        p = tg.lib().tg_hip_moe_plan_create(*mats, m["gate"], fmts.ctypes.data, *bias, m["act"], n, self.rw.ctypes.data,
                                            self.k, m["D"], m["I"])
        if not p:
            raise RuntimeError(tg.last_error())
        return p


class State:
    """What a program holds between calls; the library's handles are given back with it."""

    def __init__(self, kind):
        self.kind, self.plans, self.step, self.registered = kind, [], None, []

    def __del__(self):
        if not tg:   # the interpreter is going down
            return
        lib = tg.lib()
        if self.step:
            lib.tg_hip_decode_destroy(self.step)
        for p in self.plans:
            lib.tg_hip_moe_plan_destroy(p)
        for a in self.registered:
            lib.tg_hip_unregister(a.ctypes.data)


def _inputs(case, seed):
    """The case's inputs as torch tensors on the GPU, from the seed alone."""
    g, s = _generator(seed), State(case["kind"])
    if s.kind == "matmul":
        fmt = FORMATS[case["fmt"]]
        s.w = _weights(g, fmt, case["rows"], case["cols"])
        s.bias = _normal(g, case["rows"], scale=0.1) if case["bias"] else None
        s.x = _normal(g, case["k"], case["cols"])
    elif s.kind == "head":
        s.w = _weights(g, Q6K, case["vocab"], HEAD_COLS)
        s.norm = torch.empty(HEAD_COLS, device="cuda").uniform_(0.5, 1.5, generator=g)
        s.x = _normal(g, case["k"], HEAD_COLS, scale=1.5)
    elif s.kind == "attention":
        a, kv_max = ATTENTION[case["model"]], case["kv_max"]
        qd, kd = a["nh"] * a["hd"], a["nkv"] * a["hd"]
        shapes = ((qd, a["D"]), (kd, a["D"]), (kd, a["D"]), (a["D"], qd))
        s.w = [_weights(g, f, r, c) for f, (r, c) in zip(a["fmts"], shapes)]
        s.bias = [_normal(g, r, scale=0.1) for r, _ in shapes] if a["bias"] else [None] * 4
        s.norm = [torch.empty(a["hd"], device="cuda").uniform_(0.5, 1.5, generator=g) for _ in range(2)] if a["norm"] else [None] * 2
        s.sinks = _normal(g, a["nh"]) if a["sinks"] else None
        half = a["hd"] // 2
        angle = torch.arange(kv_max, device="cuda")[:, None] / 1e6 ** (torch.arange(half, device="cuda") / half)
        s.cos, s.sin = angle.cos().contiguous(), angle.sin().contiguous()
        s.kv = [torch.zeros(a["nkv"], kv_max, a["hd"], device="cuda") for _ in range(2)]
        for t in s.kv:
            t[:, :case["kv"]] = _normal(g, a["nkv"], case["kv"], a["hd"])
        s.x = _normal(g, 1, a["D"])
    elif s.kind in ("engine", "layer"):
        m = MODELS[case["model"]]
        s.layer = Layer(g, m, case["k"], seed)
        s.x = _normal(g, case["k"], m["D"])
        s.out = _normal(g, case["k"], m["D"])
    else:
        m = MODELS[case["model"]]
        s.layers = [Layer(g, m, case["k"], (seed, i)) for i in range(case["layers"])]
        s.norms = [torch.empty(m["D"], device="cuda").uniform_(0.5, 1.5, generator=g) for _ in range(case["layers"])]
        s.x = _normal(g, case["k"], m["D"], scale=8)   # a residual stream some times a layer's update, as inside a model
    return s


def _ptr(t):
    return None if t is None else t.data_ptr()


def prepare(case, seed):
    lib, s = tg.lib(), _inputs(case, seed)
    torch.cuda.synchronize()   # the library runs on a stream of its own: plans read the weights there
    scratch = lambda n: torch.empty(n, dtype=torch.uint8, device="cuda")   # noqa: E731
    if s.kind == "matmul":
        s.out = torch.empty(case["k"], case["rows"], device="cuda")
        s.scratch = scratch(lib.tg_hip_matmul_scratch_bytes(case["k"], case["cols"]))
        s.args = (FORMATS[case["fmt"]], _ptr(s.w), _ptr(s.bias), _ptr(s.x), _ptr(s.out), case["rows"], case["cols"],
                  case["k"], _ptr(s.scratch), None)
    elif s.kind == "head":
        k, vocab = case["k"], case["vocab"]
        s.logits = torch.empty(k, vocab, device="cuda")
        s.argmax = torch.empty(k, dtype=torch.int32, device="cuda")
        s.maxval = torch.empty(k, device="cuda")
        s.scratch = scratch(lib.tg_hip_head_scratch_bytes(k, vocab, HEAD_COLS))
        s.args = (Q6K, _ptr(s.w), _ptr(s.x), _ptr(s.norm), 1e-6, k, vocab, HEAD_COLS, _ptr(s.logits), _ptr(s.argmax),
                  _ptr(s.maxval), _ptr(s.scratch), None)
    elif s.kind == "attention":
        a = ATTENTION[case["model"]]
        s.out = torch.empty(a["D"], device="cuda")
        s.heads = torch.empty(a["nh"], a["hd"], device="cuda")
        s.scratch = scratch(lib.tg_hip_attention_scratch_bytes(a["D"], a["nh"], a["nkv"], a["hd"], case["kv_max"]))
        s.args = (*a["fmts"], *map(_ptr, s.w), *map(_ptr, s.bias), *map(_ptr, s.norm), _ptr(s.sinks), *map(_ptr, s.kv),
                  case["kv"], case["kv_max"], case["window"], _ptr(s.cos), _ptr(s.sin), _ptr(s.x), _ptr(s.out), a["D"],
                  a["nh"], a["nkv"], a["hd"], case["kv"], 1e-6, _ptr(s.heads), _ptr(s.scratch), None)
    elif s.kind == "engine":
        l = s.layer
        s.host = []
        for t in (l.gate, l.up, l.down):
            a = t.cpu().numpy()
            if lib.tg_mlock(a.ctypes.data, a.nbytes):
                raise RuntimeError(tg.last_error())
            s.registered.append(a)
            s.host.append(list(a.reshape(l.n, -1)))
        s.host_bias = [list(t.cpu().numpy()) for t in l.bias] if l.bias else [None] * 3
        s.host_x, s.host_out = s.x.cpu().numpy(), s.out.cpu().numpy()
        l.gate = l.up = l.down = None
    elif s.kind == "layer":
        s.plans.append(s.layer.plan())
    else:
        m, n = MODELS[case["model"]], case["layers"]
        s.h = torch.empty_like(s.x)
        s.plans += [l.plan() for l in s.layers]
        s.step = lib.tg_hip_decode_create((ctypes.c_void_p * n)(*s.plans), n,
                                          (ctypes.c_void_p * n)(*map(_ptr, s.norms)), m["eps"], _ptr(s.h), 2)
        if not s.step:
            raise RuntimeError(tg.last_error())
    torch.cuda.synchronize()
    return s


def run(s):
    lib = tg.lib()
    if s.kind == "matmul":
        lib.tg_hip_matmul_dev(*s.args)
        return s.out
    if s.kind == "head":
        lib.tg_hip_head_argmax_dev(*s.args)
        return dict(logits=s.logits, argmax=s.argmax, maxval=s.maxval)
    if s.kind == "attention":
        lib.tg_hip_attention_dev(*s.args)
        return dict(out=s.out, heads=s.heads, k=s.kv[0], v=s.kv[1])
    if s.kind == "engine":   # the engine adds the experts to a copy of its residual rows
        m, l = s.layer.m, s.layer
        return tg.moe_forward_rows_v2(*s.host, m["gate"], [m["down"]] * l.n, *s.host_bias, m["act"], l.rw, s.host_x,
                                      s.host_out.copy(), m["I"])
    if s.kind == "layer":    # accumulated into the residual rows, pass after pass
        lib.tg_hip_moe_plan_run(s.plans[0], _ptr(s.x), _ptr(s.out), None)
        return s.out
    lib.tg_hip_memcpy_d2d(_ptr(s.h), _ptr(s.x), s.x.numel() * 4, None)
    lib.tg_hip_decode_run(s.step, None)
    return s.h


# ------------------------------------------------------------------ work, tolerance

def _expert_work(m, seed, k):
    """Bytes of the active experts' weights and biases, and multiply-adds, of a layer's k rows."""
    n = len(_routing(seed, k, m["E"], m["top"])[0])
    D, I = m["D"], m["I"]
    size = 2 * I * _row_bytes(m["gate"], D) + D * _row_bytes(m["down"], I) + (4 * (2 * I + D) if m["bias"] else 0)
    return n * size, k * m["top"] * 3 * D * I


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        r, c, k = case["rows"], case["cols"], case["k"]
        return dict(bytes=r * _row_bytes(FORMATS[case["fmt"]], c) + 4 * k * (r + c) + (4 * r if case["bias"] else 0),
                    flops=2 * r * c * k)
    if kind == "head":
        r, k = case["vocab"], case["k"]
        return dict(bytes=r * _row_bytes(Q6K, HEAD_COLS) + 4 * k * (r + HEAD_COLS), flops=2 * r * HEAD_COLS * k)
    if kind == "attention":
        a = ATTENTION[case["model"]]
        qd, kd = a["nh"] * a["hd"], a["nkv"] * a["hd"]
        seen = case["kv"] + 1 if not case["window"] else min(case["kv"] + 1, case["window"])
        fq, fk, fv, fo = a["fmts"]
        mats = qd * _row_bytes(fq, a["D"]) + kd * (_row_bytes(fk, a["D"]) + _row_bytes(fv, a["D"])) + a["D"] * _row_bytes(fo, qd)
        return dict(bytes=mats + 8 * kd * seen + 8 * a["D"] + 4 * qd,
                    flops=2 * (2 * qd + 2 * kd) * a["D"] + 4 * qd * seen)
    m, k = MODELS[case["model"]], case["k"]
    rows = [_expert_work(m, i, k) for i in range(case.get("layers", 1))]   # a typical routing's
    return dict(bytes=sum(b for b, _ in rows) + 12 * k * m["D"], flops=2 * sum(f for _, f in rows))


def tolerance(case):
    return TOLERANCE[case["kind"]]


# Sums in another order differ by 1e-7 to 3e-7 (measured between this library's v_dot4, int8 MFMA and per-layer
# kernels, and from exact()).  Where the path rounds values that it computed to q8, such a difference now and then
# moves one of them by a whole step, and the outputs behind it by up to 3e-4 (24 layers of one row); through the 36
# or 48 layers of a step it grows to between 1e-3 and 1e-2.
TOLERANCE = {
    "matmul": {"rel": 2e-6},
    "head": {"rel": 1e-3},
    "attention": {"rel": 1e-3},
    "engine": {"rel": 1e-3},
    "layer": {"rel": 1e-3},
    "step": {"rel": 3e-2, "max": 0.2},
}


# ------------------------------------------------------------------ the same in 64 bits

def _f16_at(b, i):
    return b[:, i:i + 2].contiguous().view(torch.float16).double()   # [blocks, 1]


def _dequantize(fmt, w, rows, cols):
    """[rows][cols] in 64 bits."""
    if fmt == F16:
        return w.view(torch.float16).view(rows, cols).double()
    vals, size = BLOCK[fmt]
    b = w.view(-1, size)
    if fmt == Q4K:
        s = b[:, 4:16].to(torch.int16)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        v = q * (_f16_at(b, 0) * sc.double())[..., None] - (_f16_at(b, 2) * mn.double())[..., None]
    elif fmt == Q6K:
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        shift = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=w.device).view(1, 1, 4, 1)
        q = torch.cat([ql & 15, ql >> 4], 2) | (((qh >> shift) & 3) << 4)     # [blocks][2][4][32]
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = (q.double() - 32).reshape(-1, 16, 16) * (_f16_at(b, 208) * sc)[..., None]
    elif fmt == MXFP4:
        table = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device=w.device)
        c = b[:, 1:].long()
        v = table[torch.cat([c & 15, c >> 4], 1)] * torch.exp2(b[:, :1].double() - 127)
    else:
        v = b[:, 2:].contiguous().view(torch.int8).double() * _f16_at(b, 0)
    return v.reshape(rows, cols)


def _q8(x):
    """Rows rounded to q8 blocks of 256 values (scale amax / 127, round half to even), in 64 bits."""
    k, n = x.shape
    b = torch.nn.functional.pad(x, (0, -n % 256)).view(k, -1, 256)
    amax = b.abs().amax(2, keepdim=True)
    inv = torch.where(amax > 0, 127 / amax, torch.zeros_like(amax))
    return ((b * inv).round().double() * (amax / 127).double()).view(k, -1)[:, :n]


def _rms(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w.double()


def _act(act, g, u):
    if act == tg.ACT_GPTOSS:
        g, u = g.clamp(max=7), u.clamp(-7, 7)
        return g * torch.sigmoid(1.702 * g) * (u + 1)
    return g * torch.sigmoid(g) * u


def _moe(l, x, out):
    """out + MoE(x), one expert after the other."""
    m, out = l.m, out.clone()
    gate, up, down = (t.view(l.n, -1) for t in (l.gate, l.up, l.down))
    for e in range(l.n):
        r = np.flatnonzero(l.rw[e])
        w = torch.from_numpy(l.rw[e][r]).cuda().double()[:, None]
        r = torch.from_numpy(r).cuda()
        gu = [x[r] @ _dequantize(m["gate"], t[e], m["I"], m["D"]).T for t in (gate, up)]
        if l.bias:
            gu = [t + b[e].double() for t, b in zip(gu, l.bias)]
        y = _act(m["act"], *gu) @ _dequantize(m["down"], down[e], m["D"], m["I"]).T
        if l.bias:
            y += l.bias[2][e].double()
        out[r] += w * y
    return out


def _attend(case, s):
    a, pos = ATTENTION[case["model"]], case["kv"]
    qd, kd, hd = a["nh"] * a["hd"], a["nkv"] * a["hd"], a["hd"]
    rows = (qd, kd, kd)
    x = _q8(s.x)
    q, k, v = ((x @ _dequantize(f, w, r, a["D"]).T)[0] + (0 if b is None else b.double())
               for f, w, b, r in zip(a["fmts"], s.w, s.bias, rows))
    q, k, v = q.view(-1, hd), k.view(-1, hd), v.view(-1, hd)
    if a["norm"]:
        q, k = _rms(q, s.norm[0], 1e-6), _rms(k, s.norm[1], 1e-6)
    cos, sin = s.cos[pos].double(), s.sin[pos].double()

    def turn(t):
        u, w = t[:, :hd // 2], t[:, hd // 2:]
        return torch.cat([u * cos - w * sin, w * cos + u * sin], 1)

    q, k = turn(q), turn(k)
    keys, vals = (t.double() for t in s.kv)
    keys[:, pos], vals[:, pos] = k, v
    first = max(0, pos + 1 - case["window"]) if case["window"] else 0
    group = a["nh"] // a["nkv"]
    heads = []
    for h in range(a["nkv"]):
        z = q[h * group:(h + 1) * group] @ keys[h, first:pos + 1].T / hd ** 0.5
        if a["sinks"]:
            z = torch.cat([z, s.sinks[h * group:(h + 1) * group, None].double()], 1)
        p = z.softmax(1)[:, :pos + 1 - first]
        heads.append(p @ vals[h, first:pos + 1])
    heads = torch.cat(heads)
    out = heads.view(1, -1) @ _dequantize(a["fmts"][3], s.w[3], a["D"], qd).T
    out = out[0] + (0 if s.bias[3] is None else s.bias[3].double())
    return dict(out=out, heads=heads, k=keys, v=vals)


def exact(case, seed):
    s = _inputs(case, seed)
    if s.kind == "matmul":
        fmt = FORMATS[case["fmt"]]
        x = s.x.double() if fmt == F16 else _q8(s.x)   # 16-bit weights meet the rows themselves
        y = x @ _dequantize(fmt, s.w, case["rows"], case["cols"]).T
        return y if s.bias is None else y + s.bias.double()
    if s.kind == "head":
        x = _rms(s.x.double(), s.norm, 1e-6)
        w = s.w.view(case["vocab"], -1)
        logits = torch.cat([x @ _dequantize(Q6K, c.reshape(-1), len(c), HEAD_COLS).T for c in w.split(16384)], 1)
        return dict(logits=logits, argmax=None, maxval=logits.amax(1))
    if s.kind == "attention":
        return _attend(case, s)
    if s.kind in ("engine", "layer"):
        y = _moe(s.layer, _q8(s.x), s.out.double())
        return y.cpu().numpy() if s.kind == "engine" else y
    m, h = MODELS[case["model"]], s.x.double()
    for l, w in zip(s.layers, s.norms):
        h = _moe(l, _rms(h, w, m["eps"]), h)
    return h
