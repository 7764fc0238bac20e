"""The work that programs built on this framework have it do, as timed cases.

Every case goes through the package's own bindings (saphira-llm_amd), on
synthetic tensors made from a seed: uniform ternary I2_S weights with a
per-tensor scale U(0.5, 2) (in whole models over sqrt(2 K / 3), so that a
projection keeps its input's size as a trained one does), f32 N(0, 1)
activations, an F16 N(0, 1) embedding, norm weights N(1, 0.1^2). Kinds of case and their ranges:

linear        projections of one token, each a call that quantises its
              activation on the way: 64..32768 rows of K = 128..16384
linear_batch  one projection of a chunk or batch of tokens (quantiser, then
              the GEMM): 2..4096 tokens
plan          the projections of whole blocks for one token, as one plan
gemm_plan     the FFN projections of many blocks for a few tokens, as one plan
row           one FFN through the host-pointer kernel row, as a host program
              that dispatches its kernels through it calls them
prefill       a prompt through a whole model in chunks, the last logits back
score         one chunk of tokens through a whole model, every logit back
generate      a prompt, then greedy decoding, then the next logits

Results are the same bits whatever the route (int32 dots are exact and every
f32 operation has a fixed order), so every tolerance is "exact".
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    name = "saphira_llm_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, os.path.join(ROOT, "saphira-llm_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


amd = _package()
_device = []


def device():
    """The library, opened on the first GPU (once per process)."""
    if not _device:
        torch.cuda.init()
        _device.append(amd.Device(0))
    return _device[0]


# Model shapes: BitNet-b1.58-2B, and the small ones of the repository's tests.
SHAPES = {
    "2b": dict(n_embd=2560, n_ff=6912, n_head=20, n_head_kv=5, n_rot=128),
    "narrow": dict(n_embd=512, n_ff=1024, n_head=8, n_head_kv=2, n_rot=48),
    "odd": dict(n_embd=384, n_ff=640, n_head=6, n_head_kv=2, n_rot=64),
    "tiny": dict(n_embd=256, n_ff=512, n_head=4, n_head_kv=2, n_rot=64),
}
VOCAB_2B = 128256
EPS, ROPE_BASE = 1e-5, 500000.0


def listed():
    return [
        # the smallest calls of a decode step: K, then V of one token
        {"name": "linear_kv_640x2560", "kind": "linear", "calls": 2, "rows": 640, "k": 2560},
        # one token against a wide FFN's down projection
        {"name": "linear_wide_4096x14336", "kind": "linear", "calls": 1, "rows": 4096, "k": 14336},
        # every projection of a 30-block model for one token
        {"name": "plan_30_blocks", "kind": "plan", "shape": "2b", "blocks": 30},
        # the FFN projections of 32 blocks for a batch of 16 requests
        {"name": "gemm_plan_ffn_16", "kind": "gemm_plan", "shape": "2b", "blocks": 32, "tokens": 16},
        # gate or up for a batch of 64 requests
        {"name": "batch_64_6912x2560", "kind": "linear_batch", "tokens": 64, "rows": 6912, "k": 2560},
        # the same for a prefill chunk
        {"name": "batch_512_6912x2560", "kind": "linear_batch", "tokens": 512, "rows": 6912, "k": 2560},
        # down for a long prompt or many prompts at once
        {"name": "batch_4096_2560x6912", "kind": "linear_batch", "tokens": 4096, "rows": 2560, "k": 6912},
        # a ragged batch against a tensor of uneven sizes
        {"name": "batch_77_1000x1408", "kind": "linear_batch", "tokens": 77, "rows": 1000, "k": 1408},
        # one block's FFN behind the reference's kernel dispatch, host to host
        {"name": "row_ffn", "kind": "row", "embd": 2560, "ff": 6912},
        # a long prompt's prefill
        {"name": "prefill_2b_2048", "kind": "prefill", "shape": "2b", "layers": 30, "vocab": VOCAB_2B,
         "prompt": 2048, "chunk": 512},
        # scoring a text: the logits of every position
        {"name": "score_2b_128", "kind": "score", "shape": "2b", "layers": 30, "vocab": VOCAB_2B, "tokens": 128},
        # a chat turn: prompt, then decoding at batch 1
        {"name": "generate_2b_512_64", "kind": "generate", "shape": "2b", "layers": 30, "vocab": VOCAB_2B,
         "prompt": 512, "new": 64},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear_batch", "linear_batch", "linear_batch", "plan", "gemm_plan", "row",
                       "prefill", "score", "generate"])
    if kind == "linear":
        return {"kind": kind, "calls": rng.randint(2, 4), "rows": _log(rng, 64, 32768), "k": 128 * _log(rng, 1, 128)}
    if kind == "linear_batch":
        while True:
            c = {"kind": kind, "tokens": _log(rng, 2, 4096), "rows": _log(rng, 64, 16384), "k": 128 * _log(rng, 1, 128)}
            if c["tokens"] * c["rows"] * c["k"] <= 4096 * 2560 * 6912 and c["tokens"] * c["rows"] <= 4096 * 6912:
                return c
    if kind == "plan":
        return {"kind": kind, "shape": rng.choice(["2b", "2b", "narrow", "tiny"]), "blocks": _log(rng, 1, 30)}
    if kind == "gemm_plan":
        return {"kind": kind, "shape": rng.choice(["2b", "2b", "narrow", "tiny"]), "blocks": _log(rng, 1, 32),
                "tokens": _log(rng, 1, 64)}
    if kind == "row":
        return {"kind": kind, "embd": 128 * _log(rng, 1, 40), "ff": 128 * _log(rng, 2, 112)}
    c = {"kind": kind, "shape": rng.choice(["2b", "2b", "2b", "narrow", "odd", "tiny"]), "layers": rng.randint(1, 3),
         "vocab": _log(rng, 500, VOCAB_2B)}
    if kind == "prefill":
        c.update(prompt=_log(rng, 2, 2048), chunk=_log(rng, 16, 512))
    elif kind == "score":
        c.update(tokens=_log(rng, 2, 256))
    else:
        c.update(prompt=_log(rng, 1, 1024), new=_log(rng, 4, 64))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

class _Rng:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, dtype=torch.float32):
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=dtype)

    def integers(self, hi, n):
        return torch.randint(0, hi, (n,), generator=self.g, device="cuda", dtype=torch.int32)

    def norm_weight(self, n):
        return 1 + 0.1 * self.normal(n)

    def ternary(self, rows, k, gain=1.0):
        """A packed I2_S tensor: rows * k / 4 code bytes, then the 32-byte tail with its scale."""
        n = rows * k // 4
        v = torch.arange(81)
        codes = ((v // 27) << 6 | (v // 9 % 3) << 4 | (v // 3 % 3) << 2 | v % 3).to(torch.uint8).cuda()
        out = torch.zeros(n + 32, dtype=torch.uint8, device="cuda")
        for at in range(0, n, 1 << 26):
            m = min(n - at, 1 << 26)
            out[at:at + m] = codes[torch.randint(0, 81, (m,), generator=self.g, device="cuda")]
        scale = gain * (0.5 + 1.5 * torch.rand(1, generator=self.g, device="cuda"))
        out[n:n + 4] = scale.view(torch.uint8)
        return out


def _p(t, offset=0):
    return ctypes.c_void_p(t.data_ptr() + offset)


def _hp(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _block_shapes(shape):
    e, f = shape["n_embd"], shape["n_ff"]
    g = e // shape["n_head"] * shape["n_head_kv"]
    return {"wq": (e, e), "wk": (g, e), "wv": (g, e), "wo": (e, e), "w_gate": (f, e), "w_up": (f, e), "w_down": (e, f)}


def _model(case, seed):
    """The model's tensors on the GPU, and the case's tokens."""
    r, shape = _Rng(seed), SHAPES[case["shape"]]
    e, f = shape["n_embd"], shape["n_ff"]
    m = {"tok_embd": r.normal(case["vocab"], e, dtype=torch.float16), "output_norm": r.norm_weight(e), "layers": []}
    for _ in range(case["layers"]):
        layer = {n: r.ternary(rows, k, (2 * k / 3) ** -0.5) for n, (rows, k) in _block_shapes(shape).items()}
        for n, w in (("attn_norm", e), ("attn_sub_norm", e), ("ffn_norm", e), ("ffn_sub_norm", f)):
            layer[n] = r.norm_weight(w)
        m["layers"].append(layer)
    n_tok = case["tokens"] if case["kind"] == "score" else case["prompt"]
    return m, r.integers(case["vocab"], n_tok).cpu().numpy()


class _Decoder:
    """A loaded model with one context, freed with the object."""

    def __init__(self, case, seed):
        m, self.tokens = _model(case, seed)
        cfg = dict(SHAPES[case["shape"]], n_layer=case["layers"], n_vocab=case["vocab"], eps=EPS, rope_base=ROPE_BASE)
        host = {"cfg": cfg, "tok_embd": m["tok_embd"].view(torch.int16).cpu().numpy().view(np.uint16),
                "output_norm": m["output_norm"].cpu().numpy(),
                "layers": [{n: t.cpu().numpy() for n, t in layer.items()} for layer in m["layers"]]}
        self.decoder = amd.DeviceDecoder(device(), host, len(self.tokens) + case.get("new", 0) + 8)
        if case["kind"] == "generate":
            self.decoder.set_graph(True)

    def __del__(self):
        if hasattr(self, "decoder"):
            device().sync()
            self.decoder.close()


class _Plan:
    """A plan and the buffers it names, destroyed with the object."""

    def __init__(self, plan, run, destroy, keep):
        self.plan, self.run, self.destroy, self.keep = plan, run, destroy, keep

    def __del__(self):
        self.destroy(self.plan)


def _plan(case, seed):
    r, dev, shapes = _Rng(seed), device(), _block_shapes(SHAPES[case["shape"]])
    e, f = SHAPES[case["shape"]]["n_embd"], SHAPES[case["shape"]]["n_ff"]
    out = torch.empty(case["blocks"] * sum(n for n, _ in shapes.values()), device="cuda")
    keep, jobs, at = [out], [], 0
    for _ in range(case["blocks"]):
        xa, xo, xf, xd = r.normal(e), r.normal(e), r.normal(e), r.normal(f)
        keep += [xa, xo, xf, xd]
        for name, (n, k) in shapes.items():
            x = {"wo": xo, "w_gate": xf, "w_up": xf, "w_down": xd}.get(name, xa)
            w = r.ternary(n, k)
            keep.append(w)
            jobs.append(amd.GemvJob(w.data_ptr(), n, k, x.data_ptr(), None, None, out.data_ptr() + 4 * at, None))
            at += n
    torch.cuda.synchronize()
    return _Plan(dev.plan(jobs), dev.plan_run, dev.plan_destroy, keep)


def _gemm_plan(case, seed):
    r, dev, shapes, m = _Rng(seed), device(), _block_shapes(SHAPES[case["shape"]]), case["tokens"]
    names = ("w_gate", "w_up", "w_down")
    out = torch.empty(case["blocks"] * m * sum(shapes[n][0] for n in names), device="cuda")
    keep, jobs, at = [out], [], 0
    for _ in range(case["blocks"]):
        rows = {}
        for name in names:
            n, k = shapes[name]
            if k not in rows:
                x, q, act = r.normal(m, k), torch.empty(m, k, dtype=torch.int8, device="cuda"), torch.empty(m, 2, device="cuda")
                torch.cuda.synchronize()
                dev.quant_act(_p(x), k, m, _p(q), _p(act))
                dev.sync()
                rows[k] = (q, act)
            q, act = rows[k]
            w = r.ternary(n, k)
            keep += [w, q, act]
            jobs.append((w.data_ptr(), n, k, q.data_ptr(), act.data_ptr(), out.data_ptr() + 4 * at, None))
            at += m * n
    torch.cuda.synchronize()
    return _Plan(dev.gemm_plan(jobs, m), dev.gemm_plan_run, dev.gemm_plan_destroy, keep)


class _Row:
    """Host tensors registered with the kernel row, dropped with the object."""

    def __init__(self, case, seed):
        device()
        L, r, e, f = amd.lib(), _Rng(seed), case["embd"], case["ff"]
        amd.check(L.sllm_kdispatch_select(b"gfx950"), "kdispatch_select")
        self.x = [r.normal(e).cpu().numpy(), r.normal(f).cpu().numpy()]
        self.w, self.dots = [], []
        for n, k in ((f, e), (f, e), (e, f)):
            w = r.ternary(n, k).cpu().numpy()
            amd.check(L.sllm_gfx950_tensor_register(_hp(w), n, k), "tensor_register")
            self.w.append((w, n, k))
            self.dots.append(np.zeros(n, np.int32))
        self.q = [np.zeros(e, np.int8), np.zeros(f, np.int8)]
        self.act = [np.zeros(2, np.float32), np.zeros(2, np.float32)]
        self.L = L

    def run(self):
        L = self.L
        L.sllm_kdispatch_quant_act(_hp(self.x[0]), self.x[0].size, _hp(self.q[0]), _hp(self.act[0]))
        for (w, n, k), dots in zip(self.w[:2], self.dots):
            L.sllm_kdispatch_gemv(_hp(w), n, k, _hp(self.q[0]), _hp(dots))
        L.sllm_kdispatch_quant_act(_hp(self.x[1]), self.x[1].size, _hp(self.q[1]), _hp(self.act[1]))
        w, n, k = self.w[2]
        L.sllm_kdispatch_gemv(_hp(w), n, k, _hp(self.q[1]), _hp(self.dots[2]))
        return {"q": self.q, "act": [a.view(np.int32) for a in self.act], "dots": self.dots}

    def __del__(self):
        for w, _, _ in getattr(self, "w", []):
            amd.lib().sllm_gfx950_tensor_unregister(_hp(w))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        r, n, rows, k = _Rng(seed), case["calls"], case["rows"], case["k"]
        device()
        s = {"w": [r.ternary(rows, k) for _ in range(n)], "x": r.normal(n, k),
             "q": torch.empty(n, k, dtype=torch.int8, device="cuda"),
             "act": torch.empty(n, 2, dtype=torch.int32, device="cuda"),
             "out": [torch.empty(rows, device="cuda") for _ in range(n)]}
        s["args"] = [(_p(s["w"][i]), rows, k, _p(s["x"][i]), _p(s["q"][i]), _p(s["act"][i]), _p(s["out"][i]))
                     for i in range(n)]
    elif kind == "linear_batch":
        r, m = _Rng(seed), case["tokens"]
        device()
        s = {"w": r.ternary(case["rows"], case["k"]), "x": r.normal(m, case["k"]),
             "q": torch.empty(m, case["k"], dtype=torch.int8, device="cuda"),
             "act": torch.empty(m, 2, dtype=torch.int32, device="cuda"),
             "out": torch.empty(m, case["rows"], device="cuda")}
        s["args"] = (_p(s["w"]), case["rows"], case["k"], _p(s["x"]))
        s["ptrs"] = (_p(s["q"]), _p(s["act"]), _p(s["out"]))
    elif kind == "plan":
        s = {"plan": _plan(case, seed)}
    elif kind == "gemm_plan":
        s = {"plan": _gemm_plan(case, seed)}
    elif kind == "row":
        s = {"row": _Row(case, seed)}
    else:
        s = {"model": _Decoder(case, seed)}
    torch.cuda.synchronize()
    s["case"] = case
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        linear = device().linear
        for args in state["args"]:
            linear(*args)
        return {"q": state["q"], "act": state["act"], "out": state["out"]}
    if kind == "linear_batch":
        device().linear_batch(*state["args"], case["tokens"], *state["ptrs"])
        return {"q": state["q"], "act": state["act"], "out": state["out"]}
    if kind in ("plan", "gemm_plan"):
        p = state["plan"]
        p.run(p.plan)
        return p.keep[0]
    if kind == "row":
        return state["row"].run()
    d, tokens = state["model"].decoder, state["model"].tokens
    d.reset()
    if kind == "score":
        return d.forward_chunk(tokens, 0)
    if kind == "prefill":
        d.prefill_chunked(tokens[:-1], case["chunk"], logits=False)
        return d.forward(int(tokens[-1]), len(tokens) - 1)
    d.prefill_chunked(tokens, 512, logits=False)
    ids = d.generate([], case["new"])
    return {"ids": ids, "logits": d.forward(d.argmax(), d.n_past())}


# ---------------------------------------------------------------------------
# the work of a pass, and its result in 64 bits
# ---------------------------------------------------------------------------

def _proj(rows, k, m=1):
    """Weights, f32 rows in, f32 rows out; one multiply and add per weight and row."""
    return np.array([rows * k / 4 + 4 + 4 * m * (k + rows), 2 * rows * k * m])


def work(case):
    kind = case["kind"]
    if kind == "linear":
        w = case["calls"] * (_proj(case["rows"], case["k"]) + [case["k"] + 8, 0])
    elif kind == "linear_batch":
        m = case["tokens"]
        w = _proj(case["rows"], case["k"], m) + [m * (case["k"] + 8), 0]     # the int8 rows and their scales too
    elif kind == "plan":
        shape = SHAPES[case["shape"]]
        w = sum(_proj(n, k) for n, k in _block_shapes(shape).values())
        w = case["blocks"] * (w - [4 * 3 * shape["n_embd"], 0])              # Q, K, V share a row, gate and up another
    elif kind == "gemm_plan":
        shape, m = SHAPES[case["shape"]], case["tokens"]
        e, f = shape["n_embd"], shape["n_ff"]
        w = case["blocks"] * np.array([3 * (e * f / 4 + 4) + m * (e + f + 16) + 4 * m * (2 * f + e), 6 * e * f * m])
    elif kind == "row":
        e, f = case["embd"], case["ff"]
        w = np.array([3 * (e * f / 4) + 5 * (e + f) + 16 + 4 * (2 * f + e), 6 * e * f])
    else:
        shape = SHAPES[case["shape"]]
        e, hd = shape["n_embd"], shape["n_embd"] // shape["n_head"]
        i2s = case["layers"] * sum(n * k for n, k in _block_shapes(shape).values())
        kv = case["layers"] * 2 * shape["n_head_kv"] * hd * 4                # cache bytes of a position
        att = case["layers"] * 4 * e                                         # operations per (position, earlier position)
        head = case["vocab"] * e
        n = case["tokens"] if kind == "score" else case["prompt"]
        heads = n if kind == "score" else 1                                  # rows of logits
        # a chunk reads every weight once, each position its cache once per chunk after its own
        step = min(512, case.get("chunk", 512))
        chunks = -(-n // step)
        w = np.array([chunks * i2s / 4 + 2 * head + kv * (n + sum(range(step, n, step))) + 4 * heads * case["vocab"],
                      2 * i2s * n + att * n * (n + 1) / 2 + 2 * head * heads])
        for i in range(case.get("new", -1) + 1):                             # decoded tokens, each with its logits
            w = w + [i2s / 4 + 2 * head + kv * (n + i + 1), 2 * i2s + att * (n + i + 1) + 2 * head]
    return {"bytes": float(w[0]), "flops": float(w[1])}


def tolerance(case):
    return "exact"


def _codes(w, rows, k):
    """The ternary matrix in 64 bits, and its scale."""
    b = w[:rows * k // 4].view(rows, k // 128, 1, 32)
    c = torch.cat([(b >> s) & 3 for s in (6, 4, 2, 0)], dim=2)
    return c.reshape(rows, k).double() - 1, w[rows * k // 4:rows * k // 4 + 4].clone().view(torch.float32).double()


def _quantise(x):
    """Each row's int8 values and scale (127 over its largest magnitude, halves away from zero)."""
    amax = x.abs().amax(-1, keepdim=True)
    s = torch.where(amax > 0, 127 / amax, torch.zeros_like(amax))
    v = (x * s).double()
    return (torch.sign(v) * torch.floor(v.abs() + 0.5)).clamp(-128, 127), s.double()


def _project(x, w, rows, k):
    q, s = _quantise(x)
    c, scale = _codes(w, rows, k)
    return (q @ c.t()) * (scale / s)


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, n_rot):
    half = n_rot // 2
    ang = torch.arange(x.shape[0], device="cuda").double()[:, None] * ROPE_BASE ** (
        -2 * torch.arange(half, device="cuda").double() / n_rot)
    c, s = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = x[..., :half], x[..., half:n_rot]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., n_rot:]], dim=-1)


def _logits(case, seed):
    """Every position's final hidden row in 64 bits, and the output projection."""
    m, tokens = _model(case, seed)
    shape = SHAPES[case["shape"]]
    dims, nh, nkv = _block_shapes(shape), shape["n_head"], shape["n_head_kv"]
    hd, n = shape["n_embd"] // nh, len(tokens)
    x = m["tok_embd"][torch.from_numpy(tokens).cuda().long()].double()
    mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
    for layer in m["layers"]:
        lin = lambda v, name: _project(v, layer[name], *dims[name])  # noqa: E731
        h = _norm(x, layer["attn_norm"])
        q = _rope(lin(h, "wq").view(n, nh, hd), shape["n_rot"])
        k = _rope(lin(h, "wk").view(n, nkv, hd), shape["n_rot"])
        v = lin(h, "wv").view(n, nkv, hd)
        heads = []
        for i in range(nh):
            g = i // (nh // nkv)
            sc = (q[:, i] @ k[:, g].t()) / math.sqrt(hd)
            heads.append(torch.softmax(sc.masked_fill(mask, -math.inf), -1) @ v[:, g])
        x = x + lin(_norm(torch.cat(heads, -1), layer["attn_sub_norm"]), "wo")
        h = _norm(x, layer["ffn_norm"])
        gate = lin(h, "w_gate")
        x = x + lin(_norm(gate * torch.sigmoid(gate) * lin(h, "w_up"), layer["ffn_sub_norm"]), "w_down")
    return _norm(x, m["output_norm"]), m["tok_embd"]


def exact(case, seed):
    kind = case["kind"]
    if kind == "generate":
        return None                         # each token it picks decides all that follow
    if kind == "linear":
        r, n, rows, k = _Rng(seed), case["calls"], case["rows"], case["k"]
        w, x = [r.ternary(rows, k) for _ in range(n)], r.normal(n, k)
        return {"q": None, "act": None, "out": [_project(x[i:i + 1], w[i], rows, k)[0] for i in range(n)]}
    if kind == "linear_batch":
        r, m = _Rng(seed), case["tokens"]
        w, x = r.ternary(case["rows"], case["k"]), r.normal(m, case["k"])
        return {"q": None, "act": None, "out": _project(x, w, case["rows"], case["k"])}
    if kind == "plan":
        r, shapes, shape = _Rng(seed), _block_shapes(SHAPES[case["shape"]]), SHAPES[case["shape"]]
        out = []
        for _ in range(case["blocks"]):
            xa, xo, xf, xd = (r.normal(n) for n in (shape["n_embd"],) * 3 + (shape["n_ff"],))
            for name, (n, k) in shapes.items():
                x = {"wo": xo, "w_gate": xf, "w_up": xf, "w_down": xd}.get(name, xa)
                out.append(_project(x[None], r.ternary(n, k), n, k).view(-1))
        return torch.cat(out)
    if kind == "gemm_plan":
        r, shapes, out = _Rng(seed), _block_shapes(SHAPES[case["shape"]]), []
        for _ in range(case["blocks"]):
            rows = {}
            for name in ("w_gate", "w_up", "w_down"):
                n, k = shapes[name]
                if k not in rows:
                    rows[k] = r.normal(case["tokens"], k)
                out.append(_project(rows[k], r.ternary(n, k), n, k).view(-1))
        return torch.cat(out)
    if kind == "row":
        return None                         # whole numbers only
    x, embd = _logits(case, seed)
    if kind == "prefill":
        return (x[-1:] @ embd.double().t())[0]
    return x @ embd.double().t()
