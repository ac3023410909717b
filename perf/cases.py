"""The work that programs built on this library do, as cases to be timed.

A case is one call (or the few calls of one phase) through the public entry
points of `chat-wgpu_amd/cw.py` and the C ABI below it:

  * ``gemv``      one decode projection (q4::gemv);
  * ``gemm``      one projection of several positions at once;
  * ``attention`` one decode attention over a KV cache;
  * ``prefill``   the prompt phase of a model over a few layers;
  * ``decode``    the replayed decode loop of a model over a few layers;
  * ``generate``  model::generate, the prompt and the reply in one call.

Widths are those of the Qwen3-8B and Qwen3-0.6B configurations that the tests
and the benchmark run; the models hold one to four of their layers, which
repeat.  Weights, activations and caches have the distributions of the
library's own synthetic model: uniform nibbles under half-normal block
scales, unit-normal activations and cache rows, gains near one.
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (os.getcwd(), _ROOT):
    if os.path.isdir(os.path.join(_p, "chat-wgpu_amd")):
        sys.path.insert(0, os.path.join(_p, "chat-wgpu_amd"))
        break
import cw  # noqa: E402

EPS, THETA = 1e-6, 1e6

# layer widths: dim, n_heads, n_kv_heads, hidden (head_dim 128)
SHAPES = {
    "8b": (4096, 32, 8, 12288),
    "0.6b": (1024, 16, 8, 3072),
}
HD = 128


def listed():
    return [
        # the single 3072 x 1024 projection: the smallest launch, all latency
        {"name": "gemv_3072x1024", "kind": "gemv", "in_f": 1024, "out_f": 3072},
        # a short chat turn (16 tokens) through one wide 8B projection
        {"name": "gemm_16_4096_12288", "kind": "gemm", "m": 16, "in_f": 4096, "out_f": 12288},
        # a ragged prompt through the 8B down projection's long rows
        {"name": "gemm_100_12288_4096", "kind": "gemm", "m": 100, "in_f": 12288, "out_f": 4096},
        # the benchmark's 512-token prompt through the QKV projection
        {"name": "gemm_512_4096_6144", "kind": "gemm", "m": 512, "in_f": 4096, "out_f": 6144},
        # decode attention of the 8B workload: 4 K positions of an f16 cache
        {"name": "attn_f16_4097", "kind": "attention", "kv": "f16", "heads": 32, "kv_heads": 8,
         "head_dim": 128, "seq": 4097},
        # decode attention late in a long 0.6B chat: an f32 cache
        {"name": "attn_f32_2001", "kind": "attention", "kv": "f32", "heads": 16, "kv_heads": 8,
         "head_dim": 128, "seq": 2001},
        # a short user turn after an earlier conversation (8B, two layers)
        {"name": "prefill_8b_24_at_700", "kind": "prefill", "shape": "8b", "kv": "f16",
         "layers": 2, "n": 24, "start": 700, "vocab": 4096},
        # the benchmark's prompt phase (8B, two layers, 512 tokens)
        {"name": "prefill_8b_512", "kind": "prefill", "shape": "8b", "kv": "f16", "layers": 2,
         "n": 512, "start": 0, "vocab": 4096},
        # a long document as the prompt (8B, one layer), the largest call
        {"name": "prefill_8b_3000", "kind": "prefill", "shape": "8b", "kv": "f16", "layers": 1,
         "n": 3000, "start": 0, "vocab": 4096},
        # a chat prompt on the small model, whose cache is f32 by default
        {"name": "prefill_0.6b_128_f32", "kind": "prefill", "shape": "0.6b", "kv": "f32",
         "layers": 4, "n": 128, "start": 0, "vocab": 4096},
        # eight replayed decode steps of the 8B workload at 4 K positions
        {"name": "decode_8b_at_4096", "kind": "decode", "shape": "8b", "kv": "f16", "layers": 2,
         "n": 8, "start": 4096, "vocab": 4096},
        # model::generate on the small model: 32 prompt tokens, 32 new ones
        {"name": "generate_0.6b_32_32", "kind": "generate", "shape": "0.6b", "kv": "f32",
         "layers": 4, "n": 32, "new": 32, "start": 0, "vocab": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: projection widths from the two configurations or any
    multiple of 32, row counts and positions spread over their logarithm."""
    kind = rng.choice(["gemv", "gemm", "gemm", "attention", "prefill", "prefill", "decode",
                       "generate"])
    if kind == "gemv":
        return {"kind": kind, "in_f": rng.choice([1024, 2048, 3072, 4096, 12288,
                                                  32 * rng.randint(8, 200)]),
                "out_f": rng.choice([1024, 4096, 6144, _log(rng, 100, 40000)])}
    if kind == "gemm":
        k = rng.choice([1024, 2048, 3072, 4096, 12288, 32 * rng.randint(8, 200)])
        n = rng.choice([1024, 3072, 4096, 6144, 12288, _log(rng, 200, 8000)])
        return {"kind": kind, "m": _log(rng, 2, 1500), "in_f": k, "out_f": n}
    if kind == "attention":
        heads, kv_heads = rng.choice([(32, 8), (16, 8), (16, 2), (8, 8)])
        return {"kind": kind, "kv": rng.choice(["f16", "f32"]), "heads": heads,
                "kv_heads": kv_heads, "head_dim": rng.choice([128, 128, 128, 64]),
                "seq": _log(rng, 1, 20000)}
    shape = rng.choice(["8b", "0.6b"])
    kv = rng.choice(["f16", "f32"])
    layers = 1 if shape == "8b" else rng.randint(1, 3)
    if kind == "prefill":
        n = _log(rng, 2, 1200)
        if kv == "f32":
            n = min(n, 500)
        return {"kind": kind, "shape": shape, "kv": kv, "layers": layers, "n": n,
                "start": rng.choice([0, 0, _log(rng, 5, 3000)]), "vocab": 4096}
    if kind == "decode":
        return {"kind": kind, "shape": shape, "kv": kv, "layers": layers,
                "n": rng.randint(2, 16), "start": _log(rng, 1, 6000), "vocab": 4096}
    return {"kind": kind, "shape": shape, "kv": kv, "layers": layers, "n": _log(rng, 2, 120),
            "new": rng.randint(2, 32), "start": 0, "vocab": 4096}


# ------------------------------------------------------------------ inputs

_CTX = None


def _ctx():
    global _CTX
    if _CTX is None:
        _CTX = cw.Context(0)
    return _CTX


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _q4(g, out_f, in_f):
    """Block scales f16 [out, in/32] (half-normal, 0.02) and quants [out, in/32, 16]."""
    nb = in_f // 32
    s = (torch.randn(out_f, nb, generator=g, device="cuda") * 0.02).abs().half()
    q = torch.randint(0, 256, (out_f, nb, 16), generator=g, device="cuda", dtype=torch.uint8)
    return s, q


def _dequant(s, q):
    """The weights d (q - 8) in 64 bits: low nibbles first, then the high ones."""
    w = torch.cat([(q & 15), (q >> 4)], dim=2).double() - 8.0
    return (w * s.double().unsqueeze(2)).reshape(s.shape[0], -1)


def _kv_type(case):
    return torch.float16 if case["kv"] == "f16" else torch.float32


def _op_inputs(case, seed):
    g = _gen(seed)
    if case["kind"] == "attention":
        h, kvh, hd, seq = case["heads"], case["kv_heads"], case["head_dim"], case["seq"]
        q = torch.randn(h * hd, generator=g, device="cuda")
        k = torch.randn(seq, kvh * hd, generator=g, device="cuda").to(_kv_type(case))
        v = torch.randn(seq, kvh * hd, generator=g, device="cuda").to(_kv_type(case))
        return q, k, v
    s, q = _q4(g, case["out_f"], case["in_f"])
    x = torch.randn(case.get("m", 1), case["in_f"], generator=g, device="cuda")
    return x, s, q


def _proj_shapes(shape):
    dim, h, kvh, hidden = SHAPES[shape]
    return {"attn_q": (h * HD, dim), "attn_k": (kvh * HD, dim), "attn_v": (kvh * HD, dim),
            "attn_output": (dim, h * HD), "ffn_gate": (hidden, dim), "ffn_up": (hidden, dim),
            "ffn_down": (dim, hidden)}


def _model_inputs(case, seed):
    """The tensors of a model by their names, prompt tokens, and the cache
    rows before the start position ([layer][pos][kv_dim], or None)."""
    g = _gen(seed)
    dim, _, kvh, _ = SHAPES[case["shape"]]

    def gain(n):
        return 1.0 + 0.02 * torch.randn(n, generator=g, device="cuda")

    w = {}
    for i in range(case["layers"]):
        for name, n in (("attn_norm", dim), ("attn_q_norm", HD), ("attn_k_norm", HD),
                        ("ffn_norm", dim)):
            w[f"blk.{i}.{name}.weight"] = gain(n)
        for name, (out_f, in_f) in _proj_shapes(case["shape"]).items():
            w[f"blk.{i}.{name}.weight"] = _q4(g, out_f, in_f)
    w["output_norm.weight"] = gain(dim)
    w["token_embd.weight"] = 0.02 * torch.randn(case["vocab"], dim, generator=g, device="cuda")
    w["output.weight"] = _q4(g, case["vocab"], dim)
    tokens = torch.randint(0, case["vocab"], (case["n"],), generator=g, device="cuda")
    kv = None
    if case["start"]:
        kv = [torch.randn(case["layers"], case["start"], kvh * HD, generator=g,
                          device="cuda").to(_kv_type(case)) for _ in range(2)]
    return w, tokens, kv


def _positions(case):
    """Cache positions of the model: what the case fills and the next token,
    rounded up to a multiple of 256."""
    return (case["start"] + case["n"] + case.get("new", 0) + 256) // 256 * 256


class _State:
    """Device tensors of a call, or a loaded model, and the buffers it fills."""

    def __init__(self, case, seed):
        self.case, self.model = case, None
        ctx = _ctx()

        def dev(t):
            return cw.DeviceArray(ctx, tuple(t.shape), np.uint8, t.data_ptr())

        kind = case["kind"]
        if kind in ("gemv", "gemm", "attention"):
            self.inputs = _op_inputs(case, seed)
            rows = case["heads"] * case["head_dim"] if kind == "attention" else \
                case.get("m", 1) * case["out_f"]
            self.y = torch.empty(rows, device="cuda")
            self.dev = [dev(t) for t in self.inputs] + [dev(self.y)]
            return
        w, tokens, kv = _model_inputs(case, seed)
        dim, h, kvh, hidden = SHAPES[case["shape"]]
        cfg = cw.make_config(case["layers"], dim, h, kvh, HD, hidden, case["vocab"],
                             _positions(case), cw.CW_F16 if case["kv"] == "f16" else cw.CW_F32,
                             EPS, THETA)
        self.model = cw.Model(ctx, cfg)
        self.model.set_weights({
            n: (t[0].cpu().numpy().view(np.uint16), t[1].cpu().numpy())
            if isinstance(t, tuple) else t.cpu().numpy() for n, t in w.items()})
        self.model.finalize()
        if kv is not None:
            self.model.prefill_kv(kv[0].cpu().numpy(), kv[1].cpu().numpy(), case["start"])
        self.tokens = tokens.cpu().numpy().astype(np.uint32)

    def __del__(self):
        if self.model is not None:
            self.model.close()


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    case, ctx = state.case, _ctx()
    kind = case["kind"]
    if kind == "gemv":
        x, s, q, y = state.dev
        ctx.q4_gemv(x, s, q, case["in_f"], case["out_f"], y=y)
        return state.y
    if kind == "gemm":
        x, s, q, y = state.dev
        ctx.q4_gemm(x, case["m"], s, q, case["in_f"], case["out_f"], y=y)
        return state.y
    if kind == "attention":
        q, k, v, y = state.dev
        cw.check(cw.lib().cw_attention(ctx.h, q.ptr, k.ptr, v.ptr,
                                       cw.CW_F16 if case["kv"] == "f16" else cw.CW_F32,
                                       case["heads"], case["kv_heads"], case["seq"],
                                       case["head_dim"], y.ptr))
        return state.y
    m = state.model
    if kind == "prefill":
        token = m.prefill(state.tokens, start_pos=case["start"])
        return {"logits": m.logits(), "hidden": m.hidden(), "token": token}
    if kind == "decode":
        m.reset_state(state.tokens[0], case["start"])
        m.decode_async(case["n"])
        tokens = m.tokens(case["n"])
        return {"logits": m.logits(), "tokens": tokens.astype(np.int64)}
    tokens = m.generate(state.tokens, case["new"], start_pos=case["start"])
    return {"logits": m.logits(), "tokens": tokens.astype(np.int64)}


# --------------------------------------------------------- floors and results

def _q4_bytes(out_f, in_f):
    return out_f * (in_f // 32) * 18


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        m, k, n = case.get("m", 1), case["in_f"], case["out_f"]
        return {"bytes": _q4_bytes(n, k) + 4 * m * (k + n), "flops": 2 * m * n * k}
    es = 2 if case["kv"] == "f16" else 4
    if kind == "attention":
        h, kvh, hd, seq = case["heads"], case["kv_heads"], case["head_dim"], case["seq"]
        return {"bytes": 2 * seq * kvh * hd * es + 8 * h * hd, "flops": 4 * h * hd * seq}
    dim, h, kvh, _ = SHAPES[case["shape"]]
    shapes = _proj_shapes(case["shape"]).values()
    params = case["layers"] * sum(o * i for o, i in shapes)
    layer_bytes = case["layers"] * sum(_q4_bytes(o, i) for o, i in shapes)
    head_bytes = _q4_bytes(case["vocab"], dim) + 4 * case["vocab"]
    head_flops = 2 * case["vocab"] * dim
    row = 2 * case["layers"] * kvh * HD * es  # K and V of one position

    def attn_flops(first, n):
        return case["layers"] * 4 * h * HD * sum(range(first + 1, first + n + 1))

    n, start = case["n"], case["start"]
    if kind == "decode":
        reads = sum(range(start + 1, start + n + 1)) * row
        return {"bytes": n * (layer_bytes + head_bytes) + reads,
                "flops": n * (2 * params + head_flops) + attn_flops(start, n)}
    prompt = {"bytes": layer_bytes + head_bytes + (start + n) * row + 4 * n * dim,
              "flops": 2 * n * params + head_flops + attn_flops(start, n)}
    if kind == "prefill":
        return prompt
    more = case["new"] - 1
    reads = sum(range(n + 1, n + more + 1)) * row
    return {"bytes": prompt["bytes"] + more * (layer_bytes + head_bytes) + reads,
            "flops": prompt["flops"] + more * (2 * params + head_flops) + attn_flops(n, more)}


def tolerance(case):
    """Four times what 32-bit sums in another order show, or the f16 rounding
    of cache rows that lie on either side of a tie."""
    if case["kind"] in ("gemv", "gemm", "attention"):
        return {"rel": 2e-6, "max": 2e-5}
    if case["kv"] == "f32":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 2e-4, "max": 2e-3}


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


class _Exact:
    """The forward of the case's model in 64 bits, its cache rounded to the cache's type."""

    def __init__(self, case, seed):
        self.case = case
        w, self.tokens, kv = _model_inputs(case, seed)
        self.w = {n: _dequant(*t) if isinstance(t, tuple) else t.double() for n, t in w.items()}
        kvh = SHAPES[case["shape"]][2]
        total = _positions(case)
        self.kv = [torch.zeros(case["layers"], total, kvh * HD, device="cuda",
                               dtype=torch.float64) for _ in range(2)]
        if kv is not None:
            for dst, src in zip(self.kv, kv):
                dst[:, :case["start"]] = src.double()

    def _rope(self, x, start):
        i = torch.arange(HD // 2, device="cuda", dtype=torch.float64)
        pos = torch.arange(start, start + x.shape[0], device="cuda", dtype=torch.float64)
        a = pos[:, None] * THETA ** (-2.0 * i / HD)
        c, s = a.cos()[:, None], a.sin()[:, None]
        lo, hi = x[..., :HD // 2], x[..., HD // 2:]
        return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)

    def forward(self, tokens, start):
        """Logits and normed hidden state of the last of `tokens` from `start` on."""
        case, w = self.case, self.w
        dim, h, kvh, _ = SHAPES[case["shape"]]
        n = tokens.shape[0]
        x = w["token_embd.weight"][tokens]
        for i in range(case["layers"]):
            def t(name):
                return w[f"blk.{i}.{name}.weight"]
            y = _rms(x, t("attn_norm"))
            q = self._rope(_rms((y @ t("attn_q").T).reshape(n, h, HD), t("attn_q_norm")), start)
            k = self._rope(_rms((y @ t("attn_k").T).reshape(n, kvh, HD), t("attn_k_norm")), start)
            v = y @ t("attn_v").T
            for dst, src in zip(self.kv, (k.reshape(n, -1), v)):
                dst[i, start:start + n] = src.to(_kv_type(case)).double()
            end = start + n
            keys = self.kv[0][i, :end].reshape(end, kvh, HD)
            vals = self.kv[1][i, :end].reshape(end, kvh, HD)
            mask = torch.arange(end, device="cuda")[None] > \
                torch.arange(start, end, device="cuda")[:, None]
            o = torch.empty(n, h, HD, device="cuda", dtype=torch.float64)
            for a in range(h):
                g = a // (h // kvh)
                sc = (q[:, a] @ keys[:, g].T) * HD ** -0.5
                p = sc.masked_fill(mask, -math.inf).softmax(-1)
                o[:, a] = p @ vals[:, g]
            x = x + o.reshape(n, -1) @ t("attn_output").T
            y = _rms(x, t("ffn_norm"))
            gate = y @ t("ffn_gate").T
            x = x + (gate * torch.sigmoid(gate) * (y @ t("ffn_up").T)) @ t("ffn_down").T
        hidden = _rms(x[-1], w["output_norm.weight"])
        return w["output.weight"] @ hidden, hidden


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        x, s, q = _op_inputs(case, seed)
        return (x.double() @ _dequant(s, q).T).reshape(-1)
    if kind == "attention":
        q, k, v = (t.double() for t in _op_inputs(case, seed))
        h, kvh, hd, seq = case["heads"], case["kv_heads"], case["head_dim"], case["seq"]
        k, v = k.reshape(seq, kvh, hd), v.reshape(seq, kvh, hd)
        out = []
        for a in range(h):
            g = a // (h // kvh)
            p = (k[:, g] @ q.reshape(h, hd)[a] * hd ** -0.5).softmax(0)
            out.append(p @ v[:, g])
        return torch.cat(out)
    e = _Exact(case, seed)
    if kind == "prefill":
        logits, hidden = e.forward(e.tokens, case["start"])
        return {"logits": logits, "hidden": hidden, "token": None}
    if kind == "decode":
        token, pos, steps = e.tokens[:1], case["start"], case["n"]
    else:
        logits, _ = e.forward(e.tokens, case["start"])
        token, pos, steps = logits.argmax().reshape(1), case["start"] + case["n"], case["new"] - 1
    for i in range(steps):
        logits, _ = e.forward(token, pos + i)
        token = logits.argmax().reshape(1)
    return {"logits": logits, "tokens": None}
