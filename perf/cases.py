"""What the backend's speed is measured on: calls a program makes through
`technograd_amd.hip`, on device buffers unless a case says otherwise.

A case is a dict of plain values; "kind" says which call it is:

  linear    Program.batch_device of one quantized layer W @ x (int4 or int8
            weights), from one row (the matvec of a lone request) to full
            batches; "exact" loads it with EXACT, the reference's own f32 order
  mlp       the same for a whole model: matmul, tanh, matmul, tanh, matmul,
            rmsnorm; "host" hands numpy rows to Program.batch instead (what
            `tgc-hip batch` and a Python caller do); "fixed" runs the model in
            Q16.16 (`--fixed`)
  reasoner  a think loop with a halting step per row, in Q16.16 or f32
  ssm       a selective-SSM sequence classifier (its scan, projections, gates)
  forward   a Qwen3-shaped decoder at one fixed length: the logits of each
            sequence's last position, as `tgc batch` runs an imported model
  generate  Decoder.generate_device: a prompt, then greedy tokens over the KV
            cache; one step is a prefill, many are decoding

Weights are random, quantized per output channel by the library's own RTN
quantizer. A loaded model is kept between states of one shape (a program loads
its model once and feeds it rows); inputs come from the seed alone.
"""
import collections
import math
import os
import tempfile

import numpy as np
import torch

from technograd_amd import hip, synth

DEV = "cuda"

# A Qwen3-0.6B-shaped block (hidden 1024, 16 / 8 heads of 128, SwiGLU 3072); few layers and a smaller vocabulary keep
# one call, and the model's loading, short, with the head and the layers in about the full model's proportion.
QWEN = {"D": 1024, "NQ": 16, "NKV": 8, "HD": 128, "FF": 3072}


def listed():
    return [
        # one request through one int4 layer: latency, the weight read once
        {"name": "linear one row", "kind": "linear", "rows": 1, "k": 4096, "c": 4096, "bits": 4, "exact": False},
        # an odd-sized int8 layer on a middling batch (a server's gathered requests)
        {"name": "linear ragged", "kind": "linear", "rows": 203, "k": 1500, "c": 3001, "bits": 8, "exact": False},
        # the benchmark's layer at its largest batch
        {"name": "linear large", "kind": "linear", "rows": 4096, "k": 4096, "c": 4096, "bits": 4, "exact": False},
        # the reference's bits on request: its sequential f32 sums
        {"name": "linear exact", "kind": "linear", "rows": 333, "k": 1024, "c": 1000, "bits": 8, "exact": True},
        # the benchmark's MLP over a whole file of rows
        {"name": "mlp", "kind": "mlp", "rows": 65536, "d": 512, "h": 2048, "out": 512, "bits": 8, "host": False, "fixed": False},
        # the same model fed from and read back to ordinary host arrays
        {"name": "mlp host", "kind": "mlp", "rows": 8192, "d": 512, "h": 2048, "out": 512, "bits": 8, "host": True, "fixed": False},
        # a model of ordinary widths in Q16.16
        {"name": "mlp fixed", "kind": "mlp", "rows": 16384, "d": 64, "h": 256, "out": 16, "bits": 8, "host": False, "fixed": True},
        # the latent reasoner over a million rows, each halting when it has converged
        {"name": "reasoner", "kind": "reasoner", "rows": 1048576, "fixed": True},
        # the SSM classifier at its published widths, a batch of long sequences
        {"name": "ssm", "kind": "ssm", "rows": 512, "t": 512, "d": 256, "state": 16, "blocks": 4},
        # scoring sequences with the imported model at its fixed length
        {"name": "forward", "kind": "forward", "rows": 16, "t": 384, "layers": 2, "vocab": 20000},
        # a batch of prompts up to the first token
        {"name": "prefill", "kind": "generate", "seqs": 16, "prompt": 512, "steps": 1, "layers": 4, "vocab": 20000},
        # a batch of running conversations, token by token
        {"name": "decode", "kind": "generate", "seqs": 48, "prompt": 200, "steps": 64, "layers": 4, "vocab": 20000},
    ]


def _log(rng, lo, hi, step=1):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, v // step * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear exact", "mlp", "mlp host", "mlp fixed", "reasoner", "ssm", "forward", "prefill", "decode"])
    if kind == "linear":
        return {"kind": "linear", "rows": _log(rng, 1, 4096), "k": rng.randint(256, 4096), "c": rng.randint(256, 4096),
                "bits": rng.choice([4, 8]), "exact": False}
    if kind == "linear exact":
        return {"kind": "linear", "rows": _log(rng, 1, 512), "k": rng.randint(200, 1024), "c": rng.randint(200, 1024),
                "bits": rng.choice([4, 8]), "exact": True}
    if kind == "mlp":
        return {"kind": "mlp", "rows": _log(rng, 1, 65536), "d": rng.randint(64, 512), "h": rng.randint(256, 2048), "out": rng.randint(10, 512),
                "bits": rng.choice([4, 8]), "host": False, "fixed": False}
    if kind == "mlp host":
        return {"kind": "mlp", "rows": _log(rng, 1, 8192), "d": rng.randint(64, 512), "h": rng.randint(256, 2048), "out": rng.randint(10, 512),
                "bits": rng.choice([4, 8]), "host": True, "fixed": False}
    if kind == "mlp fixed":
        return {"kind": "mlp", "rows": _log(rng, 1, 16384), "d": rng.randint(48, 96), "h": rng.randint(128, 256), "out": rng.randint(8, 32),
                "bits": rng.choice([4, 8]), "host": False, "fixed": True}
    if kind == "reasoner":
        return {"kind": "reasoner", "rows": _log(rng, 256, 1048576), "fixed": rng.random() < 0.5}
    if kind == "ssm":
        return {"kind": "ssm", "rows": _log(rng, 1, 512), "t": rng.randint(32, 512), "d": 16 * rng.randint(4, 16), "state": rng.choice([8, 16]),
                "blocks": rng.randint(1, 4)}
    if kind == "forward":
        return {"kind": "forward", "rows": _log(rng, 1, 16), "t": rng.randint(16, 384), "layers": rng.randint(1, 2), "vocab": 20000}
    if kind == "prefill":
        return {"kind": "generate", "seqs": _log(rng, 1, 16), "prompt": rng.randint(16, 512), "steps": 1, "layers": 4, "vocab": 20000}
    return {"kind": "generate", "seqs": _log(rng, 1, 48), "prompt": _log(rng, 8, 200), "steps": rng.randint(8, 64), "layers": 4, "vocab": 20000}


# ---- models ----

_models = collections.OrderedDict()  # loaded models by shape, the last few
_dir = tempfile.TemporaryDirectory(prefix="tg_cases_")  # weight files of the models being loaded
_qwen_files = {}


def _cached(key, make, keep=4):
    if key in _models:
        _models.move_to_end(key)
    else:
        _models[key] = make()
        while len(_models) > keep:
            _models.popitem(last=False)
    return _models[key]


def _weight(seed, rows, cols, sigma):
    g = np.random.default_rng([seed, rows, cols])
    return (g.standard_normal((rows, cols), np.float32) * np.float32(sigma))


def _param(name, w, bits, axis):
    """A quantized param's TGIR text, its codes and scales in files, and its f64 values."""
    codes, scales = hip.quantize_rtn(w, bits, axis)
    base = os.path.join(_dir.name, name)
    codes.tofile(base + ".codes")
    scales.tofile(base + ".scale")
    text = "  (param %s (f32 %d %d)\n    (quant %d %d (scale-file %s.scale) (codes-file %s.codes)))\n" % (
        name, w.shape[0], w.shape[1], bits, axis, base, base)
    return text, (codes, scales, axis)


def _f64(q):
    codes, scales, axis = q
    s = torch.from_numpy(scales).to(DEV, torch.float64)
    return torch.from_numpy(codes).to(DEV, torch.float64) * (s[:, None] if axis == 0 else s[None, :])


def _linear_model(case):
    t, q = _param("W", _weight(11, case["c"], case["k"], 0.02), case["bits"], 0)
    text = "(tgir 1\n  (model linear)\n%s  (input x (f32 %d))\n  (block\n    (%%0 (f32 %d) (matmul W x))\n  )\n  (output %%0))\n" % (
        t, case["k"], case["c"])
    return hip.Program(text, flags=hip.EXACT if case["exact"] else 0, max_rows=case["rows"]), (q,)


def _mlp_model(case):
    d, h, out = case["d"], case["h"], case["out"]
    p = [_param(n, _weight(s, r, c, 1.5 / math.sqrt(c)), case["bits"], 0) for n, s, r, c in (("W1", 21, h, d), ("W2", 22, h, h), ("W3", 23, out, h))]
    text = ("(tgir 1\n  (model mlp)\n%s  (input x (f32 %d))\n  (block\n    (%%0 (f32 %d) (matmul W1 x))\n    (%%1 (f32 %d) (tanh %%0))\n"
            "    (%%2 (f32 %d) (matmul W2 %%1))\n    (%%3 (f32 %d) (tanh %%2))\n    (%%4 (f32 %d) (matmul W3 %%3))\n"
            "    (%%5 (f32 %d) (rmsnorm %%4))\n  )\n  (output %%5))\n" % ("".join(t for t, _ in p), d, h, h, h, h, out, out))
    return hip.Program(text, flags=hip.FIXED if case["fixed"] else 0, max_rows=case["rows"]), [q for _, q in p]


def _ssm_shapes(case):
    d, di, n, r = case["d"], 2 * case["d"], case["state"], 16
    shapes = []
    for _ in range(case["blocks"]):
        shapes += [(d, di), (d, di), (di, r), (r, di), (di, n), (di, n), (di, d)]
    return shapes + [(d, 8)]


def _ssm_model(case):
    text = synth.ssm_tgir(d_model=case["d"], d_inner=2 * case["d"], n_state=case["state"], dt_rank=16, T=case["t"], blocks=case["blocks"])
    return hip.Program(text, max_rows=case["rows"]), None


def _qwen_dir(case):
    """The weight files of one Qwen3-shaped model, shared by its fixed-length programs and its decoder's."""
    key = (case["layers"], case["vocab"])
    if key not in _qwen_files:
        _qwen_files[key] = (tempfile.TemporaryDirectory(prefix="tg_cases_"), {})
    return _qwen_files[key]


def _qwen_text(case, t, rope_len=None):
    where, cache = _qwen_dir(case)
    return synth.qwen3_tgir(L=case["layers"], V=case["vocab"], T=t, files=where.name, quantizer=hip.quantize_rtn, rope_len=rope_len, cache=cache, **QWEN)


def _forward_model(case):
    return hip.Program(_qwen_text(case, case["t"]), max_rows=case["rows"]), None


def _generate_model(case):
    length = case["prompt"] + case["steps"]
    prog = hip.Program(_qwen_text(case, 8, rope_len=length), max_rows=1)
    return hip.Decoder(prog, case["seqs"], case["prompt"], length), None


def _reasoner_model(case):
    return hip.Program(synth.latent_reasoner_tgir(), flags=hip.FIXED if case["fixed"] else 0, max_rows=case["rows"]), None


_MAKE = {"linear": _linear_model, "mlp": _mlp_model, "ssm": _ssm_model, "forward": _forward_model, "generate": _generate_model,
         "reasoner": _reasoner_model}


def _model(case):
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    return _cached(key, lambda: _MAKE[case["kind"]](case))


# ---- a pass ----

def _inputs(case, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    kind = case["kind"]
    if kind == "linear":
        return torch.randn(case["rows"], case["k"], generator=g, device=DEV)
    if kind == "mlp":
        x = torch.randn(case["rows"], case["d"], generator=g, device=DEV)
        if case["fixed"]:
            return torch.round(x * 65536).to(torch.int32)
        return x.cpu().numpy() if case["host"] else x
    if kind == "reasoner":  # bits, as the model's vocabulary has them
        x = torch.randint(0, 2, (case["rows"], 8), generator=g, device=DEV)
        return (x * 65536).to(torch.int32) if case["fixed"] else x.float()
    if kind == "ssm":
        return torch.randn(case["rows"], case["t"] * case["d"], generator=g, device=DEV)
    n, t = (case["rows"], case["t"]) if kind == "forward" else (case["seqs"], case["prompt"])
    return torch.randint(0, case["vocab"], (n, t), generator=g, device=DEV).float()


def prepare(case, seed):
    hip.init(0)
    model = _model(case)[0]
    s = {"kind": case["kind"], "host": case.get("host", False), "model": model, "x": _inputs(case, seed)}
    if case["kind"] == "generate":
        s["tokens"] = torch.zeros(case["seqs"], case["steps"], dtype=torch.int32, device=DEV)
        s["logits"] = torch.zeros(case["steps"], case["seqs"], case["vocab"], device=DEV)
        s["case"] = (case["seqs"], case["prompt"], case["steps"])
    elif not s["host"]:
        fixed = case.get("fixed", False)
        s["out"] = torch.zeros(case["rows"], model.nout, dtype=torch.int32 if fixed else torch.float32, device=DEV)
        if model.nthink:
            s["steps"] = torch.zeros(case["rows"], model.nthink, dtype=torch.int32, device=DEV)
    torch.cuda.synchronize()  # the inputs are there before the library's own stream reads them
    return s


def run(s):
    m = s["model"]
    if s["kind"] == "generate":
        seqs, prompt, steps = s["case"]
        m.generate_device(s["x"].data_ptr(), seqs, prompt, steps, s["tokens"].data_ptr(), s["logits"].data_ptr())
        return {"tokens": s["tokens"], "logits": s["logits"]}
    if s["host"]:
        return m.batch(s["x"])[0]
    steps = s.get("steps")
    m.batch_device(s["x"].data_ptr(), s["x"].shape[0], s["out"].data_ptr(), None if steps is None else steps.data_ptr())
    return s["out"] if steps is None else {"out": s["out"], "steps": steps}


# ---- what a pass cannot do without ----

def _qwen_macs(case):
    """multiply-adds and int4 weight bytes of one position of one layer, and of the head"""
    q = QWEN
    layer = q["D"] * (q["NQ"] + 2 * q["NKV"]) * q["HD"] + q["NQ"] * q["HD"] * q["D"] + 3 * q["D"] * q["FF"]
    return layer, q["D"] * case["vocab"]


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, c = case["rows"], case["k"], case["c"]
        return {"bytes": 4 * m * (k + c) + c * k * case["bits"] // 8 + 4 * c, "flops": 2 * m * k * c}
    if kind == "mlp":
        d, h, out, m = case["d"], case["h"], case["out"], case["rows"]
        macs = d * h + h * h + h * out
        return {"bytes": 4 * m * (d + out) + macs * case["bits"] // 8 + 4 * (2 * h + out), "flops": 2 * m * macs}
    if kind == "reasoner":  # about nine think steps a row
        return {"bytes": case["rows"] * 4 * (8 + 4 + 1), "flops": 2 * case["rows"] * (128 + 256 + 64 + 9 * 256)}
    if kind == "ssm":
        n, di, st = case["rows"] * case["t"], 2 * case["d"], case["state"]
        macs = sum(r * c for r, c in _ssm_shapes(case)[:-1]) + case["blocks"] * 3 * di * st
        return {"bytes": 4 * n * case["d"] + 4 * case["rows"] * 8 + sum(r * c for r, c in _ssm_shapes(case)), "flops": 2 * n * macs}
    layer, head = _qwen_macs(case)
    q, layers = QWEN, case["layers"]
    weights = layers * layer // 2
    if kind == "forward":
        t, n = case["t"], case["rows"]
        attn = layers * q["NQ"] * q["HD"] * t * (t + 1)  # both causal products
        return {"bytes": weights + head // 2 + 4 * n * (t + case["vocab"]) + 4 * q["D"] * n * t, "flops": 2 * n * (t * layers * layer + attn + head)}
    s, t, steps = case["seqs"], case["prompt"], case["steps"]
    kv = 8 * q["NKV"] * q["HD"] * layers  # bytes of one position's K and V
    attn = layers * q["NQ"] * q["HD"] * (t * (t + 1) + 2 * sum(range(t + 1, t + steps)))
    nbytes = steps * (weights + head // 2 + 4 * s * case["vocab"]) + s * kv * (t + sum(range(t + 1, t + steps)))
    return {"bytes": nbytes, "flops": 2 * s * ((t + steps - 1) * layers * layer + attn + steps * head)}


def tolerance(case):
    """About four times what the results are off from 64 bits: f32 sums of up to 4096 terms, and what whole models add up."""
    kind = case["kind"]
    if case.get("fixed"):
        return "exact"
    if kind == "linear":
        return {"rel": 2e-6 if case["exact"] else 1e-6}
    if kind == "mlp":
        return {"rel": 2e-6}
    if kind == "reasoner":  # a row whose last change ties the threshold may halt a step earlier or later
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-3}
    if kind == "ssm":
        return {"rel": 1e-6}
    if kind == "forward":
        return {"rel": 6e-6}
    return {"rel": 6e-6, "differ": 1e-3}  # (a choice between tied logits)


# ---- the same in 64 bits ----

def _rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)


def _exact_ssm(case, x):
    d, di, n, r, t = case["d"], 2 * case["d"], case["state"], 16, case["t"]
    shapes, ws, off = _ssm_shapes(case), [], 0
    stream = synth.normal(105, 0.02, sum(a * b for a, b in shapes))
    for a, b in shapes:
        codes, scales = hip.quantize_rtn(stream[off:off + a * b].reshape(a, b), 8, 1)
        ws.append(_f64((codes, scales, 1)))
        off += a * b
    A = -torch.arange(1, n + 1, device=DEV, dtype=torch.float64)
    bdt = float(np.float32(np.log(np.expm1(0.01))))
    x = x.double().view(-1, t, d)
    for b in range(case["blocks"]):
        wx, wz, wdtin, wdt, wb, wc, wo = ws[7 * b:7 * b + 7]
        u = torch.nn.functional.silu(x @ wx)
        dt = torch.nn.functional.softplus(u @ wdtin @ wdt + bdt, threshold=700)
        Bm, Cm = u @ wb, u @ wc
        h = torch.zeros(x.shape[0], di, n, device=DEV, dtype=torch.float64)
        y = torch.empty_like(u)
        for k in range(t):
            h = torch.exp(dt[:, k, :, None] * A) * h + (dt[:, k] * u[:, k])[:, :, None] * Bm[:, k, None, :]
            y[:, k] = (h * Cm[:, k, None, :]).sum(-1)
        y = (y + u) * torch.nn.functional.silu(x @ wz)
        x = _rms(x + y @ wo)
    return torch.softmax(x.mean(1) @ ws[-1], -1)


class _Qwen64:
    """The Qwen3-shaped decoder in 64 bits, over chunks of positions with a cache."""

    def __init__(self, case, length):
        q = QWEN
        w = synth.qwen3_weights(case["layers"], V=case["vocab"], **q)
        deq = lambda a: _f64(hip.quantize_rtn(np.ascontiguousarray(a), 4, 1) + (1,))  # noqa: E731
        cat = lambda f, l, n: torch.cat([deq(w[f % (l, h)]) for h in range(n)], 1)  # noqa: E731
        self.E = torch.from_numpy(w["E"]).to(DEV, torch.float64)
        self.LM = deq(w["E"].T)
        self.layers = []
        for l in range(case["layers"]):
            self.layers.append((cat("Wq_%d_%d", l, q["NQ"]), cat("Wk_%d_%d", l, q["NKV"]), cat("Wv_%d_%d", l, q["NKV"]),
                                torch.cat([deq(w["Wo_%d_%d" % (l, h)]) for h in range(q["NQ"])], 0),
                                deq(w["Wg_%d" % l]), deq(w["Wu_%d" % l]), deq(w["Wd_%d" % l])))
        cos, sin, rot = synth.rope_tables(length, q["HD"])
        self.cos, self.sin = (torch.from_numpy(a).to(DEV, torch.float64) for a in (cos, sin))
        self.rot = deq(rot)
        self.scale = float(np.float32("%.9g" % (1.0 / np.sqrt(q["HD"]))))
        self.kv = [None] * case["layers"]

    def __call__(self, ids, p0=0):
        """logits of the last of the positions p0 .. p0 + T - 1"""
        q = QWEN
        S, T = ids.shape
        heads = lambda a, n: a.view(S, T, n, q["HD"]).transpose(1, 2)  # noqa: E731
        turn = lambda a: a * self.cos[p0:p0 + T] + (a @ self.rot) * self.sin[p0:p0 + T]  # noqa: E731
        h = self.E[ids.long()]
        for l, (wq, wk, wv, wo, wg, wu, wd) in enumerate(self.layers):
            n = _rms(h)
            k, v, qq = turn(_rms(heads(n @ wk, q["NKV"]))), heads(n @ wv, q["NKV"]), turn(_rms(heads(n @ wq, q["NQ"])))
            if p0:
                k, v = (torch.cat([a, b], 2) for a, b in zip(self.kv[l], (k, v)))
            self.kv[l] = (k, v)
            grp = q["NQ"] // q["NKV"]
            k, v = (a.repeat_interleave(grp, 1).contiguous() for a in (k, v))
            s = (qq.contiguous() @ k.transpose(2, 3).contiguous()) * self.scale
            at = torch.arange(p0, p0 + T, device=DEV)
            s = s.masked_fill(torch.arange(p0 + T, device=DEV)[None, :] > at[:, None], -math.inf)
            h = h + (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(S, T, -1) @ wo
            n = _rms(h)
            h = h + (torch.nn.functional.silu(n @ wg) * (n @ wu)) @ wd
        return _rms(h[:, -1]) @ self.LM


def exact(case, seed):
    if case.get("fixed"):
        return None  # whole numbers: they stay the same
    kind, x = case["kind"], _inputs(case, seed)
    if kind == "linear":
        return x.double() @ _f64(_model(case)[1][0]).T.contiguous()
    if kind == "mlp":
        x = torch.from_numpy(x).to(DEV) if case["host"] else x
        w1, w2, w3 = (_f64(q).T.contiguous() for q in _model(case)[1])
        out = torch.empty(case["rows"], case["out"], device=DEV, dtype=torch.float64)
        for a in range(0, case["rows"], 16384):
            out[a:a + 16384] = _rms(torch.tanh(torch.tanh(x[a:a + 16384].double() @ w1) @ w2) @ w3)
        return out
    if kind == "reasoner":
        rand = lambda s, a, r, c: torch.from_numpy(synth.rand(s, a, r * c).reshape(r, c)).to(DEV, torch.float64)  # noqa: E731
        emb, core, inj, head = rand(11, 0.35, 16, 8), rand(23, 0.12, 16, 16), rand(37, 0.10, 16, 16), rand(41, 0.5, 4, 16)
        e = _rms(x.double() @ emb.T)
        z, live = e.clone(), torch.ones(len(e), 1, dtype=torch.bool, device=DEV)
        for _ in range(32):
            y = torch.tanh(z @ core.T + e @ inj.T + float(np.float32(0.01)))
            d = (y - z).abs().amax(1, keepdim=True)
            z = torch.where(live, y, z)
            live = live & (d > float(np.float32(9.99999975e-05)))
        return {"out": torch.softmax(z @ head.T, -1), "steps": None}
    if kind == "ssm":
        return _exact_ssm(case, x)
    if kind == "forward":
        return _Qwen64(case, case["t"])(x)
    model, logits = _Qwen64(case, case["prompt"] + case["steps"]), []
    ids, p0 = x, 0
    for _ in range(case["steps"]):
        logits.append(model(ids, p0))
        p0 += ids.shape[1]
        ids = logits[-1].argmax(-1, keepdim=True).float()
    return {"tokens": None, "logits": torch.stack(logits)}
