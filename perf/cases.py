"""What a user of the framework has it do, as cases that can be timed and checked.

Each case is one pass through the public entry points (``HipDevice``,
``Gemma2Model``), over the range that a program decoding and prefilling
Gemma-shaped GGUF models meets: one token at a time and batches of a few to 512
tokens, Q4_0 / Q8_0 / Q4_K weights, f16 / Q8_0 / Q4_0 KV caches, short and long
contexts, whole token steps and whole prefills.

Kinds:

* ``matvec``      one quantised matrix-vector product on an f32 vector;
* ``head``        the vocabulary product of a token and the sampled pick over it;
* ``ffn_token``   a GeGLU FFN for one token;
* ``ffn_batch``   the same for a batch of prompt tokens;
* ``attn_token``  attention of one token over its KV cache;
* ``attn_batch``  the attention half of a layer for a batch of prompt tokens:
                  q|k|v, RoPE and K/V append, attention, output projection;
* ``step``        one token step of a model (a captured graph replayed);
* ``prefill``     a prompt through a model.

Weights and inputs are synthetic: GGUF block bytes made on the GPU from the
seed, in the distributions of ``synth.py``.
"""

from __future__ import annotations

import importlib.util
import math
import sys
from pathlib import Path

import torch

PKG_DIR = Path(__file__).resolve().parents[1] / "qt_llama.cpp_amd"
FORMATS = {"f16": 0, "q8_0": 1, "q4_0": 2}
EPS = 1e-6
ROPE_BASE = 10000.0

# the Gemma-2-2B shape of the repository's benchmark
GEMMA2_2B = dict(layers=26, dim=2304, heads=8, kv_heads=4, head_dim=256, ffn=9216, vocab=256000, ctx=4096)

_state = {}


def _backend():
    """The package (its folder's name is no identifier, so it is loaded by path)."""
    name = "qt_llama_cpp_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, PKG_DIR / "__init__.py",
                                                      submodule_search_locations=[str(PKG_DIR)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def _device():
    """One context for the program, its scratch reserved once (as a program that captures graphs does)."""
    if "dev" not in _state:
        dev = _backend().HipDevice.new(0)
        dev.reserve_workspace(256 << 20)
        _state["dev"] = dev
    return _state["dev"]


# ---- cases -------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # the smallest call there is: a 2048x2048 Q8_0 product for one vector (launch and host time count)
        dict(name="matvec_q8_0_2048", kind="matvec", format="q8_0", rows=2048, cols=2048),
        # the FFN of every decoded token of the 2B shape: two thirds of its weight bytes
        dict(name="ffn_token_2304x9216", kind="ffn_token", dim=2304, ffn=9216),
        # the same of a model of another width
        dict(name="ffn_token_2816x8192", kind="ffn_token", dim=2816, ffn=8192),
        # the vocabulary product and sampled pick that end every decoded token, with a Q4_K table
        dict(name="head_q4_k_256000", kind="head", format="q4_k", rows=256000, cols=2304, temperature=0.8, top_k=40),
        # the FFN for the few new tokens of a chat turn
        dict(name="ffn_batch_12", kind="ffn_batch", dim=2304, ffn=9216, batch=12),
        # the FFN for a whole chunk of a prompt
        dict(name="ffn_batch_512", kind="ffn_batch", dim=2304, ffn=9216, batch=512),
        # decode attention late in a 4096-token context
        dict(name="attn_token_f16_3000", kind="attn_token", heads=8, kv_heads=4, head_dim=256, n_past=3000,
             capacity=4096, window=0, k_format="f16", v_format="f16"),
        # decode attention of a windowed layer over quantised caches, wider groups, smaller heads
        dict(name="attn_token_q8_window", kind="attn_token", heads=16, kv_heads=2, head_dim=128, n_past=5000,
             capacity=8192, window=1024, k_format="q8_0", v_format="q4_0"),
        # a ragged chat turn behind a cached prefix, attention half of a layer
        dict(name="attn_batch_77", kind="attn_batch", dim=2304, heads=8, kv_heads=4, head_dim=256, batch=77,
             start=300, capacity=4096, window=0, k_format="f16", v_format="f16"),
        # a later chunk of a long prompt, attention half of a layer
        dict(name="attn_batch_512_late", kind="attn_batch", dim=2304, heads=8, kv_heads=4, head_dim=256, batch=512,
             start=2048, capacity=4096, window=0, k_format="f16", v_format="f16"),
        # a decoded token of the 2B shape, greedy with the recent-token penalty
        dict(name="step_2b", kind="step", pos=700, numerics="exact", **GEMMA2_2B),
        # a ragged prompt through the 2B shape
        dict(name="prefill_2b_333", kind="prefill", tokens=333, start=0, numerics="exact", **GEMMA2_2B),
    ]


def _log(rng, lo: int, hi: int, unit: int = 1) -> int:
    """An integer from [lo, hi], evenly over its logarithm, rounded down to `unit`."""
    n = int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))
    return max(unit, min(n, hi) // unit * unit)


def draw(rng) -> dict:
    kind = rng.choice(["matvec", "head", "ffn_token", "ffn_batch", "ffn_batch", "attn_token", "attn_token",
                       "attn_batch", "attn_batch", "step", "prefill", "prefill"])
    if kind == "matvec":
        fmt = rng.choice(["q4_0", "q8_0", "q4_k"])
        return dict(kind=kind, format=fmt, rows=_log(rng, 256, 32768),
                    cols=_log(rng, 256, 9216, 256 if fmt == "q4_k" else 32))
    if kind == "head":
        return dict(kind=kind, format=rng.choice(["q4_0", "q8_0", "q4_k"]), rows=_log(rng, 32000, 256000),
                    cols=_log(rng, 1024, 4096, 256), temperature=rng.choice([0.0, 0.7, 1.0]),
                    top_k=rng.choice([1, 20, 40, 64]))
    dim, ffn = _log(rng, 1024, 4096, 32), _log(rng, 2048, 16384, 32)
    if kind == "ffn_token":
        return dict(kind=kind, dim=dim, ffn=ffn)
    if kind == "ffn_batch":
        return dict(kind=kind, dim=dim, ffn=min(ffn, 9216), batch=_log(rng, 2, 512))
    group = rng.choice([1, 2, 4, 8])
    kv_heads = rng.choice([1, 2, 4])
    head_dim = rng.choice([64, 128, 256, 256, 512])
    fmts = rng.choice([("f16", "f16"), ("f16", "f16"), ("q8_0", "q8_0"), ("q8_0", "q4_0"), ("q4_0", "q4_0")])
    attn = dict(heads=kv_heads * group, kv_heads=kv_heads, head_dim=head_dim, capacity=8192,
                window=rng.choice([0, 0, 512, 1024]), k_format=fmts[0], v_format=fmts[1])
    if kind == "attn_token":
        return dict(kind=kind, n_past=_log(rng, 16, 8000), **attn)
    if kind == "attn_batch":
        batch = _log(rng, 2, 400)
        attn.update(capacity=4096, heads=min(attn["heads"], 8), kv_heads=min(kv_heads, 8 // group))
        return dict(kind=kind, dim=dim, batch=batch, start=rng.choice([0, _log(rng, 16, 3600)]), **attn)
    shape = dict(layers=rng.choice([2, 3, 4]), dim=dim, heads=8, kv_heads=rng.choice([2, 4]), head_dim=256, ffn=ffn,
                 vocab=_log(rng, 32000, 256000, 32), ctx=4096, numerics=rng.choice(["exact", "exact", "fast"]))
    if kind == "step":
        return dict(kind=kind, pos=_log(rng, 16, 4000), **shape)
    return dict(kind=kind, tokens=_log(rng, 2, 512), start=rng.choice([0, 0, _log(rng, 16, 2000)]), **shape)


# ---- inputs ------------------------------------------------------------------

class _Rand:
    """Seeded tensors on the GPU."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape) -> torch.Tensor:
        return torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32)

    def ints(self, lo: int, hi: int, *shape, dtype=torch.int32) -> torch.Tensor:
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=dtype)

    def _scales(self, n: int, sigma: float) -> torch.Tensor:
        return (self.normal(n).abs() * sigma).half().view(torch.uint8).view(n, 2)

    def weights(self, fmt: str, rows: int, cols: int) -> torch.Tensor:
        """A matrix as GGUF block bytes (q4_0: values -7..7, as a quantiser's output has no mean)."""
        n = rows * cols // (256 if fmt == "q4_k" else 32)
        if fmt == "q4_0":
            qs = self.ints(1, 16, n, 16, dtype=torch.uint8) | (self.ints(1, 16, n, 16, dtype=torch.uint8) << 4)
            return torch.cat([self._scales(n, 0.02 / 8), qs], 1).reshape(-1)
        if fmt == "q8_0":
            qs = self.ints(-127, 128, n, 32, dtype=torch.int8).view(torch.uint8)
            return torch.cat([self._scales(n, 0.02 / 127), qs], 1).reshape(-1)
        head = torch.cat([self._scales(n, 0.01), self._scales(n, 0.01)], 1)  # d, dmin; then scales and quants
        return torch.cat([head, self.ints(0, 256, n, 140, dtype=torch.uint8)], 1).reshape(-1)

    def cache(self, fmt: str, *shape) -> torch.Tensor:
        """K or V rows of `shape` (last: head_dim) in a cache's format, of about unit size."""
        if fmt == "f16":
            return self.normal(*shape).half()
        n = math.prod(shape) // 32
        if fmt == "q8_0":
            qs = self.ints(-127, 128, n, 32, dtype=torch.int8).view(torch.uint8)
            return torch.cat([self._scales(n, 2.0 / 127), qs], 1).reshape(-1)
        return torch.cat([self._scales(n, 0.25), self.ints(0, 256, n, 16, dtype=torch.uint8)], 1).reshape(-1)


MATRICES = ("wq", "wk", "wv", "wo", "w_gate", "w_up", "w_down")
NORMS = ("attn_norm", "post_attn_norm", "ffn_norm", "post_ffw_norm")


def _shapes(c: dict) -> dict:
    qd, kvd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    return {"wq": (qd, c["dim"]), "wk": (kvd, c["dim"]), "wv": (kvd, c["dim"]), "wo": (c["dim"], qd),
            "w_gate": (c.get("ffn"), c["dim"]), "w_up": (c.get("ffn"), c["dim"]), "w_down": (c["dim"], c.get("ffn"))}


def _inputs(c: dict, seed: int) -> dict:
    """Everything random of a case: GGUF bytes, f32 vectors, caches, tokens."""
    r = _Rand(seed)
    kind = c["kind"]
    if kind in ("matvec", "head"):
        d = {"w": r.weights(c["format"], c["rows"], c["cols"]), "x": r.normal(c["cols"])}
        if kind == "head":
            d["valid"] = (r.ints(0, 50, c["rows"]) > 0).to(torch.uint8)
            d["recent"] = r.ints(0, c["rows"], 32)
        return d
    if kind in ("ffn_token", "ffn_batch"):
        m = {n: r.weights("q4_0", *_shapes({**c, "heads": 1, "kv_heads": 1, "head_dim": 32})[n])
             for n in ("w_gate", "w_up", "w_down")}
        return {**m, "x": r.normal(c.get("batch", 1), c["dim"])}
    if kind in ("attn_token", "attn_batch"):
        rows = (c["capacity"], c["kv_heads"], c["head_dim"])
        d = {"k": r.cache(c["k_format"], *rows), "v": r.cache(c["v_format"], *rows)}
        if kind == "attn_token":
            return {**d, "q": r.normal(c["heads"] * c["head_dim"])}
        return {**d, **{n: r.weights("q4_0", *_shapes(c)[n]) for n in ("wq", "wk", "wv", "wo")},
                "x": r.normal(c["batch"], c["dim"])}
    layers = [{**{n: r.weights("q4_0", *_shapes(c)[n]) for n in MATRICES},
               **{n: 1 + 0.1 * r.normal(c["dim"]) for n in NORMS}} for _ in range(c["layers"])]
    rows = (c["layers"], c["ctx"], c["kv_heads"], c["head_dim"])
    return {"layers": layers, "table": r.weights("q4_0", c["vocab"], c["dim"]),
            "norm": 1 + 0.1 * r.normal(c["dim"]), "k": r.cache("f16", *rows), "v": r.cache("f16", *rows),
            "tokens": r.ints(0, c["vocab"], c.get("tokens", 1))}


# ---- what a program keeps, and one pass --------------------------------------

def _upload(fmt: str, gguf: torch.Tensor, rows: int, cols: int) -> torch.Tensor:
    """GGUF bytes on the GPU -> the library's weight layout, as a model load does."""
    dev = _device()
    out = torch.empty_like(gguf)
    torch.cuda.current_stream().synchronize()
    fn = {"q4_0": dev.lib.mrml_hip_repack_q4_0, "q8_0": dev.lib.mrml_hip_repack_q8_0,
          "q4_k": dev.lib.mrml_hip_repack_q4_k}[fmt]
    dev._check(fn(dev.ctx, gguf.data_ptr(), out.data_ptr(), rows, cols))
    dev.sync()
    return out


def _f32(*shape) -> torch.Tensor:
    return torch.zeros(*shape, device="cuda", dtype=torch.float32)


def _rope_table(n: int, head_dim: int) -> torch.Tensor:
    t = _f32(n, head_dim)
    torch.cuda.current_stream().synchronize()
    _device().rope_table(t.data_ptr(), n, head_dim, ROPE_BASE)
    return t


def _model(c: dict, d: dict, s: dict):
    """The model handle over uploaded weights."""
    be, dev = _backend(), _device()
    shapes = _shapes(c)
    s["layers"] = [{**{n: _upload("q4_0", L[n], *shapes[n]) for n in MATRICES}, **{n: L[n] for n in NORMS}}
                   for L in d["layers"]]
    s["table"] = _upload("q4_0", d["table"], c["vocab"], c["dim"])
    s["norm"] = d["norm"]
    cfg = be.Gemma2Config(c["layers"], c["dim"], c["heads"], c["kv_heads"], c["head_dim"], c["ffn"], c["vocab"],
                          c["ctx"], ROPE_BASE, EPS, 1.0 / math.sqrt(c["head_dim"]), be.Q4_0,
                          be.NUMERICS_FAST if c["numerics"] == "fast" else be.NUMERICS_EXACT, 0, 0)
    m = be.Gemma2Model(dev, cfg, s["table"].data_ptr(), s["norm"].data_ptr(),
                       [{n: t.data_ptr() for n, t in L.items()} for L in s["layers"]])
    m.set_sampler(temperature=0.0, top_k=40)
    return m


def prepare(c: dict, seed: int) -> dict:
    dev, d, kind = _device(), _inputs(c, seed), c["kind"]
    s = {"c": c}
    if kind in ("matvec", "head"):
        s.update(x=d["x"], w=_upload(c["format"], d["w"], c["rows"], c["cols"]), y=_f32(c["rows"]))
        if kind == "head":
            s.update(valid=d["valid"], recent=d["recent"], token=torch.zeros(1, device="cuda", dtype=torch.int32),
                     ids=torch.zeros(c["top_k"], device="cuda", dtype=torch.int32), scores=_f32(c["top_k"]))
    elif kind in ("ffn_token", "ffn_batch"):
        f, n, b = c["ffn"], c["dim"], c.get("batch", 1)
        s.update(x=d["x"], gate=_upload("q4_0", d["w_gate"], f, n), up=_upload("q4_0", d["w_up"], f, n),
                 down=_upload("q4_0", d["w_down"], n, f), act=_f32(b, f), y=_f32(b, n))
    elif kind == "attn_token":
        s.update(q=d["q"], k=d["k"], v=d["v"], y=_f32(c["heads"] * c["head_dim"]))
    elif kind == "attn_batch":
        qd, kvd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        shapes = _shapes(c)
        s.update({n: _upload("q4_0", d[n], *shapes[n]) for n in ("wq", "wk", "wv", "wo")})
        s.update(x=d["x"], k=d["k"], v=d["v"], table=_rope_table(c["start"] + c["batch"], c["head_dim"]),
                 qkv=_f32(c["batch"], qd + 2 * kvd), o=_f32(c["batch"], qd), y=_f32(c["batch"], c["dim"]))
    else:
        s.update(model=_model(c, d, s), k=d["k"], v=d["v"], logits=_f32(c["vocab"]),
                 next=torch.zeros(1, device="cuda", dtype=torch.int32), tokens=d["tokens"])
        if kind == "prefill":
            s["model"].reserve_prefill()
        else:
            # {token, position}, put back before each step so that every pass is the same step
            s["start"] = torch.tensor([int(d["tokens"][0]), c["pos"], 0, 0], device="cuda", dtype=torch.int32)
            s["state"] = s["start"].clone()
            torch.cuda.current_stream().synchronize()

            def step():
                dev.copy_kernel(s["state"].data_ptr(), s["start"].data_ptr(), 16)
                s["model"].step(s["state"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["logits"].data_ptr(),
                                s["next"].data_ptr())
            s["graph"] = dev.capture(step)
    torch.cuda.synchronize()
    return s


def run(s: dict):
    dev, c = _device(), s["c"]
    kind = c["kind"]
    if kind in ("matvec", "head"):
        fn = {"q4_0": dev.gemv_q4_0, "q8_0": dev.gemv_q8_0, "q4_k": dev.gemv_q4_k}[c["format"]]
        fn(s["w"].data_ptr(), s["x"].data_ptr(), s["y"].data_ptr(), c["rows"], c["cols"])
        if kind == "matvec":
            return {"y": s["y"]}
        dev.vocab_select(s["y"].data_ptr(), c["rows"], s["valid"].data_ptr(), s["recent"].data_ptr(), 32, 10, 0,
                         c["temperature"], 700, c["top_k"], s["token"].data_ptr(), s["scores"].data_ptr(),
                         s["ids"].data_ptr())
        return {"logits": s["y"], "token": s["token"], "scores": s["scores"], "ids": s["ids"]}
    if kind == "ffn_token":
        dev.ffn_geglu_q4_0(s["gate"].data_ptr(), s["up"].data_ptr(), s["down"].data_ptr(), s["x"].data_ptr(),
                           s["act"].data_ptr(), s["y"].data_ptr(), c["dim"], c["ffn"])
        return {"y": s["y"], "act": s["act"]}
    if kind == "ffn_batch":
        dev.gemm_q4_0_geglu(s["gate"].data_ptr(), s["up"].data_ptr(), s["x"].data_ptr(), s["act"].data_ptr(),
                            c["ffn"], c["dim"], c["batch"])
        dev.gemm_q4_0(s["down"].data_ptr(), s["act"].data_ptr(), s["y"].data_ptr(), c["dim"], c["ffn"], c["batch"])
        return {"y": s["y"], "act": s["act"]}
    if kind == "attn_token":
        dev.attention_causal_ref(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["y"].data_ptr(),
                                 c["n_past"], c["heads"], c["kv_heads"], c["head_dim"],
                                 1.0 / math.sqrt(c["head_dim"]), c["window"] or None, c["capacity"],
                                 FORMATS[c["k_format"]], FORMATS[c["v_format"]])
        return {"y": s["y"]}
    if kind == "attn_batch":
        h, kvh, hd, b = c["heads"], c["kv_heads"], c["head_dim"], c["batch"]
        kf, vf = FORMATS[c["k_format"]], FORMATS[c["v_format"]]
        dev.gemm_q4_0_qkv(s["wq"].data_ptr(), s["wk"].data_ptr(), s["wv"].data_ptr(), s["x"].data_ptr(),
                          s["qkv"].data_ptr(), h * hd, kvh * hd, c["dim"], b)
        dev.qkv_postprocess_batch(s["qkv"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), c["start"], c["start"],
                                  h, kvh, hd, ROPE_BASE, b, c["capacity"], kf, vf, 1.0, s["table"].data_ptr(),
                                  c["start"] + b)
        dev.attention_prefill(s["qkv"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["o"].data_ptr(),
                              c["start"], b, h, kvh, hd, 1.0 / math.sqrt(hd), c["window"] or None, c["capacity"],
                              kf, vf, (h + 2 * kvh) * hd)
        dev.gemm_q4_0(s["wo"].data_ptr(), s["o"].data_ptr(), s["y"].data_ptr(), c["dim"], h * hd, b)
        return {"y": s["y"], "attn": s["o"], "k": s["k"], "v": s["v"]}
    if kind == "step":
        s["graph"].launch()
    else:
        s["model"].prefill(s["tokens"].data_ptr(), c["tokens"], c["start"], s["k"].data_ptr(), s["v"].data_ptr(),
                           s["logits"].data_ptr(), s["next"].data_ptr())
    return {"logits": s["logits"], "next": s["next"], "k": s["k"], "v": s["v"]}


# ---- bytes, operations, tolerance --------------------------------------------

BYTES_PER_WEIGHT = {"q4_0": 18 / 32, "q8_0": 34 / 32, "q4_k": 144 / 256, "f16": 2.0}


def _attention_work(c: dict, first: int, n: int) -> tuple[float, float]:
    """Bytes of the K and V rows that n queries from position `first` see, and the products' operations."""
    window = c.get("window") or (1 << 30)
    cap = c.get("capacity", c.get("ctx"))
    spans = [min(p + 1, window, cap) for p in range(first, first + n)]
    rows = min(first + n, spans[-1] + n - 1)
    kvd = c["kv_heads"] * c["head_dim"]
    per = kvd * (BYTES_PER_WEIGHT[c.get("k_format", "f16")] + BYTES_PER_WEIGHT[c.get("v_format", "f16")])
    return rows * per, 4.0 * sum(spans) * c["heads"] * c["head_dim"]


def work(c: dict) -> dict:
    kind = c["kind"]
    if kind in ("matvec", "head"):
        n = c["rows"] * c["cols"]
        b = n * BYTES_PER_WEIGHT[c["format"]] + 4 * (c["cols"] + c["rows"]) + (c["rows"] if kind == "head" else 0)
        return {"bytes": b, "flops": 2.0 * n}
    if kind in ("ffn_token", "ffn_batch"):
        n, m = 3 * c["dim"] * c["ffn"], c.get("batch", 1)
        return {"bytes": n * 18 / 32 + 4 * m * (2 * c["dim"] + c["ffn"]), "flops": 2.0 * n * m}
    if kind == "attn_token":
        b, f = _attention_work(c, c["n_past"], 1)
        return {"bytes": b + 8 * c["heads"] * c["head_dim"], "flops": f}
    if kind == "attn_batch":
        b, f = _attention_work(c, c["start"], c["batch"])
        n = sum(math.prod(_shapes(c)[w]) for w in ("wq", "wk", "wv", "wo"))
        out = 4 * c["batch"] * (2 * c["dim"] + c["heads"] * c["head_dim"])
        return {"bytes": b + n * 18 / 32 + out, "flops": f + 2.0 * n * c["batch"]}
    m, first = (1, c["pos"]) if kind == "step" else (c["tokens"], c["start"])
    b, f = _attention_work(c, first, m)
    n = c["layers"] * sum(math.prod(s) for s in _shapes(c).values())
    head = c["vocab"] * c["dim"]
    return {"bytes": (n + head) * 18 / 32 + c["layers"] * (b + 16 * c["dim"]) + 4 * c["vocab"],
            "flops": 2.0 * n * m + 2.0 * head + c["layers"] * f}


def tolerance(c: dict):
    """Every op here but the FAST numerics is defined bit by bit (the CPU path's order of operations), so
    another correct implementation gives the same values.  FAST sums in another order, and a changed last
    bit can move a quantised activation by one step, which the later layers spread."""
    if c.get("numerics") == "fast":
        return {"rel": 0.03, "max": 0.3, "differ": 0.01}
    return "exact"


# ---- the same in 64 bits -----------------------------------------------------

def _dequant(fmt: str, raw: torch.Tensor, rows: int, cols: int) -> torch.Tensor:
    if fmt == "f16":
        return raw.double().view(rows, cols)
    size = {"q4_0": 18, "q8_0": 34, "q4_k": 144}[fmt]
    raw = raw.view(-1, size)

    def half(at):
        return raw[:, at:at + 2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        return (half(0) * raw[:, 2:].contiguous().view(torch.int8).double()).view(rows, cols)
    if fmt == "q4_0":
        q = torch.cat([raw[:, 2:] & 15, raw[:, 2:] >> 4], 1).double() - 8
        return (half(0) * q).view(rows, cols)
    s = raw[:, 4:16].int()
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    qs = raw[:, 16:].view(-1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).view(-1, 8, 32).double()
    return ((half(0) * sc).unsqueeze(2) * q - (half(2) * mn).unsqueeze(2)).view(rows, cols)


def _quantised(x: torch.Tensor, levels: float = 127.0, low: float = -128.0, high: float = 127.0) -> torch.Tensor:
    """x after a block quantiser: 32 values share amax/levels, kept as a truncated half."""
    v = x.float().reshape(-1, 32)
    scale = v.abs().amax(1, keepdim=True) / levels
    h = scale.half()
    h = torch.where(h.float() > scale, (h.view(torch.int16) - 1).view(torch.float16), h)
    t = torch.where(scale > 0, v * (1 / scale), torch.zeros_like(v)).double()
    q = (torch.sign(t) * torch.floor(t.abs() + 0.5)).clamp(low, high)
    return (h.double() * q).view(x.shape)


def _product(x: torch.Tensor, fmt: str, raw: torch.Tensor, rows: int, cols: int) -> torch.Tensor:
    """Rows of x (quantised as the path does) times a quantised matrix."""
    xq = _quantised(x)
    size = raw.numel() // rows
    return torch.cat([xq @ _dequant(fmt, raw[r * size:(r + n) * size], n, cols).T
                      for r, n in ((r, min(32768, rows - r)) for r in range(0, rows, 32768))], -1)


def _geglu(g: torch.Tensor, u: torch.Tensor) -> torch.Tensor:
    return 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3))) * u


def _norm(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
    """x: [token][head][head_dim]."""
    half = x.shape[-1] // 2
    i = torch.arange(half, device="cuda", dtype=torch.float64)
    a = (pos.double()[:, None] / ROPE_BASE ** (2 * i / x.shape[-1]))[:, None, :]
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * a.cos() - hi * a.sin(), lo * a.sin() + hi * a.cos()], -1)


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, first: int, window: int) -> torch.Tensor:
    """q: [token][head][hd] at positions first ..; k, v: [position][kv head][hd]."""
    group = q.shape[1] // k.shape[1]
    at = torch.arange(first, first + q.shape[0], device="cuda")[:, None]
    t = torch.arange(k.shape[0], device="cuda")[None, :]
    seen = (t <= at) & ((t > at - window) if window else (t >= 0))
    out = []
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h // group].T / math.sqrt(q.shape[-1])
        out.append(torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[:, h // group])
    return torch.stack(out, 1)


def _stored(x: torch.Tensor, fmt: str) -> torch.Tensor:
    """K or V rows as the cache gives them back."""
    if fmt == "f16":
        return x.float().half().double()
    return _quantised(x) if fmt == "q8_0" else _quantised(x, 8.0, -8.0, 7.0)


def _layer_attention(c: dict, d: dict, x: torch.Tensor, k: torch.Tensor, v: torch.Tensor, first: int):
    """x: normed rows.  Writes their K and V into k, v; returns the attention rows and their projection."""
    n, hd, shapes = x.shape[0], c["head_dim"], _shapes(c)
    q, kn, vn = (_product(x, "q4_0", d[w], *shapes[w]).view(n, -1, hd) for w in ("wq", "wk", "wv"))
    pos = torch.arange(first, first + n, device="cuda")
    k[first:first + n] = _stored(_rope(kn, pos), c.get("k_format", "f16"))
    v[first:first + n] = _stored(vn, c.get("v_format", "f16"))
    q = _rope(q, pos)
    if c.get("k_format", "f16") != "f16":
        q = _quantised(q)
    o = _attend(q, k[:first + n], v[:first + n], first, c.get("window", 0)).reshape(n, -1)
    return o, _product(o, "q4_0", d["wo"], *shapes["wo"])


def exact(c: dict, seed: int):
    d, kind = _inputs(c, seed), c["kind"]
    if kind in ("matvec", "head"):
        y = _product(d["x"].double()[None], c["format"], d["w"], c["rows"], c["cols"])[0]
        if kind == "matvec":
            return {"y": y}
        s = 30 * torch.tanh(y / 30)
        s[d["recent"].long().unique()] -= 3.5
        s[d["valid"] == 0] = -math.inf
        return {"logits": y, "token": None, "scores": s.topk(c["top_k"]).values, "ids": None}
    if kind in ("ffn_token", "ffn_batch"):
        x = d["x"].double()
        act = _geglu(_product(x, "q4_0", d["w_gate"], c["ffn"], c["dim"]),
                     _product(x, "q4_0", d["w_up"], c["ffn"], c["dim"]))
        return {"act": act, "y": _product(act, "q4_0", d["w_down"], c["dim"], c["ffn"])}
    if kind in ("attn_token", "attn_batch"):
        rows = (c["capacity"], c["kv_heads"], c["head_dim"])
        k, v = (_dequant(c[f], d[n], c["capacity"], rows[1] * rows[2]).view(rows).clone()
                for n, f in (("k", "k_format"), ("v", "v_format")))
        if kind == "attn_token":
            n, q = c["n_past"] + 1, d["q"].double().view(1, c["heads"], c["head_dim"])
            if c["k_format"] != "f16":
                q = _quantised(q)
            return {"y": _attend(q, k[:n], v[:n], c["n_past"], c["window"])[0].reshape(-1)}
        o, y = _layer_attention(c, d, d["x"].double(), k, v, c["start"])
        return {"y": y, "attn": o, "k": k if c["k_format"] == "f16" else None,
                "v": v if c["v_format"] == "f16" else None}
    first = c["pos"] if kind == "step" else c["start"]
    h = _dequant("q4_0", d["table"].view(c["vocab"], -1)[d["tokens"].long()].reshape(-1), d["tokens"].numel(),
                 c["dim"]) * math.sqrt(c["dim"])
    k, v = d["k"].double(), d["v"].double()
    shapes = _shapes(c)
    for l, L in enumerate(d["layers"]):
        _, o = _layer_attention(c, L, _norm(h, L["attn_norm"]), k[l], v[l], first)
        h = h + _norm(o, L["post_attn_norm"])
        x = _norm(h, L["ffn_norm"])
        act = _geglu(_product(x, "q4_0", L["w_gate"], *shapes["w_gate"]),
                     _product(x, "q4_0", L["w_up"], *shapes["w_up"]))
        h = h + _norm(_product(act, "q4_0", L["w_down"], *shapes["w_down"]), L["post_ffw_norm"])
    logits = _product(_norm(h[-1:], d["norm"]), "q4_0", d["table"], c["vocab"], c["dim"])[0]
    return {"logits": logits, "next": None, "k": k, "v": v}
