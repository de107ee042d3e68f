"""Performance cases of the quantized-transformer path.

Each case is one call that a program built on ``doe_amd`` makes: a projection,
an attention, or a whole decoder call.  Matrices, caches and activations are
torch tensors on the GPU handed to ``doe_amd.ops`` by address (the ABI takes
any device pointer); the decoder cases fill a ``doe_amd.model.Decoder``.

Kinds
  gemv        one decode projection (M = 1) over Q4_K or Q8_0 rows, plain, with
              the residual add, or with RMSNorm before and GeGLU after it
  int4        one int4 group-32 projection over a batch of 1 to 8 tokens
  gemm_bf16   one prompt projection, bf16 activations, Q4_K rows
  gemm_f32    one prompt projection of the decoder's batched prompt: f32
              activations, Q4_K or Q8_0 rows, its neighbouring steps folded in
  attn_decode one decode token per sequence against an f16 KV cache
  attn_bf16   causal prompt attention over bf16 K / V
  attn_f16kv  causal prompt attention over the decoder's f16 cache
  decode      a whole generate() call: a short prompt and greedy tokens as
              replays of the captured step
  prompt      a whole prompt in one batched pass
"""
from __future__ import annotations

import math

import numpy as np
import torch

import doe_amd
from doe_amd import Stream, ops
from doe_amd.model import Decoder, DecoderConfig

DEV = "cuda"
EPS = 1e-6


class Buf:
    """A torch tensor as an operator argument (its address and its bytes)."""

    def __init__(self, t: torch.Tensor):
        self.t = t
        self.ptr = t.data_ptr()
        self.nbytes = t.numel() * t.element_size()


class _Window:
    """A library buffer's memory, for torch to read and write in place."""

    def __init__(self, buf, dtype: str, shape):
        self.keep = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": dtype, "data": (buf.ptr, False),
                                         "version": 3}


def over(buf, dtype: str, shape) -> torch.Tensor:
    return torch.as_tensor(_Window(buf, dtype, shape), device=DEV)


# ---- the cases -----------------------------------------------------------------

# The 2B-class decoder of the benchmark: 26 layers, hidden 2304, 8 / 4 heads of 256.
MODEL_2B = dict(layers=26, hidden=2304, heads=8, kv_heads=4, head_dim=256, ffn=9216, vocab=256000)


def listed() -> list[dict]:
    return [
        # the smallest calls: one projection of the 2B-class decoder, dispatched by itself
        dict(name="gemv_q4k_9216x2304", kind="gemv", fmt="q4k", form="plain", n=9216, k=2304),
        # the gate/up projection of a 31B-class decoder, norm and GeGLU folded in
        dict(name="gemv_q4k_gate_up_31b", kind="gemv", fmt="q4k", form="norm_geglu", n=43008, k=5376),
        # the FFN projection of a 27B-class decoder at batch 8, int4 weights
        dict(name="int4_up_27b_b8", kind="int4", m=8, n=25600, k=5120),
        # a 2048-token prompt's FFN projection at 31B-class shapes, bf16 activations
        dict(name="gemm_bf16_31b", kind="gemm_bf16", m=2048, n=21504, k=5376),
        # gate/up of a 1000-token prompt of the 2B-class decoder (ragged in M)
        dict(name="gemm_q4k_gate_up_1000", kind="gemm_f32", fmt="q4k", form="norm_geglu", m=1000, n=18432, k=2304),
        # down_proj of a 333-token prompt of a Q8_0 model
        dict(name="gemm_q8_0_down_333", kind="gemm_f32", fmt="q8_0", form="residual", m=333, n=2304, k=9216),
        # one token against a 4096-token context, batch 1
        dict(name="attn_decode_4096", kind="attn_decode", batch=1, hq=8, hkv=4, d=256, kv=4096, f16=True,
             layout=0, window=0, softcap=0.0),
        # eight sequences of 32768 tokens: 1 GiB of K / V
        dict(name="attn_decode_32k_b8", kind="attn_decode", batch=8, hq=64, hkv=8, d=128, kv=32768, f16=True,
             layout=0, window=0, softcap=0.0),
        # causal attention of a 2048-token prompt at 31B-class shapes
        dict(name="attn_bf16_2048", kind="attn_bf16", hq=32, hkv=16, q=2048, start=0),
        # a 1000-token prompt of the 2B-class decoder over its f16 cache
        dict(name="attn_f16kv_1000", kind="attn_f16kv", hq=8, hkv=4, d=256, q=1000, start=0, window=0, softcap=0.0),
        # the 2B-class decoder: 17 prompt tokens and 8 new ones, 24 decode steps in all
        dict(name="decode_2b", kind="decode", fmt="q4k", prompt=17, new=8, **MODEL_2B),
        # its 128-token prompt as one batched pass
        dict(name="prompt_2b_128", kind="prompt", fmt="q4k", prompt=128, new=0, **MODEL_2B),
    ]


def _log(rng, lo, hi) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["gemv", "gemv", "int4", "gemm_bf16", "gemm_f32", "gemm_f32", "attn_decode", "attn_decode",
                       "attn_bf16", "attn_f16kv", "decode", "prompt"])
    if kind == "gemv":
        fmt, form = rng.choice(["q4k", "q4k", "q8_0"]), rng.choice(["plain", "residual", "norm_geglu"])
        k = 32 * _log(rng, 20, 288)
        n = _log(rng, 500, min(65536, 230_000_000 // k))
        return dict(kind=kind, fmt=fmt, form=form, n=n + (n & 1 if form == "norm_geglu" else 0), k=k)
    if kind == "int4":
        k = 256 * _log(rng, 4, 100)
        return dict(kind=kind, m=rng.randint(1, 8), n=_log(rng, 1000, 131_000_000 // k), k=k)
    if kind == "gemm_bf16":
        k = 32 * _log(rng, 32, 288)
        return dict(kind=kind, m=_log(rng, 33, 2048), n=_log(rng, 1000, min(21504, 115_000_000 // k)), k=k)
    if kind == "gemm_f32":
        fmt, form = rng.choice(["q4k", "q8_0"]), rng.choice(["plain", "residual", "norm_geglu"])
        k = 32 * _log(rng, 20, 288)
        n = _log(rng, 600, min(32768, 80_000_000 // k))
        return dict(kind=kind, fmt=fmt, form=form, m=_log(rng, 9, 1024), n=n + (n & 1 if form == "norm_geglu" else 0),
                    k=k)
    if kind == "attn_decode":
        d, g, hkv, batch = rng.choice([64, 128, 256]), rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 4, 8]), _log(rng, 1, 8)
        kv = _log(rng, 40, min(32768, (1 << 29) // (2 * batch * hkv * d)))
        return dict(kind=kind, batch=batch, hq=g * hkv, hkv=hkv, d=d, kv=kv, f16=rng.random() < 0.5,
                    layout=rng.choice([0, 0, 1]), window=rng.choice([0, 0, 512]), softcap=rng.choice([0.0, 0.0, 50.0]))
    if kind == "attn_bf16":
        g, hkv = rng.choice([1, 2, 4]), rng.choice([4, 8, 16])
        return dict(kind=kind, hq=min(32, g * hkv), hkv=hkv, q=_log(rng, 65, 2048), start=rng.choice([0, 0, 512]))
    if kind == "attn_f16kv":
        d, g, hkv = rng.choice([64, 128, 256, 256, 512]), rng.choice([1, 2, 4]), rng.choice([1, 2, 4])
        return dict(kind=kind, hq=g * hkv, hkv=hkv, d=d, q=_log(rng, 17, 1536), start=rng.choice([0, 0, 256]),
                    window=rng.choice([0, 0, 256]), softcap=rng.choice([0.0, 0.0, 50.0]))
    heads = rng.choice([4, 8])
    small = dict(kind=kind, fmt=rng.choice(["q4k", "q4k", "q8_0"]), layers=rng.randint(2, 12),
                 hidden=128 * rng.randint(5, 20), heads=heads, kv_heads=rng.choice([1, heads // 2]), head_dim=256,
                 ffn=256 * rng.randint(8, 36), vocab=256 * rng.randint(64, 512))
    if kind == "decode":
        return dict(small, prompt=1 + 8 * rng.randint(1, 2), new=8)
    return dict(small, prompt=_log(rng, 20, 512), new=0)


# ---- inputs ----------------------------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(DEV).manual_seed(seed)


def _normal(g, shape, sigma=1.0, dtype=torch.float32, mean=0.0) -> torch.Tensor:
    return (torch.randn(shape, generator=g, device=DEV) * sigma + mean).to(dtype)


def _row_bytes(fmt: str, k: int) -> int:
    return -(-k // 256) * 144 if fmt == "q4k" else -(-k // 32) * 34


def _fill_weights(g, fmt: str, out: torch.Tensor) -> None:
    """Random rows as uint8 in place, weights of mean 0 and deviation ~0.03:
    Q4_K with d ~ |N(0, 2e-4)|, scales and quants uniform, each minimum at the
    middle of its sub-block's range (dmin m = 7.5 d sc); Q8_0 with d ~
    |N(0, 5e-4)|, quants uniform."""
    blocks = out.view(-1, 144 if fmt == "q4k" else 34)
    blocks.view(-1)[:] = torch.randint(0, 256, (blocks.numel(),), generator=g, device=DEV, dtype=torch.uint8)
    d = _normal(g, (blocks.shape[0], 1), 2e-4 if fmt == "q4k" else 5e-4).abs().half()
    blocks[:, 0:2] = d.view(torch.uint8)
    if fmt == "q4k":
        blocks[:, 2:4] = (7.5 * d.float()).half().view(torch.uint8)
        blocks[:, 8:12] = blocks[:, 4:8]  # 6-bit minima equal to the scales
        low = blocks[:, 12:16] & 15
        blocks[:, 12:16] = low | (low << 4)


def _weights(g, fmt: str, n: int, k: int) -> torch.Tensor:
    w = torch.empty((n, _row_bytes(fmt, k)), dtype=torch.uint8, device=DEV)
    _fill_weights(g, fmt, w)
    return w


def _inputs(case: dict, seed: int) -> dict:
    """The tensors of a single-operator case, from the seed alone."""
    g, c, kind = _gen(seed), case, case["kind"]
    if kind == "gemv" or kind == "gemm_f32":
        m = c.get("m", 1)
        t = {"w": _weights(g, c["fmt"], c["n"], c["k"]), "x": _normal(g, (m, c["k"]))}
        if c["form"] == "norm_geglu":
            t["norm"] = _normal(g, (c["k"],), 0.1)
        if c["form"] == "residual":
            t["res"] = _normal(g, (m, c["n"]))
        return t
    if kind == "int4":
        n, k = c["n"], c["k"]
        return {"w": torch.randint(0, 256, (n, k // 2), generator=g, device=DEV, dtype=torch.uint8),
                "s": _normal(g, (n, k // 32), 0.02).abs().half(), "x": _normal(g, (c["m"], k))}
    if kind == "gemm_bf16":
        return {"w": _weights(g, "q4k", c["n"], c["k"]), "x": _normal(g, (c["m"], c["k"]), dtype=torch.bfloat16)}
    if kind == "attn_decode":
        rows = (c["hkv"], c["kv"]) if c["layout"] == 0 else (c["kv"], c["hkv"])
        shape = (c["batch"], *rows, c["d"])
        return {"q": _normal(g, (c["batch"], c["hq"], c["d"]), dtype=torch.float16 if c["f16"] else torch.float32),
                "k": _normal(g, shape, dtype=torch.float16), "v": _normal(g, shape, dtype=torch.float16)}
    if kind == "attn_bf16":
        kv = c["start"] + c["q"]
        return {"q": _normal(g, (c["q"], c["hq"], 128), dtype=torch.bfloat16),
                "k": _normal(g, (c["hkv"], kv, 128), dtype=torch.bfloat16),
                "v": _normal(g, (c["hkv"], kv, 128), dtype=torch.bfloat16)}
    kv = c["start"] + c["q"]
    return {"q": _normal(g, (c["q"], c["hq"], c["d"])),
            "k": _normal(g, (c["hkv"], kv, c["d"]), dtype=torch.float16),
            "v": _normal(g, (c["hkv"], kv, c["d"]), dtype=torch.float16)}


def _config(c: dict) -> DecoderConfig:
    return DecoderConfig(**{f: c[f] for f in MODEL_2B}, weight_format=c["fmt"], max_seq=_rows(c) + 8, eps=EPS)


def _rows(c: dict) -> int:
    """Cache rows that one pass of a decoder case writes."""
    return c["prompt"] + max(0, c["new"] - 1)


def _model_weights(c: dict, seed: int):
    """(name, layer, fill) of every weight tensor of the model in a fixed
    order; fill(out) writes the tensor's values in place."""
    g = _gen(seed)
    for li in range(c["layers"]):
        for name in ("wqkv", "wo", "wgu", "wd"):
            yield name, li, lambda out: _fill_weights(g, c["fmt"], out)
        for name in ("norm_attn", "norm_ffn"):
            yield name, li, lambda out: out.copy_(_normal(g, out.shape, 0.1))
    for name in ("embed", "lm_head"):
        yield name, None, lambda out: out.copy_(_normal(g, out.shape, 0.02, torch.float16))
    yield "norm_final", None, lambda out: out.copy_(_normal(g, out.shape, 0.1))


def _prompt_ids(c: dict, seed: int) -> np.ndarray:
    return np.random.default_rng(seed).integers(0, c["vocab"], c["prompt"]).astype(np.int32)


class Model:
    """A decoder in a serving program's hands: weights on the device, the
    decode step captured, a prompt."""

    def __init__(self, c: dict, seed: int):
        self.dec = Decoder(_config(c), keep_logits=True)
        typ = {1: "|u1", 2: "<f2", 4: "<f4"}
        for name, li, fill in _model_weights(c, seed):
            buf = getattr(self.dec if li is None else self.dec.layers[li], name)
            fill(over(buf, typ[buf.dtype.itemsize], buf.shape))
        rows = _rows(c)
        caches = [(L.k_cache, L.v_cache) for L in self.dec.layers]
        for k, v in caches:
            k.fill_zero()
            v.fill_zero()
        self.prompt = _prompt_ids(c, seed)
        self.stream = self.graph = None
        if c["kind"] == "decode":
            torch.cuda.synchronize()
            self.stream = Stream()
            self.dec.reset(self.prompt)
            self.dec.step(self.stream)
            self.stream.synchronize()
            self.graph = self.dec.capture(self.stream, 8)
        self.out = {"logits": over(self.dec.logits, "<f4", self.dec.logits.shape),
                    "k": [over(k, "<f2", k.shape)[:, :rows] for k, _ in caches],
                    "v": [over(v, "<f2", v.shape)[:, :rows] for _, v in caches]}

    def __del__(self):
        if self.graph is not None:
            self.graph.destroy()
        if self.stream is not None:
            self.stream.destroy()


# ---- the interface ----------------------------------------------------------------

def prepare(case: dict, seed: int) -> dict:
    doe_amd.init(0)
    if case["kind"] in ("decode", "prompt"):
        return {"case": case, "model": Model(case, seed)}
    c = case
    b = {name: Buf(t) for name, t in _inputs(case, seed).items()}
    dtype = torch.float32
    if c["kind"] in ("gemv", "gemm_f32"):
        shape = (c.get("m", 1), c["n"] // 2 if c["form"] == "norm_geglu" else c["n"])
    elif c["kind"] in ("int4", "gemm_bf16"):
        shape = (c["m"], c["n"])
    elif c["kind"] == "attn_decode":
        shape, dtype = (c["batch"], c["hq"], c["d"]), torch.float16 if c["f16"] else torch.float32
    else:
        shape = (c["q"], c["hq"], c.get("d", 128))
    b["y"] = Buf(torch.zeros(shape, dtype=dtype, device=DEV))
    return {"case": case, **b}


def run(state: dict):
    c, kind = state["case"], state["case"]["kind"]
    if kind == "decode":
        m = state["model"]
        ids = m.dec.generate(m.prompt, c["new"], m.stream, graph=m.graph, steps_per_graph=8)
        return {"ids": ids, **m.out}
    if kind == "prompt":
        m = state["model"]
        m.dec.prefill(m.prompt)
        return m.out
    y = state["y"]
    if kind == "gemv":
        if c["form"] == "plain":
            f = ops.matmul_q4k if c["fmt"] == "q4k" else ops.matmul_q8_0
            f(state["w"], state["x"], y, c["n"], c["k"])
        else:
            gated = c["form"] == "norm_geglu"
            ops.matmul_q4k_fused(state["w"], state["x"], y, c["n"], c["k"], norm_weight=state.get("norm"),
                                 norm_eps=EPS, residual=state.get("res"), gated=gated, weight_format=c["fmt"])
    elif kind == "int4":
        ops.matmul_int4g32(state["w"], state["s"], state["x"], y, c["m"], c["n"], c["k"])
    elif kind == "gemm_bf16":
        ops.matmul_q4k_gemm(state["x"], state["w"], y, c["m"], c["n"], c["k"])
    elif kind == "gemm_f32":
        ops.matmul_gemm_f32_fused(state["x"], state["w"], y, c["m"], c["n"], c["k"], c["fmt"],
                                  norm_weight=state.get("norm"), norm_eps=EPS, norm_weight_offset=True,
                                  residual=state.get("res"),
                                  activation=ops.GEGLU_PAIRS if c["form"] == "norm_geglu" else 0)
    elif kind == "attn_decode":
        ops.attention(state["q"], state["k"], state["v"], y, batch=c["batch"], num_heads=c["hq"],
                      num_kv_heads=c["hkv"], head_dim=c["d"], kv_len=c["kv"], kv_stride=c["kv"],
                      scale=1.0 / math.sqrt(c["d"]), q_f16=c["f16"], out_f16=c["f16"], softcap=c["softcap"],
                      sliding_window=c["window"], kv_layout=c["layout"])
    elif kind == "attn_bf16":
        ops.attention_prefill(state["q"], state["k"], state["v"], y, num_heads=c["hq"], num_kv_heads=c["hkv"],
                              head_dim=128, q_len=c["q"], kv_len=c["start"] + c["q"], start_pos=c["start"],
                              scale=1.0 / math.sqrt(128))
    else:
        kv = c["start"] + c["q"]
        ops.attention_prefill_f16kv(state["q"], state["k"], state["v"], y, num_heads=c["hq"], num_kv_heads=c["hkv"],
                                    head_dim=c["d"], query_len=c["q"], kv_len=kv, kv_stride=kv,
                                    start_pos=c["start"], scale=1.0 / math.sqrt(c["d"]), softcap=c["softcap"],
                                    sliding_window=c["window"])
    return y.t


def _pairs(q: int, start: int, window: int) -> int:
    """(query, key) pairs of a causal prompt of q tokens after `start` others."""
    pos = range(start + 1, start + q + 1)
    return sum(min(p, window) for p in pos) if window else sum(pos)


def _model_sizes(c: dict):
    qd, kvd, h = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"], c["hidden"]
    mats = [(qd + 2 * kvd, h), (h, qd), (2 * c["ffn"], h), (h, c["ffn"])]
    return c["layers"] * sum(n * _row_bytes(c["fmt"], k) for n, k in mats), c["layers"] * sum(n * k for n, k in mats)


def work(case: dict) -> dict:
    c, kind = case, case["kind"]
    if kind in ("gemv", "gemm_f32", "gemm_bf16"):
        m, n, k = c.get("m", 1), c["n"], c["k"]
        form = c.get("form", "plain")
        b = n * _row_bytes(c.get("fmt", "q4k"), k) + m * k * (2 if kind == "gemm_bf16" else 4)
        b += m * n * {"plain": 4, "residual": 8, "norm_geglu": 2}[form] + (4 * k if form == "norm_geglu" else 0)
        return {"bytes": b, "flops": 2 * m * n * k}
    if kind == "int4":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": n * k // 2 + n * k // 16 + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "attn_decode":
        keys = min(c["kv"], c["window"]) if c["window"] else c["kv"]
        b = 4 * c["batch"] * c["hkv"] * keys * c["d"] + 2 * c["batch"] * c["hq"] * c["d"] * (2 if c["f16"] else 4)
        return {"bytes": b, "flops": 4 * c["batch"] * c["hq"] * keys * c["d"]}
    if kind in ("attn_bf16", "attn_f16kv"):
        d, kv = c.get("d", 128), c["start"] + c["q"]
        b = 4 * c["hkv"] * kv * d + c["q"] * c["hq"] * d * (6 if kind == "attn_bf16" else 8)
        return {"bytes": b, "flops": 4 * c["hq"] * d * _pairs(c["q"], c["start"], c.get("window", 0))}
    wb, params = _model_sizes(c)
    head, rows = c["vocab"] * c["hidden"], _rows(c)
    kv_row = 4 * c["layers"] * c["kv_heads"] * c["head_dim"]
    attn = 4 * c["layers"] * c["heads"] * c["head_dim"] * _pairs(rows, 0, 0)
    passes = rows if kind == "decode" else 1  # a decode step reads every weight, a prompt reads them once
    kv = kv_row * (_pairs(rows, 0, 0) + rows if kind == "decode" else rows)
    return {"bytes": passes * (wb + 2 * head) + kv + 2 * rows * c["hidden"] + 4 * passes * c["vocab"],
            "flops": 2 * rows * params + 2 * passes * head + attn}


def tolerance(case: dict):
    """About four times the distance of each path from its 64-bit result."""
    return {
        "gemv": {"rel": 1.4e-5},        # 22-bit activations, f32 sums
        "int4": {"rel": 1.6e-5},
        "gemm_bf16": {"rel": 2e-3},     # weights rounded to f16
        "gemm_f32": {"rel": 5e-6},
        "attn_decode": {"rel": 1e-3 if case.get("f16") else 1e-5},  # f16 outputs
        "attn_bf16": {"rel": 7e-4},     # probabilities rounded to f16
        "attn_f16kv": {"rel": 7e-4},
        "decode": {"rel": 2.5e-3},      # f16 caches: roundings that differ travel through the layers
        "prompt": {"rel": 3e-3},        # and probabilities rounded to f16
    }[case["kind"]]


# ---- the same results in 64 bits ---------------------------------------------------

def _dequant(fmt: str, w: torch.Tensor, k: int) -> torch.Tensor:
    """Rows of weights [n][k] in float64."""
    n = w.shape[0]
    if fmt == "q8_0":
        b = w.view(n, -1, 34)
        d = b[:, :, 0:2].contiguous().view(torch.float16).double()
        return (d * b[:, :, 2:].contiguous().view(torch.int8).double()).view(n, -1)[:, :k]
    b = w.view(n, -1, 144)
    d = b[:, :, 0:2].contiguous().view(torch.float16).double()
    dmin = b[:, :, 2:4].contiguous().view(torch.float16).double()
    lo, hi, top = b[:, :, 4:8], b[:, :, 8:12], b[:, :, 12:16]
    sc = torch.cat([lo & 63, (top & 15) | ((lo >> 6) << 4)], 2).double() * d
    mn = torch.cat([hi & 63, (top >> 4) | ((hi >> 6) << 4)], 2).double() * dmin
    q = b[:, :, 16:].reshape(n, -1, 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], 3).reshape(n, -1, 8, 32).double()
    return (sc[..., None] * q - mn[..., None]).reshape(n, -1)[:, :k]


def _linear(x: torch.Tensor, fmt: str, w: torch.Tensor, k: int) -> torch.Tensor:
    """x [m][k] float64 times the rows of w, some rows at a time."""
    step = max(1, (1 << 27) // k)
    return torch.cat([x @ _dequant(fmt, w[i:i + step], k).t() for i in range(0, w.shape[0], step)], 1)


def _rmsnorm(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * (1.0 + w.double())


def _geglu_pairs(y: torch.Tensor) -> torch.Tensor:
    g, u = y[:, 0::2], y[:, 1::2]
    return 0.5 * g * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3))) * u


def _attend(q, k, v, start, window=0, softcap=0.0):
    """Causal attention in float64: q [m][hq][d] at positions start.., k and v [hkv][kv][d]."""
    m, hq, d = q.shape
    pos = torch.arange(start, start + m, device=DEV)[:, None]
    key = torch.arange(k.shape[1], device=DEV)[None, :]
    seen = (key <= pos) & (key > pos - window if window else key >= 0)
    out = torch.empty((m, hq, d), dtype=torch.float64, device=DEV)
    for h in range(hq):
        kv = h // (hq // k.shape[0])
        s = q[:, h].double() @ k[kv].double().t() / math.sqrt(d)
        if softcap:
            s = torch.tanh(s / softcap) * softcap
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[kv].double()
    return out


def _exact_model(c: dict, seed: int):
    hd, hq, hkv, h, n = c["head_dim"], c["heads"], c["kv_heads"], c["hidden"], c["prompt"]
    fmt, rows = c["fmt"], _rows(c)
    shapes = {"wqkv": ((hq + 2 * hkv) * hd, h), "wo": (h, hq * hd), "wgu": (2 * c["ffn"], h), "wd": (h, c["ffn"])}
    layers, top = [{} for _ in range(c["layers"])], {}
    for name, li, fill in _model_weights(c, seed):
        if name in shapes:
            t = torch.empty((shapes[name][0], _row_bytes(fmt, shapes[name][1])), dtype=torch.uint8, device=DEV)
        elif name in ("embed", "lm_head"):
            t = torch.empty((c["vocab"], h), dtype=torch.float16, device=DEV)
        else:
            t = torch.empty((h,), device=DEV)
        fill(t)
        (top if li is None else layers[li])[name] = t
    half = hd // 2
    inv = 10000.0 ** (-torch.arange(half, dtype=torch.float64, device=DEV) / half)
    caches, values = [[], []], [[], []]  # rounded to f16, as attention reads them, and before that

    def rotate(t, pos):
        """Rotation pairs (2i, 2i + 1) of each head of t [m][heads][hd]."""
        a = (pos[:, None] * inv[None, :])[:, None, :]
        x0, x1 = t[..., 0::2], t[..., 1::2]
        return torch.stack([x0 * torch.cos(a) - x1 * torch.sin(a), x0 * torch.sin(a) + x1 * torch.cos(a)],
                           -1).reshape(t.shape)

    def forward(ids, start):
        """Logits after the tokens `ids` at positions start..; their K and V rows join the caches."""
        m = len(ids)
        pos = torch.arange(start, start + m, dtype=torch.float64, device=DEV)
        x = top["embed"][torch.as_tensor(ids, device=DEV).long()].double()
        for li, L in enumerate(layers):
            qkv = _linear(_rmsnorm(x, L["norm_attn"]), fmt, L["wqkv"], h).view(m, hq + 2 * hkv, hd)
            q, k = rotate(qkv[:, :hq], pos), rotate(qkv[:, hq:hq + hkv], pos)
            for i, t in enumerate((k, qkv[:, hq + hkv:])):
                t = t.transpose(0, 1)
                for kept, rows in ((caches[i], t.half()), (values[i], t)):
                    if start == 0:
                        kept.append(rows)
                    else:
                        kept[li] = torch.cat([kept[li], rows], 1)
            x = x + _linear(_attend(q, caches[0][li], caches[1][li], start).view(m, -1), fmt, L["wo"], hq * hd)
            x = x + _linear(_geglu_pairs(_linear(_rmsnorm(x, L["norm_ffn"]), fmt, L["wgu"], h)), fmt, L["wd"], c["ffn"])
        y = _rmsnorm(x[-1], top["norm_final"])
        step = 1 << 15
        return torch.cat([top["lm_head"][i:i + step].double() @ y for i in range(0, c["vocab"], step)])

    logits = forward(_prompt_ids(c, seed), 0)
    for p in range(n, rows):  # greedy tokens
        logits = forward([int(torch.argmax(logits))], p)
    out = {"logits": logits, "k": values[0], "v": values[1]}
    return {"ids": None, **out} if c["kind"] == "decode" else out


def exact(case: dict, seed: int):
    c, kind = case, case["kind"]
    if kind in ("decode", "prompt"):
        return _exact_model(c, seed)
    t = _inputs(case, seed)
    if kind in ("gemv", "gemm_f32", "gemm_bf16"):
        x = t["x"].double()
        if "norm" in t:
            x = _rmsnorm(x, t["norm"])
        y = _linear(x, c.get("fmt", "q4k"), t["w"], c["k"])
        if "res" in t:
            y = y + t["res"].double()
        return _geglu_pairs(y) if c.get("form") == "norm_geglu" else y
    if kind == "int4":
        n, k = c["n"], c["k"]
        q = torch.stack([t["w"] & 15, t["w"] >> 4], -1).view(n, k // 32, 32).double() - 8.0
        w = (q * t["s"].double()[..., None]).view(n, k)
        return t["x"].double() @ w.t()
    if kind == "attn_decode":
        out = torch.empty((c["batch"], c["hq"], c["d"]), dtype=torch.float64, device=DEV)
        for b in range(c["batch"]):
            k, v = (t[x][b] if c["layout"] == 0 else t[x][b].transpose(0, 1) for x in ("k", "v"))
            out[b] = _attend(t["q"][b][None], k, v, c["kv"] - 1, c["window"], c["softcap"])[0]
        return out
    return _attend(t["q"], t["k"], t["v"], c["start"], c.get("window", 0), c.get("softcap", 0.0))
