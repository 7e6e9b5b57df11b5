"""Performance cases: what a user of kquant_amd has the library do.

Seven families, each through the public Python entry points:

  codec     quantize a weight to MXFP8 / MXFP4 and dequantize it again (baking
            a checkpoint and measuring its error)
  linear    the dense dequant-fused linear: bf16 or fp32 rows x MXFP8 / MXFP4
            weight, and the input-quantized MXFP8 x MXFP8 form
  moe       the routed expert forward over prepared MXFP4 experts (tiled or
            X4T-coded scales; bf16, MXFP8 or MXFP4 activations)
  hessian   the calibration Hessians: one layer's damped X^T X, and every
            expert's gate^2-weighted covariance
  ldl       the trellis encoder's block LDL of a stack of H2 matrices
  qsrt      activation rows x a packed QSRT matrix (serving)
  sqg       the SQG trellis encoder on the tiles of one 16-row slab

``listed()`` gives the fixed cases, ``draw(rng)`` further ones of the same
ranges.  A case is a dict of plain values; ``prepare`` builds the inputs and
the prepared weights from a seed, ``run`` makes one pass.  ``exact`` states
each result in float64 with plain torch.
"""

from __future__ import annotations

import math

import torch

from kquant_amd import candidate_hessian, exl3_encoder_backend, linear, moe, mxfp4, mxfp8, qsrt, sqg_quantizer
from kquant_amd.io import mxfp4 as mxfp4_io
from kquant_amd.sqg_e4m3 import SQG_XOR_CHEB_T12, sqg_codebook_bytes

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZEOF = {"bf16": 2, "f16": 2, "f32": 4}
DEVICE = "cuda"


# ------------------------------------------------------------------ cases --

def listed() -> list[dict]:
    return [
        # baking a checkpoint: one large dense weight to MXFP8 and back
        {"name": "codec_mxfp8_bake", "family": "codec", "fmt": "mxfp8", "dtype": "bf16", "rows": 12288, "k": 7168},
        # one decoded token through a dense MXFP8 linear: latency and weight bytes
        {"name": "linear_decode", "family": "linear", "op": "a16", "fmt": "mxfp8", "dtype": "bf16", "m": 1,
         "n": 12288, "k": 7168},
        # a ragged chunk of a prompt through the input-quantized linear
        {"name": "linear_mm_ragged", "family": "linear", "op": "mm", "fmt": "mxfp8", "dtype": "bf16", "m": 777,
         "n": 5000, "k": 7168},
        # a full prefill chunk through the same layer
        {"name": "linear_prefill", "family": "linear", "op": "a16", "fmt": "mxfp8", "dtype": "bf16", "m": 4096,
         "n": 12288, "k": 7168},
        # one decoded token through a routed MoE layer
        {"name": "moe_decode", "family": "moe", "tokens": 1, "experts": 384, "topk": 8, "hidden": 7168, "inter": 2048,
         "acts": "bf16", "scales": "tiled", "routing": "uniform", "activation": "situ", "out": "bf16"},
        # a mixed batch (decodes and short prompts), odd token count, fp32 sums
        {"name": "moe_batch", "family": "moe", "tokens": 333, "experts": 384, "topk": 8, "hidden": 7168,
         "inter": 2048, "acts": "bf16", "scales": "x4t", "routing": "zipf", "activation": "situ", "out": "f32"},
        # a full prefill batch
        {"name": "moe_prefill", "family": "moe", "tokens": 8192, "experts": 384, "topk": 8, "hidden": 7168,
         "inter": 2048, "acts": "bf16", "scales": "tiled", "routing": "zipf", "activation": "situ", "out": "f32"},
        # calibration: one layer's input Hessian, damped
        {"name": "hessian_layer", "family": "hessian", "form": "layer", "dtype": "bf16", "rows": 65536, "k": 7168,
         "weighted": False, "experts": 0},
        # calibration: the post-activation Hessians of a GPU's share of the experts
        {"name": "hessian_experts", "family": "hessian", "form": "grouped", "dtype": "bf16", "rows": 65536, "k": 2048,
         "weighted": True, "experts": 48},
        # encoding: factor the H2 matrices of a group of experts
        {"name": "ldl_experts", "family": "ldl", "batch": 16, "n": 2048},
        # serving a QSRT matrix to a small decode batch
        {"name": "qsrt_decode", "family": "qsrt", "m": 5, "k": 3584, "n": 3072, "dtype": "bf16", "axis": "n"},
        # encoding: the tiles of one 16-row slab of a weight of 7168 columns
        {"name": "sqg_encode", "family": "sqg", "tiles": 448, "bits": 3, "context": 128},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    family = rng.choice(["codec", "linear", "linear", "moe", "moe", "hessian", "ldl", "qsrt", "sqg"])
    if family == "codec":
        return {"family": family, "fmt": rng.choice(["mxfp8", "mxfp4"]), "dtype": rng.choice(["bf16", "bf16", "f32"]),
                "rows": _log_int(rng, 1, 12288), "k": 32 * rng.randint(8, 224)}
    if family == "linear":
        # the mm form takes K in its 128-column granule, as weights are laid out for it
        op = rng.choice(["a16", "a16", "mm"])
        dtype = rng.choice(["bf16", "bf16", "f32"])
        m = _log_int(rng, 1, 1024 if dtype == "f32" and op == "a16" else 4096)
        return {"family": family, "op": op, "fmt": "mxfp8" if op == "mm" else rng.choice(["mxfp8", "mxfp4"]),
                "dtype": dtype, "m": m, "n": _log_int(rng, 64, 12288),
                "k": 128 * rng.randint(4, 56) if op == "mm" else 64 * rng.randint(4, 112)}
    if family == "moe":
        return {"family": family, "tokens": _log_int(rng, 1, 4096), "experts": rng.choice([16, 48, 96, 128, 384]),
                "topk": rng.choice([2, 4, 8]), "hidden": 512 * rng.randint(4, 14), "inter": 512 * rng.randint(1, 4),
                "acts": rng.choice(["bf16", "bf16", "mxfp8", "mxfp4"]), "scales": rng.choice(["tiled", "x4t"]),
                "routing": rng.choice(["zipf", "uniform"]), "activation": rng.choice(["situ", "swiglu"]),
                "out": rng.choice(["bf16", "f32"])}
    if family == "hessian":
        form = rng.choice(["layer", "grouped", "routed"])
        dtype = rng.choice(["bf16", "bf16", "f32"])
        if form == "layer":
            return {"family": family, "form": form, "dtype": dtype,
                    "rows": _log_int(rng, 100, 65536 if dtype == "bf16" else 16384), "k": 8 * _log_int(rng, 32, 896),
                    "weighted": rng.choice([False, True]) and dtype == "bf16", "experts": 0}
        return {"family": family, "form": form, "dtype": dtype,
                "rows": _log_int(rng, 256, 65536 if dtype == "bf16" else 8192), "k": 8 * rng.randint(32, 256),
                "weighted": True, "experts": rng.randint(4, 48)}
    if family == "ldl":
        n = 16 * rng.randint(16, 128)
        return {"family": family, "batch": rng.randint(1, 16), "n": n}
    if family == "qsrt":
        return {"family": family, "m": _log_int(rng, 1, 1024), "k": 128 * rng.randint(2, 32),
                "n": 128 * rng.randint(2, 32), "dtype": rng.choice(["bf16", "bf16", "f32"]),
                "axis": rng.choice(["k", "n"])}
    return {"family": "sqg", "tiles": _log_int(rng, 16, 512), "bits": rng.choice([2, 3, 4]),
            "context": rng.choice([16, 64, 128])}


# ------------------------------------------------- plain formats, no library --

def _plain_quantize(x: torch.Tensor, fmt: str) -> tuple[torch.Tensor, torch.Tensor]:
    """The MX rule in plain torch: E4M3 bytes (or E2M1 codes 0..15) [R, K] and E8M0 bytes [R, K/32]."""
    b = x.double().reshape(x.shape[0], -1, 32)
    qmax = 448.0 if fmt == "mxfp8" else 6.0
    ratio = (b.abs().amax(-1).float().clamp(min=1e-30) / qmax).double()
    e = torch.log2(ratio).float().ceil().clamp(-127, 128)
    y = (b / torch.exp2(e.double())[..., None]).clamp(-qmax, qmax).float().reshape(x.shape)
    scale = (e + 127).to(torch.uint8)
    if fmt == "mxfp8":
        return y.to(torch.float8_e4m3fn).view(torch.uint8), scale
    a = y.abs()
    code = torch.zeros_like(a, dtype=torch.uint8)
    # midpoints between neighbouring E2M1 values; ties go to the even code
    for i, mid in enumerate((0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)):
        code += (a >= mid) if i % 2 else (a > mid)
    return code | (torch.signbit(y).to(torch.uint8) << 3), scale


def _plain_pack(codes: torch.Tensor) -> torch.Tensor:
    return codes[:, 0::2] | (codes[:, 1::2] << 4)


def _plain_values(q: torch.Tensor, scale: torch.Tensor, fmt: str) -> torch.Tensor:
    """float64 [R, K] of E4M3 bytes or packed E2M1 codes under E8M0 scales."""
    if fmt == "mxfp8":
        v = q.view(torch.float8_e4m3fn).double()
    else:
        lut = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0],
                           dtype=torch.float64, device=q.device)
        v = lut[torch.stack([q & 15, q >> 4], dim=-1).reshape(q.shape[0], -1).long()]
    f = torch.exp2(scale.double() - 127)
    return (v.reshape(*scale.shape, 32) * f[..., None]).reshape(v.shape)


def _weight(rows: int, k: int, fmt: str, std: float, g: torch.Generator) -> tuple[torch.Tensor, torch.Tensor]:
    """A normal weight in the MX format: (E4M3 bytes or packed E2M1, scales)."""
    q, s = _plain_quantize(torch.randn(rows, k, generator=g, device=DEVICE) * std, fmt)
    return (q if fmt == "mxfp8" else _plain_pack(q)), s


def _act64(g: torch.Tensor, u: torch.Tensor, activation: str) -> torch.Tensor:
    if activation == "situ":
        return 4.0 * torch.tanh(g / 4.0) * torch.sigmoid(g) * (25.0 * torch.tanh(u / 25.0))
    return g * torch.sigmoid(g) * u


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device=DEVICE).manual_seed(int(seed) * 7919 + 13)


def _student_t(rows: int, k: int, dtype: torch.dtype, g: torch.Generator) -> torch.Tensor:
    """Heavy-tailed activations (Student-t with 4 degrees of freedom)."""
    out = torch.empty(rows, k, dtype=dtype, device=DEVICE)
    for r0 in range(0, rows, 16384):
        n = min(16384, rows - r0)
        z = torch.randn(n, k, generator=g, device=DEVICE)
        chi = sum(torch.randn(n, k, generator=g, device=DEVICE).square() for _ in range(4))
        out[r0:r0 + n] = (z / torch.sqrt(chi / 4)).to(dtype)
    return out


def _routing(tokens: int, experts: int, topk: int, kind: str, g: torch.Generator):
    """Distinct experts per token and their renormalized weights; ``zipf``
    gives the experts the popularity rank^-1.1."""
    logits = torch.randn(tokens, experts, generator=g, device=DEVICE)
    if kind == "zipf":
        rank = torch.randperm(experts, generator=g, device=DEVICE) + 1
        logits = logits - 1.1 * torch.log(rank.float())
    top, ids = torch.topk(torch.softmax(logits, -1), topk, dim=-1)
    return ids.to(torch.int32), (top / top.sum(-1, keepdim=True)).float()


# ----------------------------------------------------------------- inputs --

def _codec_inputs(c, g):
    w = torch.randn(c["rows"], c["k"], generator=g, device=DEVICE) * 0.02
    w = torch.where(torch.rand(w.shape, generator=g, device=DEVICE) < 1e-3, w * 20.0, w)  # a few outliers
    return w.to(DTYPES[c["dtype"]])


def _linear_inputs(c, g):
    channel = torch.exp(0.5 * torch.randn(c["k"], generator=g, device=DEVICE))
    x = (torch.randn(c["m"], c["k"], generator=g, device=DEVICE) * channel).to(DTYPES[c["dtype"]])
    return x, *_weight(c["n"], c["k"], c["fmt"], 0.015, g)


def _moe_inputs(c, g):
    x = torch.randn(c["tokens"], c["hidden"], generator=g, device=DEVICE).to(torch.bfloat16)
    ids, weights = _routing(c["tokens"], c["experts"], c["topk"], c["routing"], g)
    h, i, n = c["hidden"], c["inter"], c["experts"]
    w13 = torch.empty(n, 2 * i, h // 2, dtype=torch.uint8, device=DEVICE)
    s13 = torch.empty(n, 2 * i, h // 32, dtype=torch.uint8, device=DEVICE)
    w2 = torch.empty(n, h, i // 2, dtype=torch.uint8, device=DEVICE)
    s2 = torch.empty(n, h, i // 32, dtype=torch.uint8, device=DEVICE)
    for e in range(n):
        w13[e], s13[e] = _weight(2 * i, h, "mxfp4", 0.02, g)
        w2[e], s2[e] = _weight(h, i, "mxfp4", 0.02, g)
    return x, ids, weights, w13, s13, w2, s2


def _hessian_inputs(c, g):
    dtype = DTYPES[c["dtype"]]
    if c["form"] == "layer":
        x = _student_t(c["rows"], c["k"], dtype, g)
        return x, torch.rand(c["rows"], generator=g, device=DEVICE) if c["weighted"] else None
    topk = min(8, c["experts"])
    tokens = max(1, c["rows"] // topk)
    ids, gates = _routing(tokens, c["experts"], topk, "zipf", g)
    if c["form"] == "routed":
        return _student_t(tokens, c["k"], dtype, g), ids, gates
    counts = torch.bincount(ids.flatten().long(), minlength=c["experts"])
    offsets = torch.zeros(c["experts"] + 1, dtype=torch.int64)
    offsets[1:] = torch.cumsum(counts, 0).cpu()
    return (_student_t(tokens * topk, c["k"], dtype, g), offsets,
            torch.rand(tokens * topk, generator=g, device=DEVICE))


def _ldl_inputs(c, g):
    n = c["n"]
    h = torch.empty(c["batch"], n, n, device=DEVICE)
    for e in range(c["batch"]):
        x = _student_t(2 * n, n, torch.float32, g)
        h[e] = x.T @ x / (2 * n)
        h[e] = (h[e] + h[e].T) / 2
        h[e].diagonal().add_(0.025 * h[e].diagonal().mean())
    return h


def _qsrt_inputs(c, g):
    records = (c["k"] if c["axis"] == "k" else c["n"]) // 128
    bits = [3] * records  # mixed rates around K3, as a byte budget allocates them
    for r in range(records // 6):
        bits[r], bits[records - 1 - r] = 4, 2
    tiles = 8 * ((c["n"] if c["axis"] == "k" else c["k"]) // 16)
    words = sum(16 * tiles * b for b in bits)
    payload = torch.randint(-32768, 32768, (words,), generator=g, device=DEVICE, dtype=torch.int32).to(torch.int16)
    x = torch.randn(c["m"], c["k"], generator=g, device=DEVICE).to(DTYPES[c["dtype"]])
    suh = torch.where(torch.rand(c["k"], generator=g, device=DEVICE) < 0.5, -1.0, 1.0)
    svh = 0.02 * (0.5 + torch.rand(c["n"], generator=g, device=DEVICE))
    return x, payload, bits, suh, svh


def prepare(case: dict, seed: int) -> dict:
    c, g = case, _generator(seed)
    family = c["family"]
    if family == "codec":
        return {"case": c, "w": _codec_inputs(c, g)}
    if family == "linear":
        x, w, s = _linear_inputs(c, g)
        return {"case": c, "x": x, "w": w.view(torch.float8_e4m3fn) if c["fmt"] == "mxfp8" else w, "s": s}
    if family == "moe":
        x, ids, weights, w13, s13, w2, s2 = _moe_inputs(c, g)
        experts = moe.prepare_expert_weights(w13, s13, w2, s2, scale_format=c["scales"])
        return {"case": c, "x": x, "ids": ids, "weights": weights, "experts": experts}
    if family == "hessian":
        return {"case": c, "in": _hessian_inputs(c, g)}
    if family == "ldl":
        return {"case": c, "h": _ldl_inputs(c, g)}
    if family == "qsrt":
        x, payload, bits, suh, svh = _qsrt_inputs(c, g)
        out = torch.empty(c["m"], c["n"], dtype=x.dtype, device=DEVICE)
        launch = qsrt.qsrt_linear_launcher(x, payload, out, k_tiles=c["k"] // 16, n_tiles=c["n"] // 16,
                                           rate_axis=c["axis"], record_bits=bits, suh=suh, svh=svh)
        return {"case": c, "launch": launch, "out": out}
    tiles = torch.randn(c["tiles"], 256, generator=g, device=DEVICE)
    lut = sqg_codebook_bytes(c["bits"], SQG_XOR_CHEB_T12, device=torch.device(DEVICE, torch.cuda.current_device()))
    return {"case": c, "tiles": tiles, "lut": lut}


# -------------------------------------------------------------------- run --

def run(state: dict):
    c = state["case"]
    family = c["family"]
    if family == "codec":
        dtype = DTYPES[c["dtype"]]
        if c["fmt"] == "mxfp8":
            q, s = mxfp8.mxfp8_quantize(state["w"])
            return q.view(torch.uint8), s, mxfp8.mxfp8_dequantize(q, s, dtype=dtype)
        q, s = mxfp4.mxfp4_quantize(state["w"])
        return q, s, mxfp4_io.dequant(q, s, dtype=dtype)
    if family == "linear":
        if c["op"] == "mm":
            return linear.mxfp8_linear_mm(state["x"], state["w"], state["s"])
        f = linear.mxfp8_linear if c["fmt"] == "mxfp8" else linear.mxfp4_linear
        return f(state["x"], state["w"], state["s"])
    if family == "moe":
        return moe.grouped_expert_forward(state["x"], state["ids"], state["weights"], state["experts"],
                                          activation=c["activation"], out_dtype=DTYPES[c["out"]],
                                          activation_format=c["acts"])
    if family == "hessian":
        if c["form"] == "layer":
            return candidate_hessian.damped_hessian(*state["in"], damp=0.01)
        if c["form"] == "grouped":
            rows, offsets, gates = state["in"]
            return candidate_hessian.expert_hessians_from_rows(rows, offsets, gates, square_weights=True)
        rows, ids, gates = state["in"]
        return candidate_hessian.expert_hessians(rows, ids, gates, c["experts"])
    if family == "ldl":
        return exl3_encoder_backend.block_ldl_batched(state["h"], 16)
    if family == "qsrt":
        state["launch"]()
        return state["out"]
    return sqg_quantizer.quantize_tiles_sqg(state["tiles"], state["lut"], c["bits"], c["context"])


# ------------------------------------------------------------ bytes, flops --

def _active(experts: int, tokens: int, topk: int, kind: str) -> float:
    """Distinct experts a batch routes to (expected, or of one such routing)."""
    if kind == "uniform":
        return experts * (1.0 - (1.0 - topk / experts) ** tokens)
    g = torch.Generator().manual_seed(0)
    logits = torch.randn(tokens, experts, generator=g) - 1.1 * torch.log(torch.arange(1, experts + 1).float())
    return float(torch.unique(torch.topk(logits, topk, dim=-1).indices).numel())


def work(case: dict) -> dict:
    c = case
    family = c["family"]
    if family == "codec":
        n, z = c["rows"] * c["k"], SIZEOF[c["dtype"]]
        packed = n * (1.0 if c["fmt"] == "mxfp8" else 0.5) + n / 32
        return {"bytes": (n * z + packed) + (packed + n * z), "flops": 0}
    if family == "linear":
        m, n, k = c["m"], c["n"], c["k"]
        wbytes = n * k * (1.0 if c["fmt"] == "mxfp8" else 0.5) + n * k / 32
        z = SIZEOF[c["dtype"]]
        zout = 2 if c["op"] == "mm" else z
        return {"bytes": wbytes + m * k * z + m * n * zout, "flops": 2.0 * m * n * k}
    if family == "moe":
        pairs = c["tokens"] * c["topk"]
        per = 3 * c["inter"] * c["hidden"]
        used = _active(c["experts"], c["tokens"], c["topk"], c["routing"])
        return {"bytes": used * (per / 2 + per / 32) + c["tokens"] * c["hidden"] * (2 + SIZEOF[c["out"]]),
                "flops": 2.0 * pairs * per}
    if family == "hessian":
        n, k, z = c["rows"], c["k"], SIZEOF[c["dtype"]]
        if c["form"] == "layer":
            return {"bytes": n * k * z + 4.0 * k * k, "flops": 1.0 * n * k * (k + 1)}
        topk = min(8, c["experts"])
        rows = max(1, n // topk) * (topk if c["form"] == "grouped" else 1)
        pairs = max(1, n // topk) * topk
        return {"bytes": rows * k * z + 4.0 * c["experts"] * k * k, "flops": 1.0 * pairs * k * (k + 1)}
    if family == "ldl":
        return {"bytes": 8.0 * c["batch"] * c["n"] ** 2, "flops": c["batch"] * c["n"] ** 3 / 3.0}
    if family == "qsrt":
        m, k, n, z = c["m"], c["k"], c["n"], SIZEOF[c["dtype"]]
        return {"bytes": k * n * 3 / 8 + m * (k + n) * z, "flops": 2.0 * m * n * k}
    # one edge evaluation: a difference, a fused multiply-add and a compare
    steps = 256 + 2 * c["context"]
    return {"bytes": c["tiles"] * 256 * 10.0, "flops": c["tiles"] * steps * 65536 * 4.0}


# -------------------------------------------------------------- tolerance --

def tolerance(case: dict):
    """Largest relative difference another correct implementation of the same
    precision shows: about four times the distance from ``exact`` measured over
    the declared ranges (given beside each)."""
    c = case
    family = c["family"]
    if family in ("codec", "sqg"):
        return "exact"
    if family == "linear":
        # fp32 sums 1.0e-6; one rounding to bf16 1.67e-3
        return {"rel": 5e-6 if c["dtype"] == "f32" and c["op"] == "a16" else 7e-3}
    if family == "moe":
        if c["out"] == "bf16":
            return {"rel": 7e-3}  # 1.75e-3
        # the intermediate moves by one rounding step where its sum straddles it
        # (5.2e-5 / 2.8e-4); the E4M3 x E2M1 products themselves sum to 6.3e-4
        return {"rel": {"bf16": 2e-4, "mxfp8": 2.5e-3, "mxfp4": 1.2e-3}[c["acts"]]}
    if family == "hessian":
        # fp32 rows in two bf16 terms 4.7e-6, weighted bf16 rows 2.6e-6, exact products 1.2e-6
        return {"rel": 2e-5 if c["dtype"] == "f32" else 1e-5 if c["weighted"] else 5e-6}
    if family == "ldl":
        return {"rel": 1e-6}  # 1.0e-7 against float64; fp32 factors of the same matrices agree less closely
    # fp32 rows 1.7e-7; bf16 rows 2.4e-3 (rounded to bf16 after their rotation in the prefill form)
    return {"rel": 1e-6 if c["dtype"] == "f32" else 1e-2}


# ------------------------------------------------------------------ exact --

def _exact_moe(c, g):
    x, ids, weights, w13, s13, w2, s2 = _moe_inputs(c, g)

    def rounded(v):  # what the activation format keeps of a row, in float64
        if c["acts"] == "bf16":
            return v.to(torch.bfloat16).double()
        q, s = _plain_quantize(v.to(torch.bfloat16), c["acts"])
        return _plain_values(q if c["acts"] == "mxfp8" else _plain_pack(q), s, c["acts"])

    xr = rounded(x)
    out = torch.zeros(c["tokens"], c["hidden"], dtype=torch.float64, device=DEVICE)
    for e in torch.unique(ids).tolist():
        token, slot = torch.nonzero(ids == e, as_tuple=True)
        gu = xr[token] @ _plain_values(w13[e], s13[e], "mxfp4").T
        a = rounded(_act64(gu[:, :c["inter"]], gu[:, c["inter"]:], c["activation"]))
        y = a @ _plain_values(w2[e], s2[e], "mxfp4").T
        out.index_add_(0, token, weights[token, slot].double()[:, None] * y)
    return out


def _exact_hessian(c, g):
    inputs = _hessian_inputs(c, g)

    def covariance(x, w):
        x = x.double()
        total = w.sum()
        h = x.T @ (x * w[:, None])
        return (h / total if float(total) > 0 else torch.zeros_like(h)), total

    if c["form"] == "layer":
        x, w = inputs
        h, total = covariance(x, torch.ones(x.shape[0], dtype=torch.float64, device=DEVICE) if w is None
                              else w.double())
        h.diagonal().add_(0.01 * h.diagonal().mean())
        return h, float(total)
    groups = []
    if c["form"] == "grouped":
        rows, offsets, gates = inputs
        o = offsets.tolist()
        groups = [covariance(rows[a:b], gates[a:b].double().square()) for a, b in zip(o[:-1], o[1:])]
        return torch.stack([h for h, _ in groups]), torch.stack([t for _, t in groups])
    rows, ids, gates = inputs
    counts = []
    for e in range(c["experts"]):
        token, slot = torch.nonzero(ids == e, as_tuple=True)
        groups.append(covariance(rows[token], gates[token, slot].double().square()))
        counts.append(int(token.numel()))
    return (torch.stack([h for h, _ in groups]), torch.stack([t for _, t in groups]),
            torch.tensor(counts, dtype=torch.int64))


def _exact_ldl(c, g):
    h = _ldl_inputs(c, g).double()
    lower = torch.linalg.cholesky(h.cpu() if c["batch"] == 1 else h).to(DEVICE)
    for i in range(0, c["n"], 16):
        d = lower[:, i:i + 16, i:i + 16].clone()
        lower[:, i:, i:i + 16] = lower[:, i:, i:i + 16] @ torch.linalg.inv(d)
        lower[:, i:i + 16, i:i + 16] = torch.eye(16, dtype=torch.float64, device=DEVICE)
    return lower, torch.zeros(c["batch"], dtype=torch.int32)


def _hadamard128() -> torch.Tensor:
    h = torch.ones(1, 1, dtype=torch.float64, device=DEVICE)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(128.0)


def _exact_qsrt(c, g):
    """The trellis format in plain torch: 16 K-bit words per span with adjacent
    words exchanged, MSB first; a state is the 16 stream bits that end at its
    symbol (cyclic); labels are E4M3 bytes of the codebook (data, not code)."""
    x, payload, bits, suh, svh = _qsrt_inputs(c, g)
    kt, nt = c["k"] // 16, c["n"] // 16
    place = torch.empty(256, dtype=torch.long)
    for t in range(32):
        for j in range(8):
            place[8 * t + j] = (2 * (t % 4) + (0, 1, 8, 9)[j % 4]) * 16 + t // 4 + 8 * (j // 4)
    place = place.to(DEVICE)
    w = torch.empty(c["k"], c["n"], dtype=torch.float64, device=DEVICE)
    labels = {b: sqg_codebook_bytes(b, SQG_XOR_CHEB_T12, rate_axis=c["axis"], device=payload.device)
              .view(torch.float8_e4m3fn).double() for b in set(bits)}
    cursor, per = 0, 8 * (nt if c["axis"] == "k" else kt)
    for record, b in enumerate(bits):
        words = payload[cursor:cursor + per * 16 * b].to(torch.int64) & 0xFFFF
        cursor += per * 16 * b
        words = words.reshape(per, -1, 2).flip(-1).reshape(per, -1)
        shifts = torch.arange(15, -1, -1, device=DEVICE)
        stream = ((words[..., None] >> shifts) & 1).reshape(per, 256 * b)
        ends = (torch.arange(256, device=DEVICE)[:, None] + 1) * b - 16 + torch.arange(16, device=DEVICE)
        states = (stream[:, ends % (256 * b)] << shifts).sum(-1)
        tiles = torch.empty(per, 256, dtype=torch.float64, device=DEVICE)
        tiles[:, place] = labels[b][states]
        if c["axis"] == "k":
            block = tiles.reshape(8, nt, 16, 16).permute(0, 2, 1, 3).reshape(128, c["n"])
            w[128 * record:128 * record + 128] = block
        else:
            block = tiles.reshape(kt, 8, 16, 16).permute(0, 2, 1, 3).reshape(c["k"], 128)
            w[:, 128 * record:128 * record + 128] = block
    had = _hadamard128()
    xr = ((x.double() * suh.double()).reshape(-1, 128) @ had).reshape(x.shape)
    y = xr @ w
    return (y.reshape(-1, 128) @ had).reshape(y.shape) * svh.double()


def exact(case: dict, seed: int):
    c, g = case, _generator(seed)
    family = c["family"]
    if family == "codec":
        w = _codec_inputs(c, g)
        q, s = _plain_quantize(w, c["fmt"])
        q = q if c["fmt"] == "mxfp8" else _plain_pack(q)
        return q, s, _plain_values(q, s, c["fmt"])
    if family == "linear":
        x, w, s = _linear_inputs(c, g)
        xv = _plain_values(*_plain_quantize(x, "mxfp8"), "mxfp8") if c["op"] == "mm" else x.double()
        return xv @ _plain_values(w, s, c["fmt"]).T
    if family == "moe":
        return _exact_moe(c, g)
    if family == "hessian":
        return _exact_hessian(c, g)
    if family == "ldl":
        return _exact_ldl(c, g)
    if family == "qsrt":
        return _exact_qsrt(c, g)
    return None  # trellis states and the label values they select: whole numbers
