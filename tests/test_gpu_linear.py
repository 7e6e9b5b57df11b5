"""GPU parity of the dequant-fused MX linear kernel (kq_mx_linear).

Oracle: fp32 matmul of the bf16 activations and the reference-dequantized
weights (scripts/closure_mxfp8_mlp.py:146-160).  Bars:
  fp32 output: max |C - R| / max |R| <= 2e-3 (observed ~1e-6: products are
      exact, only the summation order differs);
  bf16 output: the rounding of the output alone reaches 2^-8 of an element,
      so C is compared with the oracle rounded to bf16 (as the reference's
      closure does, scripts/closure_mxfp8_mlp.py:184-186): every element
      within one bf16 ulp (+ 1e-5 max|R| for cancellation) of it, >= 99%
      bitwise equal, and
      |C - R| <= 2^-8 |R| + 1e-5 max|R| elementwise.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from kquant_amd import linear, workloads
from kquant_amd import mxfp4 as kq_mxfp4
from kquant_amd import mxfp8
from kquant_amd.io import mxfp4 as io_mxfp4

pytestmark = pytest.mark.gpu

TOL = 2e-3


def _max_rel(ref: np.ndarray, got: np.ndarray) -> float:
    return float(np.abs(got.astype(np.float64) - ref).max() / np.abs(ref).max())


def check_bf16_output(ref: np.ndarray, got: np.ndarray) -> None:
    """got: bf16 kernel output as float; ref: fp32/f64 oracle."""
    ref = np.asarray(ref, dtype=np.float64)
    r16 = oracle.round_bf16(ref.astype(np.float32)).astype(np.float64)
    slack = 1e-5 * np.abs(ref).max()  # fp32 summation-order slack (cancellation)
    ulp = np.abs(r16) * 2.0 ** -7 + slack
    assert np.all(np.abs(got - r16) <= ulp), "an element is more than one bf16 ulp off"
    assert np.mean(got == r16) >= 0.99
    bound = np.abs(ref) * 2.0 ** -8 + 1e-5 * np.abs(ref).max()
    assert np.all(np.abs(got - ref) <= bound)


def _quantized(fmt, w):
    if fmt == "mxfp8":
        q, s = mxfp8.mxfp8_quantize(w)
        return q, s, oracle.mx_dequant("mxfp8", q.view(torch.uint8).cpu().numpy(), s.cpu().numpy())
    q, s = kq_mxfp4.mxfp4_quantize(w)
    return q, s, oracle.mx_dequant("mxfp4", q.cpu().numpy(), s.cpu().numpy())


@pytest.mark.parametrize("fmt", ["mxfp8", "mxfp4"])
@pytest.mark.parametrize("m,n,k", [(256, 256, 1024), (300, 257, 192), (1, 100, 64), (17, 512, 2048), (513, 1000, 448)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_linear_matches_fp32_oracle(gpu, fmt, m, n, k, out_dtype):
    print(f"case linear {fmt} m={m} n={n} k={k} {out_dtype}", flush=True)
    g = torch.Generator().manual_seed(m * 7 + n)
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    x = (torch.randn(m, k, generator=g) * torch.exp(0.5 * torch.randn(k, generator=g))).to(torch.bfloat16)
    q, s, wd = _quantized(fmt, w)
    fn = linear.mxfp8_linear if fmt == "mxfp8" else linear.mxfp4_linear
    c = fn(x.to(gpu), q, s, out_dtype=out_dtype).float().cpu().numpy()
    ref = x.float().numpy().astype(np.float64) @ wd.astype(np.float64).T
    if out_dtype == torch.float32:
        assert _max_rel(ref, c) <= TOL
        assert _max_rel(ref, c) <= 1e-5
    else:
        check_bf16_output(ref, c)


@pytest.mark.parametrize("fmt", ["mxfp8", "mxfp4"])
def test_linear_many_tiles_per_workgroup(gpu, fmt):
    """17 x 17 tiles of 256 (more than one per workgroup of the persistent
    grid) with ragged last rows and columns."""
    m, n, k = 4200, 4200, 256
    g = torch.Generator().manual_seed(3)
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    q, s, wd = _quantized(fmt, w)
    fn = linear.mxfp8_linear if fmt == "mxfp8" else linear.mxfp4_linear
    c = fn(x.to(gpu), q, s, out_dtype=torch.float32).cpu().numpy()
    ref = x.float().numpy() @ wd.T.astype(np.float32)
    assert _max_rel(ref.astype(np.float64), c) <= 1e-5


@pytest.mark.parametrize("fmt", ["mxfp8", "mxfp4"])
@pytest.mark.parametrize("k", [384, 192])
def test_linear_fp32_source(gpu, fmt, k):
    """fp32 activations: the exact three-term bf16 split (A has 3k columns,
    column j multiplies weight column j % k); k = 384 takes the direct-to-LDS
    kernel, k = 192 the register-staged one."""
    m, n = 300, 520
    g = torch.Generator().manual_seed(k)
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    x = torch.randn(m, k, generator=g) * torch.exp(torch.randn(k, generator=g))
    q, s, wd = _quantized(fmt, w)
    fn = linear.mxfp8_linear if fmt == "mxfp8" else linear.mxfp4_linear
    c = fn(x.to(gpu), q, s).cpu().numpy()
    assert c.dtype == np.float32
    ref = x.double().numpy() @ wd.astype(np.float64).T
    assert _max_rel(ref, c) <= 1e-5


def test_cfg2_full_size(gpu):
    """X [4096, 7168] x MXFP8 W [12288, 7168] (benchmark configuration 2);
    the oracle is evaluated on 256 sampled rows of X."""
    w = workloads.cfg2_weight().to(gpu)
    x = workloads.cfg2_activations()
    q, s = mxfp8.mxfp8_quantize(w)
    c = linear.mxfp8_linear(x.to(gpu), q, s)
    rows = np.random.default_rng(0).choice(4096, 256, replace=False)
    wd = oracle.mx_dequant("mxfp8", q.view(torch.uint8).cpu().numpy(), s.cpu().numpy())
    ref = x[rows].float().numpy() @ wd.T
    got = c[torch.from_numpy(rows).to(gpu)].float().cpu().numpy()
    check_bf16_output(ref, got)
    c32 = linear.mxfp8_linear(x[rows].to(gpu), q, s, out_dtype=torch.float32).cpu().numpy()
    rel = _max_rel(ref.astype(np.float64), c32)
    print(f"cfg2 fp32-output max-rel {rel:.3e}", flush=True)
    assert rel <= TOL


def test_linear_rejects_bad_shapes(gpu):
    x = torch.zeros(4, 96, dtype=torch.bfloat16, device=gpu)
    q = torch.zeros(8, 96, dtype=torch.uint8, device=gpu)
    s = torch.zeros(8, 3, dtype=torch.uint8, device=gpu)
    with pytest.raises(ValueError, match="multiple of 64"):
        linear.mxfp8_linear(x, q, s)


# ------------------------------------------------- MXFP8 x MXFP8 (A8W8) --
# Oracle: scripts/closure_mxfp8_mlp.py:146-160 (_reference_from_packed): the
# input rows quantized with the kernel's quantizer (here the oracle's own
# restatement of the MXFP8 rule, itself pinned bit-exact elsewhere), both
# operands dequantized, the product in float64.  The block-scaled fp8 matrix
# cores do not sum a step's 64 products exactly in fp32 (an in-bounds probe of
# one instruction measured ~1e-5 relative), so the bars are the GEMM bar of the
# spec, max |C - R| / max |R| <= 2e-3, a normwise bar five times the measured
# error (relative L2 ~2e-5 at every shape here, cfg2 included), and for bf16
# output the closure's comparison after rounding the oracle
# (scripts/closure_mxfp8_mlp.py:184-186) within one bf16 ulp, with the share of
# bitwise-equal elements printed.
A8_NORM_TOL = 1e-4


def _a8_oracle(x: torch.Tensor, wq: torch.Tensor, ws: torch.Tensor) -> tuple[np.ndarray, np.ndarray, np.ndarray]:
    bits = x.contiguous().view(torch.int16).numpy().view(np.uint16)
    xq, xs = oracle.mx_quantize("mxfp8", bits, "bf16")
    xd = oracle.mx_dequant("mxfp8", xq, xs).astype(np.float64)
    wd = oracle.mx_dequant("mxfp8", wq.view(torch.uint8).cpu().numpy(), ws.cpu().numpy()).astype(np.float64)
    return xd @ wd.T, xq, xs


def _rel_l2(ref: np.ndarray, got: np.ndarray) -> float:
    return float(np.linalg.norm(got.astype(np.float64) - ref) / np.linalg.norm(ref))


def check_a8_bf16_output(ref: np.ndarray, got: np.ndarray) -> float:
    r16 = oracle.round_bf16(ref.astype(np.float32)).astype(np.float64)
    slack = A8_NORM_TOL * np.abs(ref).max()
    assert np.all(np.abs(got - r16) <= np.abs(r16) * 2.0 ** -7 + slack), "an element is more than one bf16 ulp off"
    assert np.all(np.abs(got - ref) <= np.abs(ref) * 2.0 ** -8 + slack)
    return float(np.mean(got == r16))


@pytest.mark.parametrize("m,n,k", [(256, 256, 1024), (300, 257, 384), (1, 100, 128), (17, 512, 2048),
                                   (513, 1000, 640), (4200, 520, 256)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_linear_a8_matches_operand_exact_oracle(gpu, m, n, k, out_dtype):
    print(f"case linear a8 m={m} n={n} k={k} {out_dtype}", flush=True)
    g = torch.Generator().manual_seed(m * 11 + n + k)
    w = (torch.randn(n, k, generator=g) * 0.015).to(torch.bfloat16).to(gpu)
    x = (torch.randn(m, k, generator=g) * torch.exp(0.5 * torch.randn(k, generator=g))).to(torch.bfloat16)
    q, s = mxfp8.mxfp8_quantize(w)
    ref, xq, xs = _a8_oracle(x, q, s)
    c = linear.mxfp8_linear_mm(x.to(gpu), q, s, out_dtype=out_dtype).float().cpu().numpy()
    # the same product from the oracle's quantized rows: the kernel's input quantizer is the oracle's rule
    c2 = linear.mxfp8_linear_mx(torch.from_numpy(xq).to(gpu), torch.from_numpy(xs).to(gpu), q, s,
                                out_dtype=out_dtype).float().cpu().numpy()
    assert np.array_equal(c, c2)
    rel, l2 = _max_rel(ref, c), _rel_l2(ref, c)
    if out_dtype == torch.float32:
        print(f"  fp32 out: max-rel {rel:.2e} rel-L2 {l2:.2e}", flush=True)
        assert rel <= TOL and l2 <= A8_NORM_TOL
    else:
        eq = check_a8_bf16_output(ref, c)
        print(f"  bf16 out: max-rel {rel:.2e} bitwise-equal {eq:.4f}", flush=True)


def test_linear_a8_cfg2_full_size(gpu):
    """Benchmark configuration 2 in the production operand form: X [4096,
    7168] bf16 quantized per row to MXFP8, times the MXFP8 W [12288, 7168].
    The oracle runs on 192 rows: the first and last row of each of the 16
    row tiles plus 160 sampled ones, against every column (all 48 column
    tiles)."""
    w = workloads.cfg2_weight().to(gpu)
    x = workloads.cfg2_activations()
    q, s = mxfp8.mxfp8_quantize(w)
    c = linear.mxfp8_linear_mm(x.to(gpu), q, s)
    c32 = linear.mxfp8_linear_mm(x.to(gpu), q, s, out_dtype=torch.float32)
    again = linear.mxfp8_linear_mm(x.to(gpu), q, s)
    assert torch.equal(c, again)
    edges = np.concatenate([np.arange(0, 4096, 256), np.arange(255, 4096, 256)])
    rest = np.setdiff1d(np.arange(4096), edges)
    rows = np.sort(np.concatenate([edges, np.random.default_rng(0).choice(rest, 160, replace=False)]))
    ref, _, _ = _a8_oracle(x[rows], q, s)
    sel = torch.from_numpy(rows).to(gpu)
    eq = check_a8_bf16_output(ref, c[sel].float().cpu().numpy())
    got32 = c32[sel].cpu().numpy()
    rel, l2 = _max_rel(ref, got32), _rel_l2(ref, got32)
    print(f"cfg2 a8: fp32-output max-rel {rel:.2e} rel-L2 {l2:.2e}; bf16 bitwise-equal {eq:.4f}", flush=True)
    assert rel <= TOL and l2 <= A8_NORM_TOL


def test_linear_a8_pads_k(gpu):
    """K = 96 (not a multiple of 128): source and weight are zero-padded to
    128, which adds nothing."""
    m, n, k = 33, 70, 96
    g = torch.Generator().manual_seed(96)
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    x = torch.randn(m, k, generator=g).to(torch.bfloat16)
    q, s = mxfp8.mxfp8_quantize(w)
    ref, _, _ = _a8_oracle(x, q, s)
    c = linear.mxfp8_linear_mm(x.to(gpu), q, s, out_dtype=torch.float32).cpu().numpy()
    assert _max_rel(ref, c) <= TOL and _rel_l2(ref, c) <= A8_NORM_TOL


@pytest.mark.parametrize("m", [1, 15, 17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(1, 64), (33, 128), (250, 192), (8200, 1088), (8205, 1152)])
@pytest.mark.parametrize("form", ["bf16-mxfp8", "bf16-mxfp4", "f32-mxfp8", "f32-mxfp4", "mx-mxfp8"])
def test_few_rows(gpu, form, m, n, k):
    """The one-pass kernel of few-row batches: both ends of each row-block
    class, one row and ragged columns, half windows (k % 128 == 64), fewer
    windows than waves and both workgroup widths (n from 8192 takes four
    weight row blocks).  fp32 output, so the bound is that of fp32 sums over
    k <= 1152 exact products (2^-24 sqrt(k) ~ 2e-6)."""
    dtype, fmt = form.split("-")
    if dtype == "mx" and k % 128:
        pytest.skip("MXFP8 rows take whole 128-k windows")
    g = torch.Generator().manual_seed(m * 31 + n + k)
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    x = torch.randn(m, k, generator=g) * torch.exp(0.5 * torch.randn(k, generator=g))
    x = x if dtype == "f32" else x.to(torch.bfloat16)
    q, s, wd = _quantized(fmt, w)
    if dtype == "mx":
        xq, xs = mxfp8.mxfp8_quantize(x.to(gpu))
        c = linear.mxfp8_linear_mx(xq, xs, q, s, out_dtype=torch.float32)
        xv = oracle.mx_dequant("mxfp8", xq.view(torch.uint8).cpu().numpy(), xs.cpu().numpy()).astype(np.float64)
    else:
        fn = linear.mxfp8_linear if fmt == "mxfp8" else linear.mxfp4_linear
        c = fn(x.to(gpu), q, s, out_dtype=torch.float32)
        xv = x.double().numpy()
    ref = xv @ wd.astype(np.float64).T
    assert _max_rel(ref, c.cpu().numpy()) <= 1e-5


@pytest.mark.parametrize("a_byte,w_byte", [(7, 237), (100, 247), (3, 3 + 240), (240, 9)])
def test_few_rows_extreme_scales(gpu, a_byte, w_byte):
    """MXFP8 x MXFP8 scale bytes whose products with E4M3 leave the normal
    bf16 range (2^-120 activations against 2^110 weights) multiply in fp32:
    fp32 sums of 512 exact products of one sign, at most 512 x 2^-24 = 3e-5."""
    g = torch.Generator().manual_seed(5)
    m, n, k = 3, 40, 512
    aq = torch.randint(0, 120, (m, k), generator=g, dtype=torch.uint8)
    wq = torch.randint(0, 120, (n, k), generator=g, dtype=torch.uint8)
    a_s = torch.full((m, k // 32), a_byte, dtype=torch.uint8)
    w_s = torch.full((n, k // 32), w_byte, dtype=torch.uint8)
    c = linear.mxfp8_linear_mx(aq.to(gpu).view(torch.float8_e4m3fn), a_s.to(gpu), wq.to(gpu), w_s.to(gpu),
                               out_dtype=torch.float32)

    def values(q, s):
        v = q.view(torch.float8_e4m3fn).double().reshape(q.shape[0], -1, 32)
        return (v * torch.exp2(s.double() - 127)[..., None]).reshape(q.shape).numpy()

    assert _max_rel(values(aq, a_s) @ values(wq, w_s).T, c.cpu().numpy()) <= 3e-5


@pytest.mark.parametrize("m,n,k", [(33, 130, 2176), (64, 8200, 4224), (65, 70, 4160), (257, 300, 1024), (300, 515, 2112),
                                   (777, 1030, 3200)])
@pytest.mark.parametrize("form", ["bf16-mxfp8", "bf16-mxfp4", "f32-mxfp8", "mx-mxfp8"])
def test_split_k(gpu, form, m, n, k):
    """Shapes of few tiles run K in slices (ragged rows and columns, odd N,
    K % 128 == 64 on the register-staged kernel, slices of unequal steps):
    fp32 output against float64 within the fp32 sums' 1e-5 (MXFP8 x MXFP8:
    the matrix cores' 64-product sums, 5e-5), bf16 output within one ulp; the
    unsplit call without a workspace agrees to fp32 summation order."""
    dtype, fmt = form.split("-")
    if dtype == "mx" and k % 128:
        pytest.skip("MXFP8 rows take K % 128 == 0")
    g = torch.Generator().manual_seed(m + n + k)
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    x = torch.randn(m, k, generator=g) * torch.exp(0.5 * torch.randn(k, generator=g))
    x = x if dtype == "f32" else x.to(torch.bfloat16)
    q, s, wd = _quantized(fmt, w)
    if dtype == "mx":
        xq, xs = mxfp8.mxfp8_quantize(x.to(gpu))
        xv = oracle.mx_dequant("mxfp8", xq.view(torch.uint8).cpu().numpy(), xs.cpu().numpy()).astype(np.float64)
        run = lambda out: linear.mxfp8_linear_mx(xq, xs, q, s, out_dtype=out)  # noqa: E731
    else:
        xv = x.double().numpy()
        fn = linear.mxfp8_linear if fmt == "mxfp8" else linear.mxfp4_linear
        run = lambda out: fn(x.to(gpu), q, s, out_dtype=out)  # noqa: E731
    ref = xv @ wd.astype(np.float64).T
    c = run(torch.float32)
    assert _max_rel(ref, c.cpu().numpy()) <= (5e-5 if dtype == "mx" else 1e-5)
    assert torch.equal(c, run(torch.float32))  # slices are summed in order
    if dtype == "bf16":
        check_bf16_output(ref, run(torch.bfloat16).float().cpu().numpy())
        from kquant_amd import _native as N
        plain = torch.empty(m, n, dtype=torch.float32, device=gpu)
        xg, qg = x.to(gpu), q.view(torch.uint8)
        N.call("kq_mx_linear", N.FMT_MXFP8_E4M3 if fmt == "mxfp8" else N.FMT_MXFP4_E2M1, N.ptr(xg), k, N.ptr(qg),
               N.ptr(s), m, n, k, N.DT_F32, N.ptr(plain), n, N.stream(gpu))
        assert _max_rel(ref, plain.cpu().numpy()) <= 1e-5


@pytest.mark.parametrize("m", [33, 48, 64])
def test_workspace_too_small_for_the_planes(gpu, m):
    """A workspace that does not hold the K slices' planes runs as none: the
    same kernel, bit for bit (bf16 and fp32 rows; MXFP8 rows given the scale
    planes alone against float64, at 5e-5 as everywhere for them)."""
    from kquant_amd import _native as N

    n, k = 2100, 2176
    g = torch.Generator().manual_seed(m)
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    x = torch.randn(m, k, generator=g).to(gpu)
    q, s, wd = _quantized("mxfp8", w)
    qb, lib, st = q.view(torch.uint8), N.library(), N.stream(gpu)
    xb = x.to(torch.bfloat16)
    assert lib.kq_mx_linear_workspace_size(m, n, k) > 256
    ws = torch.empty(4 * m * 3 * k * 2, dtype=torch.uint8, device=gpu)
    out = [torch.empty(m, n, device=gpu) for _ in range(5)]
    fmt = N.FMT_MXFP8_E4M3
    N.call("kq_mx_linear", fmt, N.ptr(xb), k, N.ptr(qb), N.ptr(s), m, n, k, N.DT_F32, N.ptr(out[0]), n, st)
    N.call("kq_mx_linear_ws", fmt, N.ptr(xb), k, N.ptr(qb), N.ptr(s), m, n, k, N.DT_F32, N.ptr(out[1]), n, N.ptr(ws),
           256, st)
    assert torch.equal(out[0], out[1])
    need = lib.kq_mx_linear_f32_workspace_size(m, k)
    for o, size in ((out[2], need), (out[3], (need + 255) // 256 * 256 + 256)):
        N.call("kq_mx_linear_f32", fmt, N.ptr(x), k, N.ptr(qb), N.ptr(s), m, n, k, N.ptr(o), n, N.ptr(ws), size, st)
    assert torch.equal(out[2], out[3])
    xq, xs = mxfp8.mxfp8_quantize(xb)
    planes = sum((r * (k // 32) + 255) // 256 * 256 for r in (m, n))
    N.call("kq_mx_linear_mx", fmt, N.ptr(xq.view(torch.uint8)), N.ptr(xs), k, fmt, N.ptr(qb), N.ptr(s), m, n, k,
           N.DT_F32, N.ptr(out[4]), n, N.ptr(ws), planes, st)
    xv = oracle.mx_dequant("mxfp8", xq.view(torch.uint8).cpu().numpy(), xs.cpu().numpy()).astype(np.float64)
    assert _max_rel(xv @ wd.astype(np.float64).T, out[4].cpu().numpy()) <= 5e-5


@pytest.mark.parametrize("form,m,n,k", [("bf16-mxfp8", 16, 65600, 576), ("bf16-mxfp4", 33, 65537, 320),
                                        ("bf16-mxfp8", 64, 49153, 512), ("f32-mxfp8", 33, 65540, 320),
                                        ("mx-mxfp8", 64, 12288, 2048), ("mx-mxfp8", 32, 40001, 1024)])
def test_few_rows_of_wide_weights(gpu, form, m, n, k):
    """Few rows of weights wide enough for the 256 x 256 tiles to win: fp32
    output within 1e-5 of float64 (MXFP8 rows on the matrix cores 5e-5), and
    the MXFP8 rows' workspace has the split's planes."""
    from kquant_amd import _native as N

    dtype, fmt = form.split("-")
    print(f"case wide {form} {m} {n} {k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    w = (torch.randn(n, k, generator=g, device=gpu) * 0.02).to(torch.bfloat16)
    x = torch.randn(m, k, generator=g, device=gpu).to(torch.float32 if dtype == "f32" else torch.bfloat16)
    quantize = mxfp8.mxfp8_quantize if fmt == "mxfp8" else kq_mxfp4.mxfp4_quantize
    q, s = quantize(w)
    dequant = mxfp8.mxfp8_dequantize if fmt == "mxfp8" else io_mxfp4.dequant
    if dtype == "mx":
        xq, xs = mxfp8.mxfp8_quantize(x)
        c = linear.mxfp8_linear_mx(xq, xs, q, s, out_dtype=torch.float32)
        x = mxfp8.mxfp8_dequantize(xq, xs, dtype=torch.float32)
        planes = sum((r * (k // 32) + 255) // 256 * 256 for r in (m, n))
        if n == 12288:
            assert N.library().kq_mx_linear_mx_workspace_size(m, n, k) > planes
    else:
        c = (linear.mxfp8_linear if fmt == "mxfp8" else linear.mxfp4_linear)(x, q, s, out_dtype=torch.float32)
    ref = x.double() @ dequant(q, s, dtype=torch.float32).double().T
    assert float((c.double() - ref).abs().max() / ref.abs().max()) <= (5e-5 if dtype == "mx" else 1e-5)


def _mx_values(q, s):
    v = q.view(torch.float8_e4m3fn).double().reshape(q.shape[0], -1, 32)
    return (v * torch.exp2(s.double() - 127)[..., None]).reshape(q.shape)


@pytest.mark.parametrize("m,n,k", [(3, 40, 512), (16, 16, 128), (31, 8200, 256), (64, 70, 384)])
@pytest.mark.parametrize("a_byte", [247, 254, 0, 120, -1])
def test_few_rows_scales_past_fp32(gpu, m, n, k, a_byte):
    """Operands that leave fp32's range by their own scale while the product
    does not (448 x 2^127 against 2^-127; -1: another scale for every block,
    its counterpart on the other side), in every row-block form.  Codes of one
    sign, products and the 32-k sums in fp32: k 2^-24 <= 3e-5 of float64."""
    g = torch.Generator().manual_seed(m + a_byte)
    aq = torch.randint(1, 127, (m, k), generator=g, dtype=torch.uint8)
    wq = torch.randint(1, 127, (n, k), generator=g, dtype=torch.uint8)
    base = torch.randint(0, 255, (k // 32,), generator=g) if a_byte < 0 else torch.full((k // 32,), a_byte)
    a_s = (base + torch.randint(-3, 4, (m, k // 32), generator=g)).clamp(0, 254).to(torch.uint8)
    w_s = (254 - base + torch.randint(-3, 4, (n, k // 32), generator=g)).clamp(0, 254).to(torch.uint8)
    c = linear.mxfp8_linear_mx(aq.to(gpu).view(torch.float8_e4m3fn), a_s.to(gpu), wq.to(gpu), w_s.to(gpu),
                               out_dtype=torch.float32)
    assert _max_rel((_mx_values(aq, a_s) @ _mx_values(wq, w_s).T).numpy(), c.cpu().numpy()) <= 3e-5


def test_few_rows_scale_and_code_nans(gpu):
    """A NaN code or scale byte 255 makes its own row (column) NaN and no
    other, beside a block whose scales need the fp32 products."""
    g = torch.Generator().manual_seed(9)
    m, n, k = 20, 50, 256
    aq = torch.randint(1, 127, (m, k), generator=g, dtype=torch.uint8)
    wq = torch.randint(1, 127, (n, k), generator=g, dtype=torch.uint8)
    a_s = torch.full((m, k // 32), 127, dtype=torch.uint8)
    w_s = torch.full((n, k // 32), 127, dtype=torch.uint8)
    a_s[:, 1], w_s[:, 1] = 250, 4
    aq[3, 70], aq[5, 200], w_s[7, 1], a_s[11, 6], wq[13, 33] = 127, 255, 255, 255, 127
    nan = torch.zeros(m, n, dtype=torch.bool)
    nan[[3, 5, 11]] = True
    nan[:, [7, 13]] = True
    c = linear.mxfp8_linear_mx(aq.to(gpu).view(torch.float8_e4m3fn), a_s.to(gpu), wq.to(gpu), w_s.to(gpu),
                               out_dtype=torch.float32).cpu()
    assert torch.equal(torch.isnan(c), nan)
    ref = (_mx_values(aq, a_s) @ _mx_values(wq, w_s).T)
    assert float(((c.double() - ref)[~nan] / ref[~nan]).abs().max()) <= 3e-5


@pytest.mark.parametrize("k", [128, 192, 320])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("fmt", ["mxfp8", "mxfp4"])
def test_few_rows_non_finite(gpu, fmt, dtype, k):
    """Inf and NaN stay in their rows: the last row (read again for the block's
    missing ones) and the columns a half window reads twice included."""
    g = torch.Generator().manual_seed(k)
    m, n = 21, 70
    w = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(gpu)
    x = torch.randn(m, k, generator=g).to(dtype)
    q, s, wd = _quantized(fmt, w)
    ref = x.double().numpy() @ wd.astype(np.float64).T
    x[2, 64], x[9, k - 1], x[-1, 3] = float("nan"), float("inf"), float("-inf")
    hit = np.zeros(m, dtype=bool)
    hit[[2, 9, m - 1]] = True
    fn = linear.mxfp8_linear if fmt == "mxfp8" else linear.mxfp4_linear
    c = fn(x.to(gpu), q, s, out_dtype=torch.float32).cpu().numpy()
    assert not np.isfinite(c[hit]).any() and np.isfinite(c[~hit]).all()
    assert _max_rel(ref[~hit], c[~hit]) <= 1e-5
