"""GPU parity of the SQG trellis quantizer (kq_sqg_quantize_tiles) with the
C oracle (oracle/sqg_viterbi.c, the reference kernel's search restated in
exact fp16): states and values bit-exact, for K2/K3/K4, full and short
tail-biting contexts, tie-heavy tiles (zeros, constants, tiles made of label
values) and more tiles than workgroups; and the same search against the MCG
and MUL1 procedural codebooks."""

from __future__ import annotations

import types

import numpy as np
import pytest
import torch

import oracle
from kquant_amd import _native as N
from kquant_amd import sqg_quantizer
from kquant_amd.sqg_e4m3 import sqg_xor_cheb_t12_bytes

pytestmark = pytest.mark.gpu


def _tiles(bits: int, seed: int) -> np.ndarray:
    rng = np.random.default_rng(seed)
    lut = oracle.sqg_xor_cheb_t12_bytes(bits)
    labels = oracle.e4m3_values(lut)
    return np.stack([
        rng.standard_normal(256),
        rng.standard_normal(256) * 0.3,
        np.zeros(256),                                 # every path ties
        np.full(256, 0.5),
        labels[rng.integers(0, 65536, 256)],           # exact label values
        rng.standard_normal(256) * 3.0,
    ]).astype(np.float32)


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("ctx", [128, 16])
def test_matches_oracle_bit_exact(gpu, bits, ctx):
    x = _tiles(bits, 10 * bits + ctx)
    lut_np = oracle.sqg_xor_cheb_t12_bytes(bits)
    want_vals, want_states = oracle.sqg_quantize_tiles(x, lut_np, bits, ctx)
    lut = sqg_xor_cheb_t12_bytes(bits, device=gpu)
    assert np.array_equal(lut.cpu().numpy(), lut_np)
    vals, states = sqg_quantizer.quantize_tiles_sqg(torch.from_numpy(x).to(gpu), lut, bits, ctx)
    mism = np.flatnonzero((states.cpu().numpy() != want_states).any(axis=1))
    print(f"K{bits} ctx {ctx}: mismatching tiles {mism.tolist()}", flush=True)
    assert mism.size == 0
    assert np.array_equal(vals.cpu().numpy(), want_vals)


def test_more_tiles_than_workgroups_and_install_hook(gpu, monkeypatch):
    bits = 3
    x = np.concatenate([_tiles(bits, s) for s in range(2)])  # 12 tiles
    lut_np = oracle.sqg_xor_cheb_t12_bytes(bits)
    want_vals, want_states = oracle.sqg_quantize_tiles(x, lut_np, bits, 32)
    monkeypatch.setattr(sqg_quantizer, "_workgroups", lambda device: 5)
    module = types.SimpleNamespace(quantize_tiles=lambda tiles, args: ("original", args))
    sqg_quantizer.install_sqg_quantizer(module)
    sqg_quantizer.install_sqg_quantizer(module)  # idempotent
    assert module.quantize_tiles(None, {})[0] == "original"
    args = {"devices": [gpu], "K": bits, "tailbite_context": 32,
            "sqg_e4m3_luts_by_bits": {3: torch.from_numpy(lut_np)}}
    vals, states = module.quantize_tiles(torch.from_numpy(x).to(gpu), args)
    assert np.array_equal(states.cpu().numpy(), want_states)
    assert np.array_equal(vals.cpu().numpy(), want_vals)
    with pytest.raises(ValueError, match="missing rate-specific SQG K3 LUT"):
        module.quantize_tiles(torch.from_numpy(x).to(gpu), {**args, "sqg_e4m3_luts_by_bits": {2: None}})


@pytest.mark.parametrize("codebook", [1, 2])
@pytest.mark.parametrize("bits,ctx", [(2, 128), (3, 16), (4, 128), (4, 16)])
def test_procedural_codebooks_match_oracle_bit_exact(gpu, codebook, bits, ctx):
    """MCG (1) and MUL1 (2) labels computed per state in the kernel against
    the oracle's tables (pinned by their closed forms on the CPU)."""
    rng = np.random.default_rng(100 * codebook + 10 * bits + ctx)
    labels = oracle.procedural_labels(codebook).astype(np.float32)
    x = np.stack([
        rng.standard_normal(256),
        rng.standard_normal(256) * 0.3,
        np.zeros(256),
        labels[rng.integers(0, 65536, 256)],
        rng.standard_normal(256) * 2.0,
    ]).astype(np.float32)
    want_vals, want_states = oracle.sqg_quantize_tiles_procedural(x, bits, codebook, ctx)
    vals, states = sqg_quantizer.quantize_tiles_procedural(torch.from_numpy(x).to(gpu), bits, codebook, ctx)
    mism = np.flatnonzero((states.cpu().numpy() != want_states).any(axis=1))
    print(f"codebook {codebook} K{bits} ctx {ctx}: mismatching tiles {mism.tolist()}", flush=True)
    assert mism.size == 0
    assert np.array_equal(vals.cpu().numpy(), want_vals)


def test_install_hook_routes_none_to_mcg(gpu):
    """A None entry of sqg_e4m3_luts_by_bits selects the MCG control
    (kquant/sqg_quantizer.py:99-119, tests/test_sqg_quantizer.py:11-48)."""
    x = np.random.default_rng(7).standard_normal((3, 256)).astype(np.float32)
    want_vals, want_states = oracle.sqg_quantize_tiles_procedural(x, 2, 1, 128)
    module = types.SimpleNamespace(quantize_tiles=lambda tiles, args: "upstream")
    sqg_quantizer.install_sqg_quantizer(module)
    vals, states = module.quantize_tiles(torch.from_numpy(x).to(gpu), {
        "K": 2, "devices": [gpu], "sqg_e4m3_luts_by_bits": {2: None, 3: None, 4: None}})
    assert np.array_equal(states.cpu().numpy(), want_states)
    assert np.array_equal(vals.cpu().numpy(), want_vals)
    with pytest.raises(ValueError, match="1 \\(MCG\\) or 2 \\(MUL1\\)"):
        sqg_quantizer.quantize_tiles_procedural(torch.from_numpy(x).to(gpu), 2, 3)


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("ctx", [1, 127])
def test_two_tiles_per_cu(gpu, bits, ctx):
    """More tiles than CUs take 512-thread workgroups, two per CU (other node
    ownership and decision packing), at the shortest context and an odd one:
    every copy of the same few tiles gives the oracle's states and values, and
    so does the one-tile-per-CU form."""
    x = _tiles(bits, 5 * bits + ctx)
    lut_np = oracle.sqg_xor_cheb_t12_bytes(bits)
    want_vals, want_states = oracle.sqg_quantize_tiles(x, lut_np, bits, ctx)
    lut = sqg_xor_cheb_t12_bytes(bits, device=gpu)
    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    for copies in (1, -(-(cus + 1) // x.shape[0]), -(-(2 * cus + 1) // x.shape[0])):
        vals, states = sqg_quantizer.quantize_tiles_sqg(torch.from_numpy(x).to(gpu).repeat(copies, 1), lut, bits, ctx)
        assert np.array_equal(states.cpu().numpy(), np.tile(want_states, (copies, 1)))
        assert np.array_equal(vals.cpu().numpy(), np.tile(want_vals, (copies, 1)))


def test_workspace_is_the_calls_own(gpu):
    """A call of few tiles holds the decisions of its own workgroups only (six
    of 1 MiB at K2) and none of them after it."""
    x = torch.from_numpy(_tiles(2, 3)).to(gpu)
    lut = sqg_xor_cheb_t12_bytes(2, device=gpu)
    before = torch.cuda.memory_allocated(gpu)
    torch.cuda.reset_peak_memory_stats(gpu)
    out = sqg_quantizer.quantize_tiles_sqg(x, lut, 2, 16)
    assert torch.cuda.max_memory_allocated(gpu) - before <= 8 << 20
    assert torch.cuda.memory_allocated(gpu) - before <= 4096 + sum(o.numel() * o.element_size() for o in out)


@pytest.mark.parametrize("bits", [2, 3, 4])
def test_table_and_workspace_at_odd_addresses(gpu, bits):
    """The C entry takes the table and the decisions at any address."""
    x = _tiles(bits, 7)
    lut_np = oracle.sqg_xor_cheb_t12_bytes(bits)
    want_vals, want_states = oracle.sqg_quantize_tiles(x, lut_np, bits, 16)
    t = torch.from_numpy(x).to(gpu)
    lut = torch.empty(65537, dtype=torch.uint8, device=gpu)[1:]
    lut.copy_(torch.from_numpy(lut_np))
    need = int(N.library().kq_sqg_quantize_workspace_size(bits, len(x)))
    ws = torch.empty(need + 1, dtype=torch.uint8, device=gpu)[1:]
    assert lut.data_ptr() % 2 and ws.data_ptr() % 2
    out, states = torch.empty_like(t), torch.empty(t.shape, dtype=torch.int16, device=gpu)
    N.call("kq_sqg_quantize_tiles", N.ptr(t), len(x), N.ptr(lut), bits, 16, N.ptr(out), N.ptr(states), N.ptr(ws), need,
           len(x), N.stream(gpu))
    assert np.array_equal(states.cpu().numpy(), want_states)
    assert np.array_equal(out.cpu().numpy(), want_vals)
