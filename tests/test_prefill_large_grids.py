"""Prefill grids of more than one 128-row item per CU: one-half blocks
(csrc/prefill.hip, use_one_half): every place a ragged end or the causal
diagonal can fall in a block's tiles, against the oracle, and their rounding
against that of two-half blocks."""

import ctypes
import math
import os

import numpy as np
import pytest
import torch

import flashattn_cuda
import oracle

pytestmark = pytest.mark.gpu

BOUND = 2.44e-4  # fp32 output; the fp16 output is its rounding


def _check_prefill(batch, heads, kv_heads, seq, d, causal, scale, spread=1.0, check=None):
    gen = torch.Generator().manual_seed(seq * 10 + d + causal)
    q = (torch.randn(batch, heads, seq, d, generator=gen) * spread).half()
    k = (torch.randn(batch, kv_heads, seq, d, generator=gen) * spread).half()
    v = torch.randn(batch, kv_heads, seq, d, generator=gen).half()
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    out32 = flashattn_cuda._prefill_gqa_fp32(qd, kd, vd, causal, scale)
    out16 = flashattn_cuda.prefill_gqa(qd, kd, vd, causal, scale)
    torch.cuda.synchronize()
    assert torch.equal(out16, out32.half())
    group = heads // kv_heads
    # Every K/V head's first query head, or the first, last and a few between.
    some = sorted({h // group * group for h in (check or range(heads))})
    ref = oracle.prefill_gqa(q[:, some].numpy(), k[:, [h // group for h in some]].numpy(),
                             v[:, [h // group for h in some]].numpy(), causal, scale)
    err = np.abs(out32[:, some].cpu().numpy() - ref).max()
    assert err <= BOUND, err


def _heads_for(seq, per_cu):
    """Query heads of one sequence that give more than per_cu items per CU
    (above two, and below 8192 keys, use_one_half takes every grid)."""
    cu = torch.cuda.get_device_properties(0).multi_processor_count
    tiles = -(-seq // 128)
    heads = int(per_cu * cu) // tiles + 1
    assert heads * tiles > per_cu * cu and seq < 8192
    return heads


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("seq", [1, 129, 255, 257, 288, 321, 384, 415, 511, 673])
def test_one_half_blocks_at_every_tail(seq, causal, d):
    heads = _heads_for(seq, 2)
    _check_prefill(1, heads, heads, seq, d, causal, d ** -0.5)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("kind", ["grouped", "negative scale", "wide scale", "wide inputs"])
def test_one_half_blocks_options(kind, d):
    """Grouped K/V heads; a negative scale; a scale that splits P on every
    row; inputs whose rows are peaky, so that blocks run again with split P."""
    heads = 2 * (_heads_for(600, 2) // 2 + 1)
    scale = {"negative scale": -1.0, "wide scale": 2.4}.get(kind, 1.0) * d ** -0.5
    _check_prefill(1, heads, heads // 2 if kind == "grouped" else heads, 600, d, True, scale,
                   1.5 if kind == "wide inputs" else 1.0)


def _unplanned(q, k, v, causal, scale):
    """fp32 output of the C entry without a workspace: whole items, and for
    these few of them two-half blocks."""
    lib = ctypes.CDLL(os.path.join(os.path.dirname(flashattn_cuda.__file__), "libflashattn_hip.so"))
    out = torch.empty(q.shape, dtype=torch.float32, device="cuda")
    b, h, s, d = q.shape
    ptr = [ctypes.c_void_p(t.data_ptr()) for t in (q, k, v, out)]
    rc = lib.fa_prefill_hd(*ptr, 1, b, h, k.shape[1], s, d, int(causal), ctypes.c_float(scale), None,
                           ctypes.c_size_t(0), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    return out


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("seq,causal,per_cu", [
    (300, False, 2), (545, True, 2), (1100, False, 2), (1100, True, 2), (1733, True, 2), (700, True, 1.5),
])
@pytest.mark.parametrize("spread", [1.0, 1.5])
def test_one_half_blocks_round_as_two_half_blocks(spread, seq, causal, per_cu, d):
    """A row's result does not depend on the kind of block its grid takes:
    P is rounded to fp16 against the same max (its own for the even and for the
    odd key tiles), and with wide inputs the same 128 rows run again with split
    P. What may differ is the order of fp32 sums of up to 1733 terms: a relative
    2-norm of a few 2^-24 sqrt(1733) ~ 2.5e-6. (Rounded against another max the
    results differ by 1.5e-5 to 2e-4.)"""
    heads = _heads_for(seq, per_cu)
    gen = torch.Generator(device="cuda").manual_seed(seq + d)
    q, k = ((torch.randn(1, heads, seq, d, generator=gen, device="cuda") * spread).half() for _ in "qk")
    v = torch.randn(1, heads, seq, d, generator=gen, device="cuda").half()
    one = flashattn_cuda._prefill_fp32(q, k, v, causal, d ** -0.5)[:, :3]
    two = _unplanned(*(t[:, :3].contiguous() for t in (q, k, v)), causal, d ** -0.5)
    diff = ((one - two).norm() / two.norm()).item()
    assert diff <= 1e-5, diff


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("kind", ["late rise in slack", "late rise", "dominant keys", "odd tiles far below",
                                  "even tiles far below", "odd tiles last"])
def test_one_half_blocks_moving_max(kind, causal, d):
    """Rows of 1100 keys (lazy max) whose scores rise late, by less or by more
    than the slack of 8 (log2 units); that a few keys dominate; whose odd or
    even key tiles lie further apart than one accumulator can be rescaled over
    (250 log2 units); whose highest scores are in the last odd tile."""
    seq, scale = 1100, d ** -0.5
    tile = 64 if d == 64 else 32
    heads = _heads_for(seq, 2)
    gen = torch.Generator().manual_seed(d + causal)
    q = torch.randn(1, heads, seq, d, generator=gen) * 0.25
    k = torch.randn(1, heads, seq, d, generator=gen) * 0.25
    v = torch.randn(1, heads, seq, d, generator=gen).half()
    # Dim 0 carries a score of x log2 units through q[..., 0] = 8.
    q[..., 0] = 8.0
    unit = math.log(2) / (8.0 * scale)
    key = torch.arange(seq)
    odd = key // tile % 2 == 1
    x = torch.zeros(seq)
    if kind == "late rise in slack":
        x = (key >= 700) * 6.0
    elif kind == "late rise":
        x = (key >= 700) * 20.0
    elif kind == "dominant keys":
        x = (key % 257 == 100) * 9.0
    elif kind == "odd tiles far below":
        x = odd * -250.0
    elif kind == "even tiles far below":
        x = ~odd * -250.0
    elif kind == "odd tiles last":
        x = odd * -30.0 + (key >= 1050) * 60.0
    k[..., 0] = x * unit
    q, k = q.half(), k.half()
    check = [0, heads // 2, heads - 1]
    out = flashattn_cuda._prefill_fp32(q.cuda(), k.cuda(), v.cuda(), causal, scale)[:, check].cpu()
    ref = oracle.prefill(q[:, check].numpy(), k[:, check].numpy(), v[:, check].numpy(), causal, scale)
    err = np.abs(out.numpy() - ref).max()
    assert err <= BOUND, err


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal,seq", [
    *[(False, s) for s in (512, 513, 544, 575, 577, 608, 639, 700, 768, 1024, 1100, 2090)],
    *[(True, s) for s in (1024, 1100, 2048, 2049, 2079, 2111, 2145, 2240)],
])
def test_one_half_blocks_at_every_tail_of_long_rows(seq, causal, d):
    heads = _heads_for(seq, 2)
    _check_prefill(1, heads, heads, seq, d, causal, d ** -0.5, check=[0, heads // 2, heads - 1])


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("kind", ["grouped", "negative scale", "wide scale", "wide inputs"])
def test_one_half_blocks_options_on_long_rows(kind, causal, d):
    seq = 2090 if causal else 1100
    heads = 2 * (_heads_for(seq, 2) // 2 + 1)
    scale = {"negative scale": -1.0, "wide scale": 2.4}.get(kind, 1.0) * d ** -0.5
    _check_prefill(1, heads, heads // 2 if kind == "grouped" else heads, seq, d, causal, scale,
                   1.5 if kind == "wide inputs" else 1.0, [0, 1, heads // 2, heads - 1])
