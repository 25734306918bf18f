"""Prefill grids of more than two 128-row items per CU: one-half blocks
(csrc/prefill.hip, use_one_half) and, at head_dim 64, 256-row blocks
(csrc/prefill_wide.hip, prefill_wide_pays): every place a ragged end or the
causal diagonal can fall in a block's tiles, against the oracle."""

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
    """Query heads of one sequence that give more than per_cu items per CU."""
    cu = torch.cuda.get_device_properties(0).multi_processor_count
    return per_cu * cu // -(-seq // 128) + 1


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


def _wide_case(seq, causal):
    """Heads that give a grid the 256-row blocks take, and heads to check."""
    cu = torch.cuda.get_device_properties(0).multi_processor_count
    tiles = -(-seq // 256)
    heads = 5 * cu // tiles + 1 if causal else 2 * cu // tiles
    return heads - heads % 2, [0, 1, heads // 3, heads // 2, heads - 3]


@pytest.mark.parametrize("causal,seq", [
    *[(False, s) for s in (512, 513, 544, 575, 577, 608, 639, 700, 768)],
    *[(True, s) for s in (2048, 2049, 2079, 2111, 2145, 2240)],
])
def test_wide_blocks_at_every_tail(seq, causal):
    heads, check = _wide_case(seq, causal)
    _check_prefill(1, heads, heads, seq, 64, causal, 0.125, check=check)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("kind", ["grouped", "negative scale", "wide scale", "wide inputs"])
def test_wide_blocks_options(kind, causal):
    seq = 2090 if causal else 720
    heads, check = _wide_case(seq, causal)
    scale = {"negative scale": -0.125, "wide scale": 0.3}.get(kind, 0.125)
    _check_prefill(1, heads, heads // 2 if kind == "grouped" else heads, seq, 64, causal, scale,
                   1.5 if kind == "wide inputs" else 1.0, check)
