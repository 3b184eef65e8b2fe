"""The prompt-attention kernel at the edges of its tiles and under each split of its waves."""
from __future__ import annotations

import math

import pytest
import torch

from texelator_amd import layers

pytestmark = pytest.mark.gpu


def reference(q, k, v, heads, scale):
    tokens, group = q.shape[0], heads // k.shape[0]
    qf = q.double().view(tokens, heads, 128)
    mask = torch.triu(torch.ones(tokens, tokens, dtype=torch.bool, device="cuda"), 1)
    out = torch.empty(tokens, heads, 128, dtype=torch.float64, device="cuda")
    for head in range(heads):
        scores = (qf[:, head] @ k[head // group, :tokens].double().t()) * scale
        out[:, head] = torch.softmax(scores.masked_fill(mask, float("-inf")), dim=1) @ v[head // group, :tokens].double()
    return out.view(tokens, -1)


def inputs(tokens, heads, kv_heads, seed, context=None, spread=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    context = context or tokens
    k = torch.full((kv_heads, context, 128), float("nan"), device="cuda", dtype=torch.bfloat16)  # stale rows
    v = k.clone()
    k[:, :tokens] = torch.randn(kv_heads, tokens, 128, device="cuda", generator=g).bfloat16()
    v[:, :tokens] = torch.randn(kv_heads, tokens, 128, device="cuda", generator=g).bfloat16()
    q = (torch.randn(tokens, heads * 128, device="cuda", generator=g) * spread).bfloat16()
    return q, k, v


def check(got, want):
    # probabilities and the output rounded to bf16 (2^-9 each at most): 5e-3 relative is over twice their sum
    assert torch.isfinite(got.float()).all()
    assert float((got.double() - want).norm() / want.norm()) < 5e-3


# heads x tokens that run each split on 256 CUs: (4, 1) short and long, (4, 2), (1, 4), (2, 4)
@pytest.mark.parametrize("tokens,heads,kv_heads", [
    (1, 8, 8), (31, 8, 1), (32, 5, 5), (33, 16, 2), (64, 40, 8),
    (65, 8, 2), (96, 8, 2), (97, 16, 2), (129, 7, 7), (513, 8, 1),
    (300, 40, 8), (323, 28, 4), (448, 32, 8),
    (641, 48, 8), (704, 40, 8),
    (1289, 56, 8), (1409, 56, 7),
])
def test_tile_edges_and_splits(ext, tokens, heads, kv_heads):
    q, k, v = inputs(tokens, heads, kv_heads, tokens, context=tokens + 70)
    scale = 1 / math.sqrt(128)
    check(layers.prefill_attention(q, k, v, heads, kv_heads, scale), reference(q, k, v, heads, scale))


@pytest.mark.parametrize("scale", [1.0, -0.7, 0.0])
@pytest.mark.parametrize("tokens,heads", [(200, 8), (40, 8), (300, 40)])
def test_scores_that_grow_along_the_keys(ext, tokens, heads, scale):
    """Running maxima that rise by far more than the kernel's slack, block after block, and large, negative and
    zero scales."""
    q, k, v = inputs(tokens, heads, heads, 3, spread=0.5)
    k = (k.float() * torch.linspace(0.05, 4, tokens, device="cuda")[None, :, None]).bfloat16()
    check(layers.prefill_attention(q, k, v, heads, heads, scale), reference(q, k, v, heads, scale))


@pytest.mark.parametrize("tokens,heads,kv_heads", [(64, 8, 8), (512, 8, 1), (323, 28, 4), (704, 40, 8), (1409, 56, 7)])
def test_a_token_does_not_reach_the_others(ext, tokens, heads, kv_heads):
    """A query of far larger scores (its running maxima rise in other blocks) leaves the bits of every other query's
    output, the earlier ones of its wave among them: under each split of the waves."""
    q, k, v = inputs(tokens, heads, kv_heads, 11)
    scale = 1 / math.sqrt(128)
    want = layers.prefill_attention(q, k, v, heads, kv_heads, scale)
    loud = 32 * (tokens // 32) - 1  # the last of the last whole group of 32 queries
    q[loud] *= 30
    got = layers.prefill_attention(q, k, v, heads, kv_heads, scale)
    rows = [t for t in range(tokens) if t != loud]
    assert torch.equal(got[rows], want[rows]) and not torch.equal(got[loud], want[loud])


@pytest.mark.parametrize("tokens,heads", [(77, 4), (300, 40)])
def test_caches_and_outputs_off_alignment(ext, tokens, heads):
    """Caches 2 bytes off a 16-byte boundary and output rows at odd strides give the aligned call's bits."""
    q, k, v = inputs(tokens, heads, heads, 5)
    scale = 1 / math.sqrt(128)
    want = layers.prefill_attention(q, k, v, heads, heads, scale)
    shifted = [torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view_as(t) for t in (k, v)]
    assert shifted[0].data_ptr() % 16 != 0
    assert torch.equal(layers.prefill_attention(q, *shifted, heads, heads, scale), want)
    wide = torch.zeros(tokens, heads * 128 + 1, device="cuda", dtype=torch.bfloat16)
    layers.prefill_attention(q, k, v, heads, heads, scale, out=wide[:, 1:])
    assert torch.equal(wide[:, 1:], want) and not wide[:, 0].any()
