"""Prefill of up to 255 tokens: the split-group tile's token and row blocks, finer K splits, the partials' reduce."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import bc4, clib

from .helpers import bf16_bits, bf16_vector, f16_vector, lognormal_scales, random_blocks

pytestmark = pytest.mark.gpu


def pack(ext, m, k, mode):
    blocks, scales = random_blocks(m, k, m + k), lognormal_scales(m, m + 1)
    bias = (f16_vector if mode.startswith("f16") else bf16_vector)((m,), 7, scale=0.5) if mode.endswith("bias") else None
    handle = ext.pack_encoded(torch.from_numpy(blocks.reshape(-1)), torch.from_numpy(scales), None if bias is None else bias.cuda())
    lut = None
    if mode == "lut":
        base = bc4.palette()
        lut = (base * (1 + 0.01 * np.random.default_rng(5).standard_normal(base.shape))).astype(np.float32)
        ext.set_palette_table(handle, torch.from_numpy(lut).cuda())
    return handle, blocks, scales, bias, lut


def splits(ext, handle, m, tokens):
    return ext.workspace_bytes(handle, tokens) // (4 * tokens * ((m + 15) // 16 * 16))


@pytest.mark.parametrize("m,k,tokens,ks", [
    (2048, 2048, 17, 4), (2033, 2176, 32, 4),                           # one token block
    (2033, 2048, 33, 4), (1025, 8192, 128, 4),                          # one block a wave, several tiles
    (4097, 2048, 64, 4), (3072, 2176, 65, 4), (8159, 2048, 127, 4),     # two blocks, the last one partial or empty
    (7168, 2048, 96, 4), (5121, 2304, 77, 4),                           # three
    (1024, 5120, 20, 10), (1000, 4848, 100, 9), (33, 2064, 200, 4),     # finer splits, partials and reduce
])
@pytest.mark.parametrize("mode", ["bf16", "bf16_bias", "f16_bias", "lut"])
def test_tiles_agree_and_match_float64(ext, oracle_threads, m, k, tokens, ks, mode):
    """The default call is every tile's bits, and the float64 product of the decoded weights within the output's
    rounding plus the fp32 sums' 1e-3."""
    f16 = mode.startswith("f16")
    handle, blocks, scales, bias, lut = pack(ext, m, k, mode)
    x = (f16_vector if f16 else bf16_vector)((tokens, k), tokens)
    try:
        assert splits(ext, handle, m, tokens) == ks, "the shape must split as listed"
        got = ext.linear(handle, x.cuda())
        for candidate in range(5, 10):
            assert torch.equal(ext.prefill(handle, candidate, x.cuda()), got), candidate
    finally:
        ext.free(handle)
    if f16:
        w = bc4.decode_f16_bits(blocks, scales).view(np.float16).astype(np.float64)
        want = x.double().numpy() @ w.T
    else:
        want = clib.gemm_f64(bf16_bits(x), clib.decode_bf16_bits(blocks, scales, lut))
    # A bias is added to the rounded product and the sum rounded again: each rounding is at most half an ulp (2^-8 of
    # a bf16 value, 2^-11 of an fp16 one) of its own value, so a bias that cancels the product leaves the product's.
    half_ulp = 2 ** -11 if f16 else 2 ** -8
    bound = 1e-3 * np.maximum(np.abs(want), np.sqrt(np.mean(want ** 2))) + half_ulp * np.abs(want)
    if bias is not None:
        want = want + bias.double().numpy()[None, :]
        bound = bound + half_ulp * np.abs(want) * 1.01
    assert (np.abs(want - got.double().cpu().numpy()) <= bound).all()


def test_k_that_was_whole_stays_whole(ext):
    """K below 2048 is not split, at any token count: the SwiGLU epilogue takes such calls."""
    handle = pack(ext, 2048, 1920, "bf16")[0]
    try:
        assert [splits(ext, handle, 2048, t) for t in (2, 32, 33, 128, 200)] == [0] * 5
    finally:
        ext.free(handle)


@pytest.mark.parametrize("m,k,tokens,ks", [(3000, 4848, 128, 9), (3000, 4848, 129, 4), (1536, 8960, 200, 8),
                                           (2560, 2048, 200, 4), (2048, 11008, 127, 16), (2048, 11008, 128, 10),
                                           (4096, 4848, 127, 8), (4096, 4848, 128, 4),
                                           (1024, 4096, 32, 4), (960, 4096, 33, 8), (256, 4992, 17, 4), (1024, 4112, 32, 8)])
def test_finer_splits_only_where_they_pay(ext, m, k, tokens, ks):
    """Past 128 tokens where they at least double the splits; below 16 MiB of partials; up to 32 tokens not where the
    split-group tile runs."""
    handle = pack(ext, m, k, "bf16")[0]
    try:
        assert splits(ext, handle, m, tokens) == ks
    finally:
        ext.free(handle)


@pytest.mark.parametrize("tokens", [256, 257, 384, 385, 513, 640, 767, 768])
@pytest.mark.parametrize("m,mode", [(3072, "bf16"), (3000, "f16_bias")])
def test_sides_of_the_large_tiles_padding_rule(ext, oracle_threads, m, mode, tokens):
    """Where the 256- and 512-token tiles would be mostly padding at their end the 128-token tile takes the call, with
    its own K splits: the default is every tile's bits, and rows at both ends match float64 (bound as above)."""
    handle, blocks, scales, bias, _ = pack(ext, m, 4096, mode)
    x = (f16_vector if mode.startswith("f16") else bf16_vector)((tokens, 4096), tokens)
    try:
        got = ext.linear(handle, x.cuda())
        for candidate in range(5, 10):
            assert torch.equal(ext.prefill(handle, candidate, x.cuda()), got), candidate
    finally:
        ext.free(handle)
    rows = np.r_[0:33, m - 33:m]
    blocks, scales = blocks.reshape(m, -1)[rows], scales[rows]
    if mode == "f16_bias":
        want = x.double().numpy() @ bc4.decode_f16_bits(blocks, scales).view(np.float16).astype(np.float64).T
    else:
        want = clib.gemm_f64(bf16_bits(x), clib.decode_bf16_bits(blocks, scales))
    half_ulp = 2 ** -11 if mode == "f16_bias" else 2 ** -8
    bound = 1e-3 * np.maximum(np.abs(want), np.sqrt(np.mean(want ** 2))) + half_ulp * np.abs(want)
    if bias is not None:
        want = want + bias.double().numpy()[None, rows]
        bound = bound + half_ulp * np.abs(want) * 1.01
    assert (np.abs(want - got[:, rows].double().cpu().numpy()) <= bound).all()
