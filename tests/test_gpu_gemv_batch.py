"""The GEMV of a few tokens split along K: edges of its row groups, tokens, columns and splits."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import bc4, clib
from texelator_amd import _lib

from .helpers import bf16_bits, bf16_vector, f16_vector, lognormal_scales, max_rel_err_floor, random_blocks

pytestmark = pytest.mark.gpu


def pack(ext, m, k, seed, bias=None):
    blocks, scales = random_blocks(m, k, seed), lognormal_scales(m, seed + 1)
    return ext.pack_encoded(torch.from_numpy(blocks.reshape(-1)), torch.from_numpy(scales), bias), blocks, scales


def split_bytes(handle, tokens):
    out = ctypes.c_int64(0)
    _lib.check(_lib.load().tx_linear_workspace_bytes(handle, tokens, ctypes.byref(out)))
    return out.value


@pytest.mark.parametrize("tokens", [2, 4, 5, 13, 15])
@pytest.mark.parametrize("m,k", [(1, 10128), (16, 10240), (129, 10368), (1040, 8208), (2064, 27648)])
@pytest.mark.parametrize("mode", ["bf16", "bf16_bias", "f16_bias", "lut"])
def test_batch_matches_float64(ext, oracle_threads, m, k, tokens, mode):
    """Against the float64 product of the decoded weights: the output's rounding (2^-8 bf16, 2^-11 fp16 of
    the value) plus the fp32 sums' 1e-3."""
    f16 = mode.startswith("f16")
    vector = f16_vector if f16 else bf16_vector
    bias = vector((m,), 7, scale=0.5) if mode.endswith("bias") else None
    handle, blocks, scales = pack(ext, m, k, m + k, None if bias is None else bias.cuda())
    x = vector((tokens, k), tokens)
    lut = None
    if mode == "lut":
        base = bc4.palette()
        lut = (base * (1 + 0.01 * np.random.default_rng(5).standard_normal(base.shape))).astype(np.float32)
        ext.set_palette_table(handle, torch.from_numpy(lut).cuda())
    try:
        assert split_bytes(handle, tokens) > 0, "the shape must run the split kernel"
        y = ext.linear(handle, x.cuda()).double().cpu().numpy()
    finally:
        ext.free(handle)
    if f16:
        w = bc4.decode_f16_bits(blocks, scales).view(np.float16).astype(np.float64)
        want = x.double().numpy() @ w.T
    else:
        want = clib.gemm_f64(bf16_bits(x), clib.decode_bf16_bits(blocks, scales, lut))
    if bias is not None:
        want = want + bias.double().numpy()[None, :]
    assert max_rel_err_floor(want, y) <= (2 ** -11 if f16 else 2 ** -8) + 1e-3


@pytest.mark.parametrize("k", [10256, 10368])
def test_tokens_do_not_reach_each_other(ext, k):
    """A token of infinities (next to the others' padding columns where K is not a multiple of 128) leaves the
    others' outputs as they are."""
    handle, _, _ = pack(ext, 48, k, 3)
    try:
        assert split_bytes(handle, 6) > 0
        x = bf16_vector((6, k), 4).cuda()
        want = ext.linear(handle, x)
        x[3] = float("inf")
        got = ext.linear(handle, x)
        keep = [0, 1, 2, 4, 5]
        assert torch.equal(got[keep], want[keep])
    finally:
        ext.free(handle)


def linear_with(handle, x, y, workspace=None):
    """tx_linear with the given workspace address and size (none by default)."""
    address, size = workspace or (None, 0)
    status = _lib.load().tx_linear(handle, ctypes.c_void_p(x.data_ptr()), _lib.TX_DTYPE_BF16, x.numel(), x.shape[-1], 0,
                                   ctypes.c_void_p(y.data_ptr()), address, size, None)
    torch.cuda.synchronize()
    assert status == _lib.TX_OK


def test_without_a_workspace_the_call_runs_unsplit(ext):
    """tx_linear with a null, short or misaligned workspace still runs; the static-scratch entry point splits as linear
    does."""
    handle, _, _ = pack(ext, 96, 10240, 9)
    try:
        x = bf16_vector((5, 10240), 10).cuda()
        need = split_bytes(handle, 5)
        assert need > 0
        want = ext.linear(handle, x)
        y = torch.empty_like(want)
        ext.linear_noalloc_into(handle, x, y)
        assert torch.equal(y, want)
        plain = torch.empty_like(want)
        linear_with(handle, x, plain)
        assert torch.allclose(plain.float(), want.float(), rtol=2 ** -7, atol=1e-2)
        scratch = torch.full((need + 16,), 0x55, dtype=torch.uint8, device="cuda")
        for workspace in ((scratch.data_ptr(), need - 1), (scratch.data_ptr() + 8, need)):
            linear_with(handle, x, y, workspace)
            assert torch.equal(y, plain) and bool((scratch == 0x55).all())
    finally:
        ext.free(handle)


@pytest.mark.parametrize("m,k,tokens", [(96, 10240, 5), (1024, 8192, 15), (22016, 4224, 8), (11008, 5120, 13), (64, 4112, 7)])
def test_the_documented_workspace_gives_the_static_scratch_entry_points_bits(ext, m, k, tokens):
    """tx_linear with a workspace of tx_workspace_bytes, as a C caller allocates it, and tx_linear_noalloc."""
    handle, _, _ = pack(ext, m, k, 19)
    try:
        x = bf16_vector((tokens, k), 20).cuda()
        y, want = (torch.empty((tokens, m), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        scratch = torch.empty(max(16, ext.workspace_bytes(handle, tokens)), dtype=torch.uint8, device="cuda")
        assert split_bytes(handle, tokens) <= ext.workspace_bytes(handle, tokens)
        linear_with(handle, x, y, (scratch.data_ptr(), ext.workspace_bytes(handle, tokens)))
        ext.linear_noalloc_into(handle, x, want)
        assert torch.equal(y, want) and torch.equal(ext.linear(handle, x), want)
    finally:
        ext.free(handle)


# Both sides of each line of the split's rule: K with rows, and tokens x K x rows; and a count of splits set by
# how the workgroups share the CUs (22016 rows: four splits, not three).
@pytest.mark.parametrize("m,k,tokens,split", [
    (1008, 8192, 8, False), (1024, 8192, 8, True), (1024, 8064, 8, False),
    (64, 10112, 2, False), (64, 10128, 2, True),
    (5104, 7168, 2, False), (5120, 7168, 2, True), (5120, 7040, 2, False),
    (11008, 4224, 12, False), (11008, 4224, 13, True), (22016, 4224, 8, True), (60000, 4096, 15, False),
])
def test_sides_of_the_splits_lines(ext, m, k, tokens, split):
    """The call agrees with the unsplit one (no workspace): bitwise where the rule does not split, within the output's
    rounding and the sums' order elsewhere."""
    handle, _, _ = pack(ext, m, k, 17)
    try:
        need = split_bytes(handle, tokens)
        assert (need > 0) == split
        if m == 22016:
            assert need == 4 * tokens * m * 4
        x = bf16_vector((tokens, k), 18).cuda()
        got = ext.linear(handle, x)
        want = torch.empty_like(got)
        linear_with(handle, x, want)
        if split:
            error = (got.float() - want.float()).abs()
            assert bool((error <= 2 ** -7 * want.float().abs() + 1e-3 * want.float().square().mean().sqrt()).all())
        else:
            assert torch.equal(got, want)
    finally:
        ext.free(handle)


def test_unsplit_where_the_plan_says_so(ext):
    """Short K, one token and more than sixteen tokens keep the other kernels."""
    handle, _, _ = pack(ext, 64, 4096, 11)
    long, _, _ = pack(ext, 64, 10240, 12)
    try:
        assert split_bytes(handle, 8) == 0
        ext.set_prefill(long, 1 << 20, 1024)
        assert split_bytes(long, 16) > 0 and split_bytes(long, 17) == 0
        x = bf16_vector((17, 10240), 13).cuda()
        y16, y17 = ext.linear(long, x[:16]), ext.linear(long, x)
        assert torch.allclose(y16.float(), y17[:16].float(), rtol=2 ** -7, atol=1e-2)
    finally:
        ext.free(handle)
        ext.free(long)
