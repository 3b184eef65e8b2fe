"""The encoder kernel gives, byte for byte, the torch operations' blocks and scales on the same GPU."""
from __future__ import annotations

import pytest
import torch

from texelator_amd import _hip, encoder, hardware

pytestmark = pytest.mark.gpu


def torch_encode(weight, hdiag, lut):
    rows = weight.float()
    scales = rows.abs().amax(1).clamp_min(1e-12)
    e0, e1, idx = encoder.endpoint_opt(rows, hdiag, scales, lut)
    return encoder.pack_blocks_tensor(e0, e1, idx).reshape(rows.shape[0], -1), scales


def matrix(m, k, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randn(m, k, device="cuda", generator=g) * 0.02 * torch.exp(0.3 * torch.randn(1, k, device="cuda", generator=g))
    return w.to(dtype), torch.exp(torch.randn(k, device="cuda", generator=g))


@pytest.mark.parametrize("m,k,dtype", [
    (1, 16, torch.float32), (3, 48, torch.bfloat16), (5, 1040, torch.float16),   # one block; idle lanes; two waves
    (2, 8192, torch.bfloat16), (2, 8208, torch.float32), (3, 27648, torch.bfloat16),  # one pass, two, four
    (700, 4096, torch.float32), (300, 5120, torch.bfloat16),
])
def test_encoder_kernel_is_bitwise_the_torch_operations(ext, m, k, dtype):
    weight, hdiag = matrix(m, k, dtype, seed=m + k)
    lut = hardware.device_palette("cuda").reshape(255, 255, 8)
    want_blocks, want_scales = torch_encode(weight, hdiag, lut)
    blocks, scales = encoder.encode_matrix_tensor(weight, hdiag, lut)
    assert torch.equal(scales, want_scales)
    assert torch.equal(blocks, want_blocks)


@pytest.mark.parametrize("palette", ["defined", "random"])
def test_encoder_kernel_on_edge_rows(ext, palette):
    """Zeros, constants, a spike, exact palette values, huge and tiny rows, zero and huge moments, NaN and
    infinite weights; and a table of arbitrary values (ties and unordered palettes)."""
    lut = hardware.device_palette("cuda").reshape(255, 255, 8)
    if palette == "random":
        g = torch.Generator(device="cuda").manual_seed(1)
        lut = (torch.randint(-8, 9, lut.shape, device="cuda", generator=g) / 8).float()
    weight, hdiag = matrix(16, 256, torch.float32, seed=9)
    weight[0] = 0
    weight[1] = 0.25
    weight[2] = 0
    weight[2, 7] = 3.0
    weight[3] = torch.arange(256, device="cuda") % 16 / 15 - 0.5
    weight[4] *= 1e30
    weight[5] *= 1e-30
    weight[6, 5] = float("nan")
    weight[7, 9] = float("inf")
    weight[8] = weight[8].abs()
    hdiag[:32] = 0
    hdiag[32:48] = 1e30
    hdiag[64] = float("nan")
    hdiag[80] = float("inf")
    want_blocks, want_scales = torch_encode(weight, hdiag, lut)
    blocks, scales = encoder.encode_matrix_tensor(weight, hdiag, lut)
    assert torch.equal(scales.view(torch.int32)[want_scales == want_scales], want_scales.view(torch.int32)[want_scales == want_scales])
    assert torch.equal(scales.isnan(), want_scales.isnan())
    assert torch.equal(blocks, want_blocks)


@pytest.mark.parametrize("signs", ["some", "all"])
def test_encoder_kernel_on_nan_blocks_under_negative_moments(ext, signs):
    """Negative importances (nothing forbids them) next to NaN and infinite weights: the torch operations' bytes."""
    lut = hardware.device_palette("cuda").reshape(255, 255, 8)
    weight, hdiag = matrix(12, 256, torch.float32, seed=6)
    weight[3, 5] = float("nan")
    weight[4, 9] = float("inf")
    weight[5, 200] = float("-inf")
    weight[6] = float("nan")
    hdiag[:: 3 if signs == "some" else 1] *= -1
    want_blocks, _ = torch_encode(weight, hdiag, lut)
    assert torch.equal(encoder.encode_matrix_tensor(weight, hdiag, lut)[0], want_blocks)


def test_encoder_takes_strided_offset_and_host_rows(ext):
    """What the torch operations accept: a transposed view, rows at an odd offset, float64, a CPU matrix in
    chunks; and encode_rows' chunks are the same bytes."""
    lut = hardware.device_palette("cuda").reshape(255, 255, 8)
    weight, hdiag = matrix(64, 528, torch.float32, seed=4)
    views = [weight.t().contiguous().t(), torch.nn.functional.pad(weight, (1, 0))[:, 1:], weight.double(),
             torch.nn.functional.pad(weight.bfloat16().reshape(-1), (1, 0))[1:].view(64, 528)]
    for view in views:
        want_blocks, want_scales = torch_encode(view, hdiag, lut)
        blocks, scales = encoder.encode_matrix_tensor(view, hdiag, lut, rows_per_chunk=24)
        assert torch.equal(blocks, want_blocks) and torch.equal(scales, want_scales)
    want_blocks, want_scales = torch_encode(weight, hdiag, lut)
    blocks, scales = encoder.encode_matrix_tensor(weight.cpu(), hdiag.cpu(), lut, rows_per_chunk=24)
    assert torch.equal(blocks, want_blocks) and torch.equal(scales, want_scales)
    blocks, scales = encoder.encode_matrix(weight, hdiag, lut, rows_per_chunk=24)
    assert (blocks == want_blocks.cpu().numpy()).all() and (scales == want_scales.cpu().numpy()).all()
    with pytest.raises(_hip.TexelatorError):
        _hip.encode_bc4(weight, hdiag[:-1].contiguous(), lut)


def test_tables_of_another_shape_are_refused(ext):
    """A palette table must be [255, 255, 8]: the torch operations cannot index a flat one, with a GPU table either."""
    lut = hardware.device_palette("cuda").reshape(255, 255, 8)
    weight, hdiag = matrix(4, 64, torch.float32, seed=1)
    with pytest.raises(IndexError):
        encoder.encode_matrix_tensor(weight, hdiag, lut.reshape(-1))
    with pytest.raises(IndexError):
        encoder.encode_matrix(weight, hdiag, lut.reshape(-1))


@pytest.mark.parametrize("form", ["transposed", "float64", "offset"])
def test_matrices_that_must_be_copied_are_copied_in_chunks(ext, form):
    """A matrix the kernel cannot read where it lies is staged rows_per_chunk rows at a time: the scratch stays a
    fraction of the matrix, and the bytes are those of the matrix in place."""
    lut = hardware.device_palette("cuda").reshape(255, 255, 8)
    weight, hdiag = matrix(4096, 1024, torch.float32, seed=2)
    want_blocks, want_scales = encoder.encode_matrix_tensor(weight, hdiag, lut)
    view = {"transposed": lambda: weight.t().contiguous().t(), "float64": weight.double,
            "offset": lambda: torch.nn.functional.pad(weight.reshape(-1), (1, 0))[1:].view(4096, 1024)}[form]()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    blocks, scales = encoder.encode_matrix_tensor(view, hdiag, lut, rows_per_chunk=256)
    scratch = torch.cuda.max_memory_allocated() - before - blocks.numel() - 4 * scales.numel()
    assert scratch < weight.numel() * 4 // 4
    assert torch.equal(blocks, want_blocks) and torch.equal(scales, want_scales)
