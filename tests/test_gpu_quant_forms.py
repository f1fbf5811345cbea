"""The forms of the blockwise quantisation kernels (vector tiles for power-of-two blocks of aligned buffers, the
general one for every other size and alignment) against the oracle, bit for bit: tile edges, tails, blocks over a
quarter round, a round, a wavefront and several, and blocks with infinities, NaNs, subnormals and scales outside the
reciprocal division's range."""
import pytest
import torch

from oracle import came8_oracle as orc

pytestmark = pytest.mark.gpu


def _check(x, signed, block, offset=0):
    from came_amd import blockwise_quantization as bq
    q_ref, a_ref = orc.quantize_blockwise(x, signed=signed, block_size=block)
    pad = torch.empty(x.numel() + offset, device="cuda")
    xd = pad[offset:].copy_(x)  # offset 1: not 16-byte aligned
    q, a = bq.quantize_blockwise(xd, signed=signed, block_size=block)
    known = ~x.isnan()  # a NaN has no code
    assert torch.equal(q.cpu()[known], q_ref[known])
    assert torch.equal(a.cpu(), a_ref)
    qd = torch.empty(x.numel() + offset, device="cuda", dtype=q.dtype)[offset:].copy_(q_ref)
    d = bq.dequantize_blockwise(qd, a_ref.cuda(), signed=signed, block_size=block)
    d_ref = orc.dequantize_blockwise(q_ref, a_ref, signed=signed, block_size=block)
    assert torch.equal(d.cpu().nan_to_num(7.0, 8.0, 9.0), d_ref.nan_to_num(7.0, 8.0, 9.0))  # code 0 of an inf block


@pytest.mark.parametrize("n", [3, 4095, 4096, 4097, 3 * 4096 + 1021])
@pytest.mark.parametrize("block", [4, 8, 128, 256, 512, 1000, 1024, 1028, 2048, 4096, 8192])
@pytest.mark.parametrize("signed", [True, False])
def test_forms_match_the_oracle(n, block, signed):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    gen = torch.Generator().manual_seed(n + 13 * block)
    x = torch.randn(n, generator=gen) * torch.exp(4 * torch.randn(n, generator=gen))
    for offset in (0, 1):
        _check(x if signed else x.abs(), signed, block, offset)


@pytest.mark.parametrize("block", [64, 100, 256, 1024, 4096])
@pytest.mark.parametrize("signed", [True, False])
def test_special_blocks(block, signed):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    gen = torch.Generator().manual_seed(block)
    rows = torch.randn(9, block, generator=gen)
    rows[0] *= 1e-42  # subnormal
    rows[1] *= 1e-30  # below the reciprocal division's range
    rows[2] *= 1e25   # above it
    rows[3, 5] = float("inf")
    rows[4, 7] = float("nan")
    rows[5, 1], rows[5, 2], rows[5, 3] = float("inf"), float("nan"), -float("inf")
    rows[6] = 0.0
    rows[7] = -rows[7].abs()  # unsigned: a negative maximum
    rows[8, 3] = -1e30
    _check(rows.reshape(-1)[: 9 * block - 1], signed, block)
