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


@pytest.mark.parametrize("n", [2**19, 2**19 + 1, 2**19 + 3 * 4096 + 1021])
@pytest.mark.parametrize("block", [4, 8, 64, 128, 256, 512, 1000, 1024, 1028, 2048, 4096, 8192])
@pytest.mark.parametrize("signed", [True, False])
def test_forms_of_many_elements_match_the_oracle(n, block, signed):
    """Both sides of the size from which the vector tiles are taken, which the tests above stay below."""
    test_forms_match_the_oracle(n, block, signed)


@pytest.mark.parametrize("block", [4, 64, 256, 512, 1024, 2048, 4096])
@pytest.mark.parametrize("signed", [True, False])
def test_special_blocks_among_many(block, signed):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    gen = torch.Generator().manual_seed(block)
    rows = torch.randn(2**19 // block + 7, block, generator=gen)
    at = torch.randperm(rows.shape[0], generator=gen)[: 9 * 12].view(9, 12)
    rows[at[0]] *= 1e-42
    rows[at[1]] *= 1e-30
    rows[at[2]] *= 1e25
    rows[at[3], 2] = float("inf")
    rows[at[4], 3] = float("nan")
    rows[at[5], 1], rows[at[5], 2], rows[at[5], 3] = float("inf"), float("nan"), -float("inf")
    rows[at[6]] = 0.0
    rows[at[7]] = -rows[at[7]].abs()
    rows[at[8], 3] = -1e30
    _check(rows.reshape(-1)[: rows.numel() - 1], signed, block)


@pytest.mark.parametrize("block,few", [(128, 640), (256, 1280), (1000, 5000), (1024, 5120), (64, 8192), (100, 8192)])
def test_workgroup_and_wavefront_blocks(block, few):
    """Around the block counts up to which a block of the general form takes a workgroup."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    for nb in (few, few + 1):
        gen = torch.Generator().manual_seed(nb)
        x = torch.randn(nb * block - 3, generator=gen)
        _check(x, True, block, 1)
        _check(x.abs(), False, block, 0)
