"""Edge shapes of the thread-per-matrix passes and of the kernels for small and narrow tensors, each step teacher-forced
against the oracle under the tolerances of test_gpu_parity.py, and steps over unaligned buffers against aligned ones."""
import pytest
import torch

import came_amd
from tests import parity as P
from tests.test_gpu_parity import _tight_step_check

pytestmark = pytest.mark.gpu

HP = dict(lr=1e-3, weight_decay=1e-2)
# matrices of 1 to 64 elements, around the counts staged at a time (256; 128 above 48 elements), and one item of
# several batches' worth of matrices
TINY = [(1, 1, 1), (255, 3, 3), (256, 3, 3), (257, 1, 1), (129, 7, 7), (128, 8, 8), (300, 2, 31), (513, 6, 8),
        (40, 30, 5, 5), (4099, 3, 1)]


def _run(cls, shapes, dtype, block, exact_norm, heavy, seed):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    params = P.make_params(shapes, dtype, seed=seed)
    gen = torch.Generator().manual_seed(seed + 1)
    grads = [[P.heavy_grad(gen, s, dtype) if heavy else (torch.randn(s, generator=gen) * 1e-3).to(dtype)
              for s in shapes] for _ in range(2)]
    P.run_teacher_forced(cls, params, grads, dict(HP, block_size=block), 2, exact_norm=exact_norm,
                         check=_tight_step_check(f"{dtype} block {block} exact {exact_norm}", block=block))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("block", [64, 256, 2048])
@pytest.mark.parametrize("exact_norm", [False, True])
def test_tiny_matrices(dtype, block, exact_norm):
    _run(came_amd.CAME8bitFull, TINY, dtype, block, exact_norm, heavy=block == 256, seed=71)


# one workgroup's steps: a row, a column, both sizes' edges (4096 and 32768 elements, 2560 rows and columns) and just
# past them, rows of fewer and more columns than threads, lengths with every tail of the norm's chains
SMALL = [(1,), (7,), (12,), (4095,), (4096,), (4099,), (32768,), (32769,), (1, 1), (1, 300), (300, 1), (5, 8), (96, 200),
         (16, 1280), (1280, 16), (2560, 12), (12, 2548), (13, 2548), (64, 64), (65, 63), (181, 181), (256, 128),
         (129, 255), (31, 1057), (1, 32767), (1, 4, 1000), (3, 40, 60)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("block", [64, 100, 256, 4096])
@pytest.mark.parametrize("exact_norm", [False, True])
def test_small_tensors(dtype, block, exact_norm):
    heavy = block == 64 and dtype != torch.float16
    _run(came_amd.CAME8bitFull, SMALL, dtype, block, exact_norm, heavy=heavy, seed=91)


@pytest.mark.parametrize("cls", ["CAME8bitFull", "CAMECUDA"])
def test_unaligned_buffers_match_aligned_ones(cls):
    """The vector forms and the ones that buffers off 16-byte boundaries take: the same step.  Sums may be ordered
    otherwise, hence the tolerances of the parity tests (codes one apart, 1e-5 of parameters and scales)."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    shapes = TINY + [(96, 200), (64, 16), (1000, 3), (33,), (2048,), (17, 1024)]
    out = []
    for offset in (0, 1):
        gen = torch.Generator().manual_seed(5)
        ps = []
        for s in shapes:
            n = torch.Size(s).numel()
            p, g = (torch.empty(n + offset, device="cuda")[offset:].view(s) for _ in range(2))
            p.copy_(torch.randn(s, generator=gen) * 0.02)
            g.copy_(torch.randn(s, generator=gen) * 1e-3)
            q = torch.nn.Parameter(p)
            q.grad = g
            ps.append(q)
        opt = getattr(came_amd, cls)(ps, **HP)
        for _ in range(2):
            opt.step()
        out.append((ps, [opt.state[p] for p in ps]))
    for i, s in enumerate(shapes):
        a, b = out[0][0][i].data.double(), out[1][0][i].data.double()
        assert ((a - b).abs() <= 1e-5 * (b.abs() + 0.02) + 1e-3 * HP["lr"]).all(), s
        for k, v in out[1][1][i].items():
            if not isinstance(v, torch.Tensor) or v.numel() == 0:
                continue
            w = out[0][1][i][k]
            if v.dtype.is_floating_point:
                assert torch.allclose(w, v, rtol=1e-4, atol=1e-5 * v.abs().max().item()), (s, k)
            else:
                assert (w.int() - v.int()).abs().max() <= 1, (s, k)


@pytest.mark.parametrize("cls", ["CAME8bit", "CAME8bitMemory"])
def test_block_sizes_far_past_the_tensors(cls):
    """Every block size from the largest state's length up is one block a state: the same bits for all of them, also where
    a length and a block size together pass 2^31."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    out = []
    for block in (32768, 2**31 - 1000, 2**31 - 1):
        gen = torch.Generator().manual_seed(3)
        ps = []
        for s in [(5, 7), (96, 200), (10,), (32768,), (1, 2048)]:
            ps.append(torch.nn.Parameter((torch.randn(s, generator=gen) * 0.02).cuda()))
            ps[-1].grad = (torch.randn(s, generator=gen) * 1e-3).cuda()
        opt = getattr(came_amd, cls)(ps, block_size=block, **HP)
        for _ in range(2):
            opt.step()
        out.append([p.detach() for p in ps] + [v for p in ps for v in opt.state[p].values() if isinstance(v, torch.Tensor)])
    for got in out[1:]:
        assert len(got) == len(out[0]) and all(torch.equal(a, b) for a, b in zip(got, out[0]))
