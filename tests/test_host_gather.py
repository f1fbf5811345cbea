"""The native descriptor gathering (csrc/came8_host.cpp): the same bytes as the Python's descriptors in the plain case, and
None with nothing changed in every other."""
import ctypes

import pytest
import torch

import came_amd
from came_amd import _lib


def _gather(opt, params):
    descs = (_lib.Came8Tensor * max(len(params), 1))()
    used = _lib.host().gather(params, opt.state, ctypes.addressof(descs), len(params), opt._STATE_KIND,
                              opt._group_block_size(opt.param_groups[0]))
    return used, bytes(descs)


def test_cpu_parameters_are_left_to_the_python():
    p = torch.nn.Parameter(torch.zeros(4, 4))
    p.grad = torch.zeros(4, 4)
    opt = came_amd.CAME8bit([p], lr=1e-3)
    assert _gather(opt, [p])[0] is None
    opt._init_state(opt.state[p], p.grad, 256)
    assert _gather(opt, [p])[0] is None and opt.state[p]["step"] == 0
    p.grad = None
    assert _gather(opt, [p])[0] == []


@pytest.mark.parametrize("block", [0, -1])
def test_block_sizes_without_blocks_are_left_to_the_python(block):
    """Before any tensor is looked at, so also for a group without gradients."""
    p = torch.nn.Parameter(torch.zeros(4, 4))
    opt = came_amd.CAME8bit([p], lr=1e-3)
    opt.param_groups[0]["block_size"] = block
    assert _gather(opt, [p])[0] is None


@pytest.mark.gpu
@pytest.mark.parametrize("block", [0, -1])
def test_block_sizes_without_blocks_raise(block):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    p = torch.nn.Parameter(torch.zeros(4, 6, device="cuda"))
    p.grad = torch.ones_like(p)
    opt = came_amd.CAME8bit([p], lr=1e-3)
    opt.step()  # with a state, which the native gathering would otherwise take
    before = p.detach().clone()
    opt.param_groups[0]["block_size"] = block
    with pytest.raises(ValueError, match="block_size must be > 0"):
        opt.step()
    assert torch.equal(p.detach(), before) and opt.state[p]["step"] == 1


@pytest.mark.gpu
@pytest.mark.parametrize("cls", ["CAME8bit", "CAME8bitFull", "CAME8bitMemory", "CAMECUDA"])
def test_same_descriptors_as_the_python(cls):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    params = [torch.nn.Parameter(torch.zeros(s, device="cuda", dtype=d)) for s, d in
              [((5, 7), torch.float32), ((300,), torch.bfloat16), ((3, 4, 5, 6), torch.float16), ((), torch.float32),
               ((1, 1), torch.bfloat16), ((2, 3, 400), torch.float32)]]
    for p in params:
        p.grad = torch.ones_like(p)
    opt = getattr(came_amd, cls)(params, lr=1e-3)
    opt.step()
    items = [(p, opt.state[p], p.grad) for p in params]
    want = bytes(opt._descriptors(items)[0])
    used, got = _gather(opt, params)
    assert got == want and len(used) == len(params) and all(a is b for a, b in zip(used, params))
    assert all(opt.state[p]["step"] == 2 for p in params)
    params[1].grad = None  # parameters without a gradient are left out
    used, got = _gather(opt, params)
    assert all(a is b for a, b in zip(used, params[:1] + params[2:])) and opt.state[params[1]]["step"] == 2


@pytest.mark.gpu
def test_other_cases_change_nothing():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")

    def fresh():
        ps = [torch.nn.Parameter(torch.zeros(s, device="cuda")) for s in ((4, 6), (9,))]
        for p in ps:
            p.grad = torch.ones_like(p)
        opt = came_amd.CAME8bitFull(ps, lr=1e-3)
        opt.step()
        return ps, opt

    def noncontiguous(ps, opt):
        ps[0].grad = torch.ones(6, 4, device="cuda").t()

    def float64(ps, opt):
        ps[1].data = ps[1].data.double()
        ps[1].grad = None
        ps[1].grad = torch.ones(9, device="cuda", dtype=torch.float64)

    def no_state(ps, opt):
        opt.state.pop(ps[1])

    def per_matrix(ps, opt):
        opt.state[ps[0]]["_cuda_factored_nd_ext_path"] = True

    def other_mode(ps, opt):
        opt.state[ps[1]]["_mode"] = "8bit1d"

    def other_blocks(ps, opt):
        opt.state[ps[1]]["exp_avg_absmax"] = torch.ones(2, device="cuda")

    def other_rows(ps, opt):
        opt.state[ps[0]]["factored_row_q"] = torch.zeros(2, 5, device="cuda", dtype=torch.uint8)

    def state_elsewhere(ps, opt):
        opt.state[ps[0]]["exp_avg_q"] = opt.state[ps[0]]["exp_avg_q"].cpu()

    def empty(ps, opt):
        ps[1].data, ps[1].grad = ps[1].data[:0], None
        ps[1].grad = torch.ones(0, device="cuda")

    for change in (noncontiguous, float64, no_state, per_matrix, other_mode, other_blocks, other_rows, state_elsewhere, empty):
        ps, opt = fresh()
        change(ps, opt)
        assert _gather(opt, ps)[0] is None, change.__name__
        assert opt.state[ps[0]]["step"] == 1, change.__name__
