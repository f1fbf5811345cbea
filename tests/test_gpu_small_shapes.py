"""Edge shapes of the thread-per-matrix passes, of the kernels for small and narrow tensors and of the one-workgroup step,
each step teacher-forced against the oracle under the tolerances of test_gpu_parity.py; the one-workgroup step against the
passes, and steps over unaligned buffers against aligned ones."""
import ctypes

import pytest
import torch

import came_amd
from came_amd import _lib
from oracle import came8_oracle as orc
from tests import parity as P
from tests.test_gpu_parity import _tight_step_check
from tests.test_gpu_side_stream import _static_step

pytestmark = pytest.mark.gpu

HP = dict(lr=1e-3, weight_decay=1e-2)
# matrices of 1 to 64 elements, around the counts staged at a time and of a work item (256; 128 above 48 elements)
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


@pytest.mark.parametrize("exact_norm", [False, True])
def test_items_of_several_batches(exact_norm):
    """Above 4096 work items of 256 matrices an item takes more of them."""
    _run(came_amd.CAME8bitFull, [(256 * 4096 + 300, 1, 1), (9, 3, 3)], torch.bfloat16, 256, exact_norm, heavy=False, seed=72)


# Many row bands in few state blocks, whose column sums are spread over wavefronts, and the same matrix among others, whose
# columns a thread adds: band counts with every remainder of its batches of sixteen and four, blocks over several matrices
BANDS = [(1000, 300)]
COLUMNS = [(1000, 300)] * 12 + [(8 * k + r, 264) for k, r in ((1, 0), (1, 1), (3, 7), (4, 0), (15, 8), (16, 1), (18, 8), (35, 0))] + [
    (5, 200, 40), (70, 24, 9), (3, 130, 300)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("exact_norm", [False, True])
@pytest.mark.parametrize("shapes", [BANDS, COLUMNS], ids=["spread", "columns"])
def test_band_sums(shapes, dtype, exact_norm):
    _run(came_amd.CAME8bitFull, shapes, dtype, 64, exact_norm, heavy=False, seed=33)


# Small and just larger tensors in one call: the larger ones take them all through the passes, with rows of fewer and more
# columns than threads and lengths with every tail of the norm's chains.
SMALL = [(1,), (7,), (12,), (4095,), (4096,), (4099,), (32768,), (32769,), (1, 1), (1, 300), (300, 1), (5, 8), (96, 200),
         (16, 1280), (1280, 16), (2560, 12), (12, 2548), (13, 2548), (64, 64), (65, 63), (181, 181), (256, 128),
         (129, 255), (31, 1057), (1, 32767), (1, 4, 1000), (3, 40, 60)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("block", [64, 100, 256, 4096])
@pytest.mark.parametrize("exact_norm", [False, True])
def test_small_tensors(dtype, block, exact_norm):
    heavy = block == 64 and dtype != torch.float16
    _run(came_amd.CAME8bitFull, SMALL, dtype, block, exact_norm, heavy=heavy, seed=91)


# One workgroup's steps.  SHORT takes 256 threads a tensor (up to 2048 elements), LONG 1024 (up to 32768 elements and 2560
# rows and columns): a row, a column, both sizes' edges, rows of fewer and more columns than threads, and lengths with
# every remainder of the norm's eight chains below and above their 16-element batches.
SHORT = [(1,), (2,), (3,), (4,), (5,), (6,), (7,), (8,), (12,), (13,), (14,), (15,), (127,), (129,), (2041,), (2042,),
         (2043,), (2044,), (2045,), (2046,), (2047,), (2048,), (1, 1), (1, 300), (300, 1), (5, 8), (64, 32), (45, 45),
         (2, 1024), (1024, 2), (1, 2048), (2048, 1), (1, 4, 500)]
LONG = [(2049,), (4095,), (4096,), (4099,), (20003,), (32761,), (32766,), (32767,), (32768,), (96, 200), (16, 1280), (1280, 16),
        (2547, 12), (12, 2548), (13, 2520), (64, 64), (65, 63), (181, 181), (256, 128), (127, 258), (31, 1057),
        (1, 2559), (2559, 1), (1, 40, 800), (1, 1, 16, 2032)]
# just past an edge, each of which takes a whole call through the passes
PAST = [(32769,), (129, 255), (13, 2548), (1, 2560), (2560, 1), (3, 40, 60)]


def _count(shape):
    return torch.Size(shape).numel()


def _phases(step):
    """The kernels that step() launched, by name."""
    _lib.profile_enable(True)
    try:
        _lib.profile_read(reset=True)
        step()
        torch.cuda.synchronize()
        return {k for k, v in _lib.profile_read(reset=True).items() if v[0]}
    finally:
        _lib.profile_enable(False)


def _optimizer(cls, shapes, dtype=torch.float32, gdtype=None, offset=0, seed=5, std=1e-3, **kw):
    """An optimizer over tensors `offset` elements into their buffers."""
    gen = torch.Generator().manual_seed(seed)
    ps = []
    for s in shapes:
        n = _count(s)
        p = torch.empty(n + offset, device="cuda", dtype=dtype)[offset:].view(s)
        g = torch.empty(n + offset, device="cuda", dtype=gdtype or dtype)[offset:].view(s)
        p.copy_(torch.randn(s, generator=gen) * 0.02)
        g.copy_(torch.randn(s, generator=gen) * std)
        q = torch.nn.Parameter(p)
        if gdtype is not None:
            q.grad_dtype = gdtype
        q.grad = g
        ps.append(q)
    return ps, getattr(came_amd, cls)(ps, **{**HP, **kw})


@pytest.mark.parametrize("shapes", [SHORT, LONG, SHORT + LONG], ids=["short", "long", "both"])
@pytest.mark.parametrize("cls", ["CAME8bitFull", "CAMECUDA"])
def test_calls_of_small_tensors_take_one_launch(shapes, cls):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    _, opt = _optimizer(cls, shapes)
    assert _phases(opt.step) == {"small_step"}
    for s in PAST:
        _, opt = _optimizer(cls, SHORT[:3] + [s])
        ran = _phases(opt.step)
        assert "small_step" not in ran and ran, s


# (tensors, class, whether one launch takes them with the default clip, and with the exact one): both sides of each line
# that the host draws where the passes are the faster (small_call)
LINES = [([(4096,)], "CAME8bit", True, True), ([(4097,)], "CAME8bit", True, False),
         ([(4097,)] * 191, "CAME8bit", True, False), ([(4097,)] * 192, "CAME8bit", True, True),
         ([(8192,)], "CAMECUDA", True, True), ([(8193,)] * 63, "CAMECUDA", True, False),
         ([(8193,)] * 64, "CAMECUDA", True, True), ([(128, 128), (16384,)], "CAME8bit", True, True),
         ([(16, 1025)] * 95 + [(8,)] * 9, "CAME8bit", True, False), ([(16, 1025)] * 96, "CAME8bit", True, True),
         ([(16, 1025)] * 63, "CAMECUDA", True, False), ([(16, 1025)] * 64, "CAMECUDA", True, True),
         ([(28672,)], "CAME8bit", True, False), ([(28673,)] * 31, "CAME8bit", False, False),
         ([(28673,)] * 32, "CAME8bit", True, False), ([(28673,)], "CAMECUDA", True, False),
         ([(28673,), (8, 8)], "CAME8bit", True, False), ([(16, 1024)] * 640, "CAME8bit", True, True),
         ([(16, 1024)] * 641, "CAME8bit", True, False), ([(16, 1023)] * 641, "CAME8bit", True, True),
         ([(16, 2048)] * 768, "CAME8bit", True, False), ([(16, 2048)] * 769, "CAME8bit", False, False),
         ([(16, 2048)] * 769, "CAMECUDA", True, True)]


@pytest.mark.parametrize("line", LINES, ids=lambda c: f"{len(c[0])}x{c[0][0]}-{c[1]}")
def test_lines_between_one_launch_and_the_passes(line):
    """Each mode by itself and after the other one (the plan of a step serves both)."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    shapes, cls, default, exact = line
    _, opt = _optimizer(cls, shapes)
    for mode, small in ((True, exact), (False, default), (True, exact)):
        opt.exact_norm = mode
        ran = _phases(opt.step)
        assert ("small_step" in ran) == small and (ran == {"small_step"}) == small, (mode, ran)


@pytest.mark.parametrize("shapes", [[(8192,), (16384,), (4099,)], [(96, 200), (181, 181), (9,)]], ids=["vectors", "matrices"])
def test_modes_of_different_routes_match_the_oracle(shapes):
    """The default clip in one launch, the exact one through the passes, of one set."""
    for exact_norm in (False, True):
        _run(came_amd.CAME8bitFull, shapes, torch.float32, 256, exact_norm, heavy=False, seed=17)


def test_one_launch_where_the_passes_do_not_fit():
    """A call that the passes would take, in a workspace that is too small for their scratch (the 32 MiB of the static
    entry point): one launch, and the same step."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    shapes = [(16, 2048)] * 900
    out = []
    for entry in (lambda opt, ps: opt.step(), _static_step):
        ps, opt = _optimizer("CAME8bit", shapes)
        out.append((ps, opt, _phases(lambda: entry(opt, ps))))
    assert "small_step" not in out[0][2] and out[1][2] == {"small_step"}
    _same_steps([(ps, [opt.state[p] for p in ps]) for ps, opt, _ in out], shapes)


def test_workspace_sizes_of_one_plan():
    """A workspace of more bytes than a call needs has the plan that those bytes made (what a step under capture relies
    on); one too small for the passes has a plan without them, until it is larger again."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lib = _lib.load()
    ps, opt = _optimizer("CAME8bit", [(20003,), (32768,)])
    opt.step()
    descs, _, _ = opt._descriptors([(p, opt.state[p], p.grad) for p in ps])
    hp = opt._group_hparams(opt.param_groups[0])
    need = ctypes.c_size_t(0)
    _lib.check(lib.came8_workspace_size(descs, 2, 256, ctypes.byref(need)), "came8_workspace_size")
    ws, tag = torch.empty(2 * need.value, dtype=torch.uint8, device="cuda"), _lib.new_workspace_tag()
    stream = torch.cuda.current_stream().cuda_stream

    def step(nbytes, flags=0):
        hp.flags = flags
        return _phases(lambda: _lib.check(lib.came8_step(descs, 2, ctypes.byref(hp), ws.data_ptr(), nbytes, tag, stream),
                                          "came8_step"))

    assert step(need.value, _lib.CAME8_FLAG_PLAN_ONLY) == set()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        stream = torch.cuda.current_stream().cuda_stream
        hp.flags = 0
        _lib.check(lib.came8_step(descs, 2, ctypes.byref(hp), ws.data_ptr(), 2 * need.value, tag, stream), "came8_step")
    graph.replay()
    torch.cuda.synchronize()
    del graph
    stream = torch.cuda.current_stream().cuda_stream
    assert "small_step" not in step(need.value)
    assert step(need.value - 1) == {"small_step"}
    assert "small_step" not in step(need.value)
    with pytest.raises(RuntimeError):
        step(1024)
    lib.came8_release_workspace(ws.data_ptr())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("block", [64, 100, 256, 4096])
@pytest.mark.parametrize("exact_norm", [False, True])
@pytest.mark.parametrize("shapes", [SHORT, LONG], ids=["short", "long"])
def test_one_workgroup_steps(shapes, dtype, block, exact_norm):
    if exact_norm:  # past 16384 elements it takes a crowd (test_one_launch_matches_the_passes)
        shapes = [s for s in shapes if _count(s) <= 16384]
    heavy = block == 64 and dtype != torch.float16
    _run(came_amd.CAME8bitFull, shapes, dtype, block, exact_norm, heavy=heavy, seed=91)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("block", [256, 100])
def test_small_vectors_with_the_fp16_rounded_update(dtype, block):
    """Teacher-forced against the oracle's fp16_update branch, as test_gpu_fp16_update.py runs it on calls that hold a
    large tensor."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    shapes = [s for s in SHORT + LONG if len(s) == 1 and s[0] <= 28672]
    params = P.make_params(shapes, dtype, seed=block)
    gen = torch.Generator().manual_seed(block + 1)
    hp = dict(HP, block_size=block)
    ps = [torch.nn.Parameter(p.cuda()) for p in params]
    opt = came_amd.CAME8bitFull(ps, cuda_nonfactored_use_fp16_update=True, **hp)
    sts = [orc.init_full8bit_state(p.shape, block) for p in params]
    check = _tight_step_check(f"small fp16 update {dtype} B={block}", block=block)
    for step in range(2):
        with torch.no_grad():
            for p, r, st in zip(ps, params, sts):
                p.data.copy_(r)
                for k in P.STATE_KEYS:
                    if len(opt.state[p]) and k in st:
                        opt.state[p][k].copy_(st[k])
        grads = [P.heavy_grad(gen, s, dtype) for s in shapes]
        for p, g in zip(ps, grads):
            p.grad = g.cuda()
        assert _phases(opt.step) == {"small_step"}
        for i, (r, g, st) in enumerate(zip(params, grads, sts)):
            before, cap = r.double(), {}
            orc.full8bit_step(r, g, st, capture=cap, fp16_update=True, **P.oracle_hp(hp))
            check(step + 1, i, ps[i].data, r, opt.state[ps[i]], st, (r.double() - before).abs(), cap)


# the one launch against the passes, which one large tensor more in the call brings about: every class, pair of types,
# alignment, block size and mode that both take
ROUTES = [dict(cls="CAME8bitFull"), dict(cls="CAME8bitFull", block_size=100), dict(cls="CAME8bitFull", block_size=2048),
          dict(cls="CAME8bitFull", offset=1), dict(cls="CAME8bitFull", exact_norm=True),
          dict(cls="CAME8bitFull", cuda_nonfactored_use_fp16_update=True, block_size=64),
          dict(cls="CAME8bitFull", dtype=torch.bfloat16, offset=3), dict(cls="CAME8bitFull", dtype=torch.float16),
          dict(cls="CAME8bitFull", dtype=torch.bfloat16, gdtype=torch.float32),
          dict(cls="CAME8bitFull", dtype=torch.float32, gdtype=torch.float16),
          dict(cls="CAME8bitMemory", betas=(0.9, 0.95, 0.995), weight_decay=0.0), dict(cls="CAME8bit", clip_threshold=0.25),
          dict(cls="CAMECUDA"), dict(cls="CAMECUDA", offset=1, exact_norm=True), dict(cls="CAMECUDA", dtype=torch.bfloat16)]


@pytest.mark.parametrize("route", ROUTES, ids=lambda r: "-".join(str(v) for v in r.values()))
def test_one_launch_matches_the_passes(route):
    """Sums may be ordered otherwise, hence the tolerances of the parity tests (codes one apart, 1e-5 of parameters and
    scales); a 16-bit parameter may round to its neighbour."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    route = dict(route)
    exact = route.pop("exact_norm", False)
    cls = route.pop("cls")
    shapes = SHORT + LONG + ([(181, 181), (31, 1057), (2547, 12), (20003,)] * 24 if exact else [])
    out = []
    for more in ([], [(300, 200)]):
        ps, opt = _optimizer(cls, shapes + more, **route)
        opt.exact_norm = exact
        ran = _phases(opt.step)
        assert (ran == {"small_step"}) == (not more)
        out.append((ps, [opt.state[p] for p in ps]))
    _same_steps(out, shapes, {torch.float32: 0.0, torch.bfloat16: 2**-7, torch.float16: 2**-10}[out[0][0][0].dtype])


def _same_steps(out, shapes, ulp=0.0):
    for i, s in enumerate(shapes):
        a, b = out[0][0][i].data.double(), out[1][0][i].data.double()
        assert ((a - b).abs() <= (1e-5 + ulp) * b.abs() + 2e-7 + 1e-3 * HP["lr"]).all(), s
        for k, v in out[1][1][i].items():
            if not isinstance(v, torch.Tensor) or v.numel() == 0:
                continue
            w = out[0][1][i][k]
            if v.dtype.is_floating_point:
                assert torch.allclose(w, v, rtol=1e-4, atol=1e-5 * v.abs().max().item()), (s, k)
            else:
                assert (w.int() - v.int()).abs().max() <= 1, (s, k)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("cls", ["CAME8bitFull", "CAMECUDA"])
def test_non_finite_gradients_match_the_passes(cls, bad):
    """One infinite or NaN gradient in each of some tensors: the same parameters, scales and fp32 states come out NaN,
    infinite and finite as from the passes, and the other tensors step bit for bit as without it."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    shapes = [(9,), (2048,), (4099,), (5, 8), (96, 200), (1, 300), (64, 32)]
    hit = (1, 2, 3, 4)
    out = []
    for more, where in (([], hit), ([(300, 200)], hit), ([], ())):
        ps, opt = _optimizer(cls, shapes + more)
        for i in where:
            ps[i].grad.view(-1)[7] = bad
        ran = _phases(opt.step)
        assert (ran == {"small_step"}) == (not more)
        out.append([[p.data] + [v for v in opt.state[p].values() if isinstance(v, torch.Tensor) and v.dtype == torch.float32]
                    for p in ps[: len(shapes)]])
    for i, s in enumerate(shapes):
        for a, b, c in zip(*(o[i] for o in out)):
            assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()), s
            fin = a.isfinite()
            assert torch.allclose(a[fin], b[fin], rtol=1e-4, atol=1e-6), s
            assert i in hit or torch.equal(a, c), s


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
