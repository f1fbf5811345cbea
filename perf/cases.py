"""Performance cases of the CAME 8-bit optimizers: what one optimizer step (or one blockwise quantisation round
trip) costs over the range of parameter sets that the classes are used on.

A case is a dict of plain values:

  opt       the class stepped (CAME8bit, CAME8bitFull, CAME8bitMemory, CAME8bit2D, CAMECUDA), or "quant" for
            quantize_blockwise / dequantize_blockwise
  shapes    the parameter set, "4*4096x4096;2*4096" = four 4096x4096 matrices and two vectors of 4096, in order
  dtype     of parameters and gradients
  grad      "normal" (each tensor N(0, std^2)), "heavy" (Student-t with nu = 2, a tenth exact zeros, and +-1e3
            outliers: the ragged stress set's distribution) or "scales" (N(0, std^2) times a scale per tensor,
            log-uniform in [1e-5, 1e-2])
  std       of the gradients
  vscale    the second moments held against the gradients' own: below 1 the update's RMS is above the clip
            threshold (the gradients grew, the clip acts), above 1 it is below it
  block     quantisation block size
  exact     the exactly rounded clip norm (opt.exact_norm) instead of the reference's float32 order

A state is what a training program holds in the middle of a run: parameters, gradients and 8-bit states as views of
flat buffers, one per kind (how sharded and bucketed training keeps them; every tensor starts 512 bytes aligned, as
torch's allocator places one by itself).  run() is one optimizer step; its outputs are those flat buffers, updated.
"""
from __future__ import annotations

import math

import torch

import came_amd
from came_amd import blockwise_quantization as bq

LR, WD, EPS0, EPS1 = 2e-4, 1e-2, 1e-30, 1e-16
BETAS = {"CAME8bitMemory": (0.9, 0.95, 0.995)}
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
ALIGN = 512  # bytes
TILE = 16    # CAME8bit2D's momentum tiles


def _layers(n, d, ffn, head=True):
    """n decoder layers: attention 4 x (d, d), gated MLP 2 x (ffn, d) + (d, ffn), two norm weights."""
    return ";".join([f"4*{d}x{d};2*{ffn}x{d};{d}x{ffn};2*{d}"] * n) + (f";{d}" if head else "")


def _gpt(n, d, vocab, pos):
    """n decoder layers with fused qkv and biases, tied embedding, learned positions."""
    layer = f"2*{d};{3 * d}x{d};{3 * d};{d}x{d};{d};2*{d};{4 * d}x{d};{4 * d};{d}x{4 * d};{d}"
    return ";".join(([f"{vocab}x{d};{pos}x{d}"] if vocab else []) + [layer] * n + [f"2*{d}"])


def _lora(n, rank, dims):
    """n adapters of that rank on projections between the widths `dims`, down and up matrices."""
    out = []
    for i in range(n):
        a, b = dims[i % len(dims)], dims[(i // 2) % len(dims)]
        out.append(f"{rank}x{a};{b}x{rank}")
    return ";".join(out)


def _case(name, opt, shapes, dtype="fp32", grad="normal", std=1e-3, vscale=1.15, block=256, exact=False):
    return dict(name=name, opt=opt, shapes=shapes, dtype=dtype, grad=grad, std=std, vscale=vscale, block=block,
                exact=exact)


# Named shapes of the ragged stress set, with 1-D lengths and odd matrices of its ranges.
RAGGED = ("17;4097;1;2011;640;3333;1000x3;3x50257;4097x129;320x320x3x3;1280x640x1x1;1283x2741;4999x33;77x4801;"
          "2501x2503;611x1999;3847x1201;5x4999;1751x4459;4423x2377;127x3001;2999x799;1597x4093;950;3001x3011;"
          "45x45;1023x1;1x1023;3971x4871;211x4241;4001x2003")


def listed():
    return [
        # the smallest: a small network's few tensors, a step that is all latency
        _case("small_net_fp32", "CAME8bit", "96x200;96;10x96;10"),
        # one linear layer of a fine-tune (a single 2048x2048 matrix and its bias)
        _case("linear_2048_fp32", "CAME8bit", "2048x2048;2048"),
        # low-rank adapters of an image model's attention: hundreds of small matrices (the usual adapter training)
        _case("adapters_fp32", "CAME8bit", _lora(96, 16, (640, 1280, 1280, 2048)), std=2e-4, vscale=0.8),
        # convolution and projection weights of an image model's blocks, N-D states
        _case("conv_blocks_bf16", "CAME8bit",
              "320x4x3x3;320;2*320x320x3x3;2*320;640x320x3x3;640;640x640x3x3;640;1280x640x1x1;1280;1280x1280x3x3;1280;"
              "1280x1280;5120x1280", "bf16", std=5e-4),
        # all of a medium language model in fp32: the many-tensor step of ordinary size
        _case("gpt2_medium_fp32", "CAME8bit", _gpt(24, 1024, 50257, 1024), grad="scales", vscale=0.9),
        # a 1B-style model's layers with an odd MLP width and its embedding, compact states
        _case("llama1b_memory_bf16", "CAME8bitMemory", "32000x2048;" + _layers(4, 2048, 5461), "bf16", std=5e-4),
        # the largest: embedding, four layers and head of a 7B-shape model
        _case("llama7b_bf16", "CAME8bit", "32000x4096;" + _layers(4, 4096, 11008) + ";32000x4096", "bf16", std=2e-4,
              vscale=1.0),
        # ragged tensors, heavy-tailed gradients: no shape or alignment is a round one
        _case("ragged_heavy_fp32", "CAME8bitFull", RAGGED, grad="heavy"),
        # one 7B layer's matrices with tile-quantised momentum
        _case("layer_2d_bf16", "CAME8bit2D", "4*4096x4096;2*11008x4096;4096x11008", "bf16", std=2e-4),
        # one 7B layer with fp32 optimizer states
        _case("layer_fp32states_bf16", "CAMECUDA", _layers(1, 4096, 11008, False), "bf16", std=2e-4),
        # transformer blocks trained in fp16 with the exactly rounded clip, small quantisation blocks
        _case("blocks_exact_fp16", "CAME8bit", _gpt(4, 1536, 0, 0), "fp16", std=1e-2, vscale=0.9, block=128, exact=True),
        # the blockwise quantisation helpers on one large momentum tensor (state conversion, checkpoints): encode and
        # decode
        dict(name="quant_roundtrip_fp32", opt="quant", shapes="11008x4096", signed=True, block=256),
    ]


def _spread(rng, lo, hi):
    """A whole number in [lo, hi], uniform over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("quant", "few", "few", "model", "model", "adapters", "ragged", "conv", "2d", "fp32states"))
    dtype = rng.choice(("fp32", "bf16", "bf16", "fp16"))
    std = {"fp16": 1e-2}.get(dtype, 10.0 ** rng.uniform(-4, -2.5))
    more = dict(dtype=dtype, std=std, vscale=round(rng.uniform(0.8, 1.25), 3))
    block = rng.choice((64, 128, 256, 256, 256, 512, 1024, 2048))
    opt = rng.choice(("CAME8bit", "CAME8bitFull", "CAME8bitMemory"))
    if kind == "quant":
        c = dict(name="", opt="quant", shapes=f"{_spread(rng, 1, 11008)}x{_spread(rng, 64, 8192)}",
                 signed=rng.random() < 0.5, block=rng.choice((64, 100, 256, 256, 1000, 2048, 4096)))
    elif kind == "few":  # a few matrices of any size, and vectors
        shapes = [f"{_spread(rng, 8, 8192)}x{_spread(rng, 8, 8192)}" for _ in range(rng.randint(1, 4))]
        shapes += [str(_spread(rng, 1, 20000)) for _ in range(rng.randint(0, 3))]
        c = _case("", opt, ";".join(shapes), block=block, exact=rng.random() < 0.2, **more)
    elif kind == "model":  # a decoder stack with its embedding
        d = 64 * _spread(rng, 4, 64)
        n = max(1, min(24, int(4e8 / (12 * d * d))))
        if rng.random() < 0.5:
            shapes = f"{_spread(rng, 1000, 32000)}x{d};" + _layers(rng.randint(1, n), d, int(d * rng.uniform(2.5, 2.8)))
        else:
            shapes = _gpt(rng.randint(1, n), d, _spread(rng, 1000, 50257), 1024)
        c = _case("", opt, shapes, block=block, exact=rng.random() < 0.2, **more)
    elif kind == "adapters":
        dims = [64 * _spread(rng, 5, 64) for _ in range(4)]
        c = _case("", opt, _lora(_spread(rng, 8, 140), rng.choice((4, 8, 16, 32, 64, 128)), dims), block=block, **more)
    elif kind == "ragged":
        shapes = [str(rng.randint(1, 4097)) for _ in range(rng.randint(2, 12))]
        shapes += [f"{rng.randint(1, 5000)}x{rng.randint(1, 5000)}" for _ in range(rng.randint(2, 20))]
        c = _case("", "CAME8bitFull", ";".join(shapes), "fp32", "heavy", 1e-3, 1.15, block)
    elif kind == "conv":
        shapes = []
        for _ in range(rng.randint(2, 8)):
            k = rng.choice((1, 3, 3, 5))
            shapes.append(f"{_spread(rng, 4, 1280)}x{_spread(rng, 3, 1280)}x{k}x{k}")
            shapes.append(shapes[-1].split("x")[0])
        c = _case("", opt, ";".join(shapes), block=block, **more)
    elif kind == "2d":
        shapes = [f"{_spread(rng, 16, 8192)}x{_spread(rng, 16, 8192)}" for _ in range(rng.randint(1, 6))]
        c = _case("", "CAME8bit2D", ";".join(shapes), **more)
    else:
        shapes = [f"{_spread(rng, 16, 8192)}x{_spread(rng, 16, 8192)}" for _ in range(rng.randint(1, 4))]
        shapes += [str(_spread(rng, 1, 20000)) for _ in range(2)]
        c = _case("", "CAMECUDA", ";".join(shapes), **more)
    c.pop("name")
    return c


# ------------------------------------------------------------------------------------------- inputs
def _shapes(case):
    out = []
    for part in case["shapes"].split(";"):
        n, _, s = part.rpartition("*")
        out += [tuple(int(x) for x in s.split("x"))] * (int(n) if n else 1)
    return out


def _blocks(n, block):
    return max(1, -(-n // block))


class _Flat:
    """One buffer holding a tensor per shape, each 512-byte aligned."""

    def __init__(self, shapes, dtype, fill=0):
        size = torch.empty((), dtype=dtype).element_size()
        at, offs = 0, []
        for s in shapes:
            offs.append(at)
            at += -(-math.prod(s) * size // ALIGN) * ALIGN // size
        self.all = torch.full((max(at, 1),), fill, dtype=dtype, device="cuda")
        self.views = [self.all[o : o + math.prod(s)].view(s) for o, s in zip(offs, shapes)]


def _gradient(case, shape, scale, gen):
    n = math.prod(shape)
    if case["grad"] != "heavy":
        return torch.randn(shape, device="cuda", generator=gen).mul_(case["std"] * scale)
    g = torch.randn(n, device="cuda", generator=gen)
    g /= torch.rand(n, device="cuda", generator=gen).clamp_min_(1e-30).log_().neg_().sqrt_()
    g.mul_(case["std"]).masked_fill_(torch.rand(n, device="cuda", generator=gen) < 0.1, 0.0)
    pos = torch.arange(-(-n // 256), device="cuda") * 256
    pos = pos + torch.randint(0, 256, pos.shape, device="cuda", generator=gen)
    hit = (torch.rand(pos.shape, device="cuda", generator=gen) < 0.5) & (pos < n)
    sign = torch.randint(0, 2, pos.shape, device="cuda", generator=gen) * 2.0 - 1.0
    g.index_copy_(0, pos[hit], 1e3 * sign[hit])
    return g.view(shape)


def _codes(x, signed, block, q, a):
    """Blockwise codes and scales of x into q and a (the state a past step would have left)."""
    flat = x.reshape(-1)
    n, qmax = flat.numel(), 127.0 if signed else 255.0
    pad = _blocks(n, block) * block
    buf = flat if pad == n else torch.cat([flat, flat.new_zeros(pad - n)])
    buf = buf.view(-1, block)
    amax = buf.abs().amax(1)
    amax = torch.where(amax > 0, amax, torch.ones_like(amax))
    a.copy_(amax.view(a.shape))
    q.copy_(torch.round(buf / amax[:, None] * qmax).clamp_(-qmax, qmax).reshape(-1)[:n].view(q.shape))


def _tile_codes(x, q, a):
    """Codes and scales of x in 16x16 tiles."""
    r, c = x.shape
    tr, tc = -(-r // TILE), -(-c // TILE)
    buf = x.new_zeros(tr * TILE, tc * TILE)
    buf[:r, :c] = x
    amax = buf.view(tr, TILE, tc, TILE).abs().amax((1, 3))
    amax = torch.where(amax > 0, amax, torch.ones_like(amax))
    a.copy_(amax.reshape(-1))
    wide = amax.repeat_interleave(TILE, 0).repeat_interleave(TILE, 1)[:r, :c]
    q.copy_(torch.round(x / wide * 127.0).clamp_(-127, 127))


def _inputs(case, seed):
    """Parameters, gradients and states of a case, from the seed alone: flat buffers, and their views per tensor."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["opt"] == "quant":
        shape, = _shapes(case)
        x = torch.randn(shape, device="cuda", generator=gen)
        x.mul_(torch.exp(torch.randn(shape[:-1] + (1,), device="cuda", generator=gen)))  # rows of their own scale
        return {"x": x if case["signed"] else x.abs_()}
    shapes, dt, B = _shapes(case), DTYPES[case["dtype"]], case["block"]
    opt = case["opt"]
    fp32st, tiles = opt == "CAMECUDA", opt == "CAME8bit2D"
    rows = [s[:-1] if len(s) >= 2 else (0,) for s in shapes]
    cols = [s[:-2] + s[-1:] if len(s) >= 2 else (0,) for s in shapes]
    vecs = [s if len(s) < 2 else (0,) for s in shapes]
    buf = {"p": _Flat(shapes, dt), "g": _Flat(shapes, dt)}
    f32 = torch.float32
    if fp32st:
        buf.update(m=_Flat(shapes, f32), sq_row=_Flat(rows, f32), sq_col=_Flat(cols, f32), res_row=_Flat(rows, f32),
                   res_col=_Flat(cols, f32), v=_Flat(vecs, f32))
    else:
        two = [(2,) + r for r in rows], [(2,) + c for c in cols]
        nblk = lambda ss, k: [(k, _blocks(math.prod(s), B)) for s in ss]  # noqa: E731
        mblk = ([(-(-s[0] // TILE) * -(-s[1] // TILE),) for s in shapes] if tiles
                else [(_blocks(math.prod(s), B),) for s in shapes])
        buf.update(mq=_Flat(shapes, torch.int8), ma=_Flat(mblk, f32),
                   rq=_Flat(two[0], torch.uint8), ra=_Flat(nblk(rows, 2), f32, 1.0),
                   cq=_Flat(two[1], torch.uint8), ca=_Flat(nblk(cols, 2), f32, 1.0))
        if not tiles:
            buf.update(vq=_Flat(vecs, torch.uint8), va=_Flat([(_blocks(math.prod(s), B),) for s in vecs], f32, 1.0))
    draw1 = lambda s, lo, hi: torch.rand(s, device="cuda", generator=gen).mul_(hi - lo).add_(lo)  # noqa: E731
    scales = ([1.0] * len(shapes) if case["grad"] != "scales"
              else torch.pow(10.0, draw1((len(shapes),), -5.0, -2.0)).tolist())
    for i, s in enumerate(shapes):
        buf["p"].views[i].copy_(torch.randn(s, device="cuda", generator=gen).mul_(0.02))
        g = _gradient(case, s, scales[i], gen)
        buf["g"].views[i].copy_(g)
        m = torch.randn(s, device="cuda", generator=gen).mul_(0.25)  # about the running mean of the updates
        sq = g.square_()
        if len(s) < 2:
            v = draw1(s, 0.7, 1.3).mul_(sq.mean() * case["vscale"])
            if fp32st:
                buf["m"].views[i].copy_(m)
                buf["v"].views[i].copy_(v)
            else:
                _codes(m, True, B, buf["mq"].views[i], buf["ma"].views[i])
                _codes(v, False, B, buf["vq"].views[i], buf["va"].views[i])
            continue
        state = [[sq.mean(-1) * case["vscale"], sq.mean(-2) * case["vscale"]],
                 [torch.full(rows[i], 0.9, device="cuda"), torch.full(cols[i], 0.9, device="cuda")]]
        for pair in state:
            for x in pair:
                x.mul_(draw1(x.shape, 0.8, 1.2))
        if fp32st:
            buf["m"].views[i].copy_(m)
            for k, pair in zip(("sq", "res"), state):
                for ax, x in zip(("row", "col"), pair):
                    buf[f"{k}_{ax}"].views[i].copy_(x)
            continue
        if tiles:
            _tile_codes(m, buf["mq"].views[i], buf["ma"].views[i])
        else:
            _codes(m, True, B, buf["mq"].views[i], buf["ma"].views[i])
        for k, pair in enumerate(state):
            _codes(pair[0], False, B, buf["rq"].views[i][k], buf["ra"].views[i][k])
            _codes(pair[1], False, B, buf["cq"].views[i][k], buf["ca"].views[i][k])
    return buf


def _state_of(case, buf, i, shape):
    """The optimizer state of tensor i over its views (the layouts that checkpoints hold)."""
    v = {k: f.views[i] for k, f in buf.items()}
    if case["opt"] == "CAMECUDA":
        st = dict(step=1, _mode="cudafp", factored=len(shape) >= 2, exp_avg=v["m"])
        if len(shape) >= 2:
            st.update(exp_avg_sq_row=v["sq_row"], exp_avg_sq_col=v["sq_col"], exp_avg_res_row=v["res_row"],
                      exp_avg_res_col=v["res_col"])
        else:
            st["exp_avg_sq"] = v["v"]
        return st
    if case["opt"] == "CAME8bit2D":
        r, c = shape
        tr, tc = -(-r // TILE), -(-c // TILE)
        st = dict(_mode="8bit2d", rows=r, cols=c, tile_rows=tr, tile_cols=tc, num_tiles=tr * tc, exp_avg_q=v["mq"],
                  exp_avg_absmax=v["ma"], res_row_partial=torch.empty(tc * r, device="cuda"),
                  res_col_partial=torch.empty(tr * c, device="cuda"))
        for k, kind in enumerate(("sq", "res")):
            for ax, n in (("row", "r"), ("col", "c")):
                st[f"exp_avg_{kind}_{ax}_q"], st[f"exp_avg_{kind}_{ax}_absmax"] = v[n + "q"][k], v[n + "a"][k]
        return st
    st = dict(step=1, _mode="full8bit", RMS=0, factored=len(shape) >= 2, exp_avg_q=v["mq"], exp_avg_absmax=v["ma"])
    if len(shape) >= 2:
        st.update(factored_row_q=v["rq"], factored_row_absmax=v["ra"], factored_col_q=v["cq"],
                  factored_col_absmax=v["ca"])
    else:
        st.update(exp_avg_sq_q=v["vq"], exp_avg_sq_absmax=v["va"])
    return st


def prepare(case, seed):
    buf = _inputs(case, seed)
    if case["opt"] == "quant":
        return dict(case=case, x=buf["x"])
    shapes = _shapes(case)
    params = []
    for p, g in zip(buf["p"].views, buf["g"].views):
        q = torch.nn.Parameter(p)
        q.grad = g
        params.append(q)
    kw = dict(lr=LR, eps=(EPS0, EPS1), betas=BETAS.get(case["opt"], (0.9, 0.999, 0.9999)), weight_decay=WD)
    if case["opt"] not in ("CAMECUDA", "CAME8bit2D"):
        kw["block_size"] = case["block"]
    opt = getattr(came_amd, case["opt"])(params, **kw)
    if case["exact"]:
        opt.exact_norm = True
    for i, (p, s) in enumerate(zip(params, shapes)):
        opt.state[p] = _state_of(case, buf, i, s)
    return dict(case=case, opt=opt, out={k: f.all for k, f in buf.items() if k != "g"})


def run(state):
    if "opt" in state:
        state["opt"].step()
        return state["out"]
    c = state["case"]
    q, a = bq.quantize_blockwise(state["x"], signed=c["signed"], block_size=c["block"])
    return {"q": q, "a": a, "x": bq.dequantize_blockwise(q, a, signed=c["signed"], block_size=c["block"])}


# ------------------------------------------------------------------------------- work and tolerance
def work(case):
    if case["opt"] == "quant":
        n = math.prod(_shapes(case)[0])
        return {"bytes": n * (4 + 1 + 4) + 4 * _blocks(n, case["block"]), "flops": 4 * n}
    tot = flops = 0
    s = 4 if case["dtype"] == "fp32" else 2
    for shape in _shapes(case):
        n = math.prod(shape)
        pr = math.prod(shape[:-1])
        pc = math.prod(shape[:-2] + shape[-1:])
        B = case["block"]
        flops += 30 * n
        tot += 3 * s * n  # the gradient read, the parameter read and written
        if case["opt"] == "CAMECUDA":
            tot += 8 * n + (16 * (pr + pc) if len(shape) >= 2 else 8 * n)
        elif len(shape) < 2:
            tot += 4 * n + 16 * _blocks(n, B)
        else:
            scales = -(-pr // TILE) * -(-pc // TILE) if case["opt"] == "CAME8bit2D" else _blocks(n, B)
            tot += 2 * n + 8 * scales + 4 * (pr + pc) + 16 * (_blocks(pr, B) + _blocks(pc, B))
    return {"bytes": tot, "flops": flops}


def tolerance(case):
    if case["opt"] == "quant":
        return "exact"  # one formula, every rounding of it fixed
    # Row and column means added in another order differ by about 1e-7, which moves a code only where its value lies
    # that near a rounding tie: about 1e-5 of the codes, one in a small state, and with equal outliers (heavy) up to
    # a hundredth of a row state, whose means are then halves of each other.  A 16-bit parameter then rounds to its
    # neighbour as rarely.
    rel, most = {"fp32": (2e-6, 2e-4), "bf16": (1e-4, 0.01), "fp16": (1e-4, 0.0015)}[case["dtype"]]
    few = case["grad"] == "heavy" or sum(math.prod(s) for s in _shapes(case)) < 1_000_000
    return {"rel": rel, "max": most, "differ": 1e-2 if few else 1e-3}


# --------------------------------------------------------------------------------- in 64 bits
def _deq(q, a, signed, block):
    """Flat codes and their scales as float64."""
    return q.double() * a.double().repeat_interleave(block)[: q.numel()] / (127.0 if signed else 255.0)


def _amax(x, block):
    flat = x.reshape(-1)
    pad = _blocks(flat.numel(), block) * block - flat.numel()
    a = torch.nn.functional.pad(flat, (0, pad)).view(-1, block).abs().amax(1)
    return torch.where(a > 0, a, torch.ones_like(a))


def exact(case, seed):
    """The step in float64 from the same inputs.  The clip divides by the exactly rounded norm; the default norm's
    own summation order is a property of 32-bit sums, so where the clip acts its share shows in every output."""
    work_bytes = work(case)["bytes"]
    if work_bytes > 9e9:
        return None
    buf = _inputs(case, seed)
    B = case["block"]
    if case["opt"] == "quant":
        x = buf["x"].double()
        a = _amax(x, B)
        wide = a.repeat_interleave(B)[: x.numel()].view(x.shape)
        qmax = 127.0 if case["signed"] else 255.0
        return {"q": None, "a": a, "x": torch.round(x / wide * qmax) * (wide / qmax)}
    out = {k: (f.all.double() if f.all.is_floating_point() else None) for k, f in buf.items() if k != "g"}
    b1, b2, b3 = BETAS.get(case["opt"], (0.9, 0.999, 0.9999))
    fp32st, tiles = case["opt"] == "CAMECUDA", case["opt"] == "CAME8bit2D"

    def view(k, i):  # the float64 buffer's part that is tensor i's
        v = buf[k].views[i]
        o = v.storage_offset()
        return out[k][o : o + v.numel()].view(v.shape)

    for i, s in enumerate(_shapes(case)):
        g = buf["g"].views[i].double()
        n, fact = g.numel(), len(s) >= 2
        u2 = g * g + EPS0
        if fp32st:
            m = view("m", i).clone()
            old = ([view("sq_row", i), view("sq_col", i), view("res_row", i), view("res_col", i)] if fact
                   else [view("v", i)])
        else:
            mq, ma = buf["mq"].views[i], buf["ma"].views[i]
            if tiles:
                tr, tc = -(-s[0] // TILE), -(-s[1] // TILE)
                wide = ma.double().view(tr, tc).repeat_interleave(TILE, 0).repeat_interleave(TILE, 1)[: s[0], : s[1]]
                m = mq.double() * wide / 127.0
            else:
                m = _deq(mq.reshape(-1), ma, True, B).view(s)
            if fact:
                rq, ra, cq, ca = (buf[k].views[i] for k in ("rq", "ra", "cq", "ca"))
                old = [_deq(q[k].reshape(-1), a[k], False, B).view(q.shape[1:]) for k in (0, 1)
                       for q, a in ((rq, ra), (cq, ca))]
            else:
                old = [_deq(buf["vq"].views[i], buf["va"].views[i], False, B)]

        def factors(row, col):
            mean = row.mean(-1, keepdim=True)
            mean = torch.where(mean > 0, mean, torch.ones_like(mean)) if tiles else mean.clamp_min(1e-30)
            return (row / mean).rsqrt().unsqueeze(-1) * col.unsqueeze(-2).rsqrt()

        new = []
        if fact:
            floor = 0.0 if tiles else 1e-30
            row = old[0] * b2 + (1 - b2) * u2.mean(-1)
            col = (old[1] * b2 + (1 - b2) * u2.mean(-2)).clamp_min(floor)
            u = factors(row, col) * g
        else:
            row = (old[0] * b2 + (1 - b2) * u2).clamp_min(1e-30)
            u = row.rsqrt() * g
        u /= max(1.0, float(u.norm()) / math.sqrt(n))
        m = m * b1 + (1 - b1) * u
        p = view("p", i)
        if fact:
            res = (u - m) ** 2 + EPS1
            rrow = old[2] * b3 + (1 - b3) * res.mean(-1)
            rcol = (old[3] * b3 + (1 - b3) * res.mean(-2)).clamp_min(floor)
            new = [row, col, rrow, rcol]
            step = factors(rrow, rcol)
            if tiles:
                tm = torch.zeros(tr * TILE, tc * TILE, dtype=torch.float64, device="cuda")
                tm[: s[0], : s[1]] = m
                amax = tm.view(tr, TILE, tc, TILE).abs().amax((1, 3))
                amax = torch.where(amax > 0, amax, torch.ones_like(amax))
                wide = amax.repeat_interleave(TILE, 0).repeat_interleave(TILE, 1)[: s[0], : s[1]]
                view("ma", i).copy_(amax.reshape(-1))
                step *= torch.round(m / wide * 127.0) * wide / 127.0
            else:
                step *= m
        else:
            new, step = [row], m
        p.mul_(1 - LR * WD).sub_(step, alpha=LR)
        if fp32st:
            view("m", i).copy_(m)
            for k, x in zip(("sq_row", "sq_col", "res_row", "res_col") if fact else ("v",), new):
                view(k, i).copy_(x)
            continue
        if not tiles:
            view("ma", i).copy_(_amax(m, B))
        if fact:
            for k in (0, 1):
                view("ra", i)[k].copy_(_amax(new[2 * k], B))
                view("ca", i)[k].copy_(_amax(new[2 * k + 1], B))
        else:
            view("va", i).copy_(_amax(new[0], B))
    return out
