"""The optimizer's work, as a program that uses it calls it, at the sizes it is used at.

Kinds of case:

* ``step``: one effective batch of the optimizer.  The forward and cotangent
  hooks of every selected matrix see a microbatch's recorded activations and
  cotangents, then ``step()`` updates the matrices (momentum, whitening, S8,
  mapback, graft) and the auxiliary parameters (AdamW).  The model is a
  GPT-shaped set of Linears whose forward hands on a recorded output, so that
  the pass is the optimizer's own work and not the model's matrix products.
* ``mlp``: a training step of one transformer MLP under bf16 autocast with the
  statistics fused into its passes: forward, backward, ``step()``.
* ``s8``: the stand-alone S8 polar map of a batch of matrices.
* ``direction``: the module-level helpers composed to one update direction:
  inverse square roots, rank-one whitening, S8, mapback, graft.

Every quantity is drawn on the GPU from the seed.
"""
from __future__ import annotations

import math

import torch
from torch import nn
from torch.nn import functional as F

from sandmuon_amd import DiagonalWeightedPE, RankOneAWeightedPE
from sandmuon_amd import optimizer as smx
from sandmuon_amd.fused import fuse_statistics

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
LR = 1e-2


# ------------------------------------------------------------------ cases ---
def _step(layers, width, mlp, vocab, ctx, rows, micro=1, variant="rank1", mode="comp_bf16", dtype="f32", name=None):
    case = dict(kind="step", layers=layers, width=width, mlp=mlp, vocab=vocab, ctx=ctx, rows=rows, micro=micro,
                variant=variant, mode=mode, dtype=dtype)
    return dict(case, name=name) if name else case


def _mlp(width, mlp, batch, seq, name=None):
    case = dict(kind="mlp", width=width, mlp=mlp, batch=batch, seq=seq)
    return dict(case, name=name) if name else case


def _s8(batch, rows, cols, mode, name=None):
    case = dict(kind="s8", batch=batch, rows=rows, cols=cols, mode=mode)
    return dict(case, name=name) if name else case


def _direction(batch, rows, cols, mode, name=None):
    case = dict(kind="direction", batch=batch, rows=rows, cols=cols, mode=mode)
    return dict(case, name=name) if name else case


def listed():
    return [
        # The smallest model of the tests (2 blocks, width 32): a unit test's
        # or a toy run's step, all latency and launches.
        _step(2, 32, 128, 97, 16, rows=64, name="step_tiny"),
        # A single 768 x 768 Linear (layers = 0) with four fp32 microbatches
        # of 16 x 1024 rows: one layer tried by itself.
        _step(0, 768, 768, 0, 0, rows=16384, micro=4, name="step_one_linear"),
        # The 103M GPT (54 matrices, 39.5M auxiliary parameters) after a
        # microbatch of 16 x 1024 tokens: the production run's step.
        _step(9, 768, 3072, 50257, 1024, rows=16384, name="step_gpt103m"),
        # Two blocks of the 2048-wide GPT after a microbatch of 8 x 1024
        # tokens: the large matrices, in the mixed mode.
        _step(2, 2048, 8192, 50257, 1024, rows=8192, mode="mixed", name="step_gpt2048_mixed"),
        # The parity mode (FP32 products) on three 768-wide blocks.
        _step(3, 768, 3072, 4096, 1024, rows=4096, mode="fp32", name="step_fp32"),
        # A small 16-bit model with sizes no tile divides and the diagonal
        # variant: width 400, MLP 1608, bf16 parameters and gradients.
        _step(6, 400, 1608, 5003, 256, rows=2048, variant="diagonal", dtype="bf16", name="step_ragged_bf16"),
        # A training step of the 103M GPT's MLP, statistics fused.
        _mlp(768, 3072, 16, 1024, name="mlp_fused"),
        # The S8 map by itself, at its default mode (fp32): the 36 square
        # matrices of the isolated workload, a wide batch in the compensated
        # mode, and many small ragged ones.
        _s8(36, 768, 768, "fp32", name="s8_square_fp32"),
        _s8(9, 3072, 768, "comp_bf16", name="s8_tall_comp"),
        _s8(24, 72, 200, "fp32", name="s8_small_fp32"),
        # One matrix at a time, as an interactive check or a per-layer
        # analysis calls it, and a direction built from the helpers.
        _s8(1, 512, 512, "comp_bf16", name="s8_single"),
        _direction(4, 640, 1280, "comp_bf16", name="direction"),
    ]


def _log_int(rng, lo, hi, multiple=1):
    return max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / multiple)) * multiple)


def _cost(case):
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / 2e14


def draw(rng):
    """A case of the listed ranges: sizes over their logarithm, every third or
    so with no common factor, none dearer than the largest listed one."""
    top = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["step", "step", "step", "mlp", "s8", "s8", "direction"])
        multiple = rng.choice([1, 8, 8, 64])
        mode = rng.choice(["comp_bf16", "comp_bf16", "fp32", "mixed"])
        if kind == "step":
            width = _log_int(rng, 24, 2048, multiple)
            mlp = max(1, int(width * rng.choice([2, 8 / 3, 4])))
            case = _step(rng.choice([1, 2, 3, 4, 6, 9]), width, mlp, _log_int(rng, 64, 50257), _log_int(rng, 16, 1024),
                         rows=_log_int(rng, 64, 16384), micro=rng.choice([1, 1, 2, 4]),
                         variant=rng.choice(["rank1", "rank1", "diagonal"]), mode=mode,
                         dtype=rng.choice(["f32", "f32", "bf16", "f16"]))
        elif kind == "mlp":
            width = _log_int(rng, 64, 1024, max(8, multiple))
            case = _mlp(width, 4 * width, rng.choice([1, 2, 4, 8, 16]), _log_int(rng, 64, 1024, 8))
        elif kind == "s8":
            case = _s8(_log_int(rng, 1, 64), _log_int(rng, 8, 3072, multiple), _log_int(rng, 8, 3072, multiple), mode)
        else:
            case = _direction(_log_int(rng, 1, 16), _log_int(rng, 8, 2048, multiple),
                              _log_int(rng, 8, 2048, multiple), mode)
        if _cost(case) <= top:
            return case


# ------------------------------------------------------- the recorded model ---
class _Recorded(torch.autograd.Function):
    """An output of the recorded shape and dtype; its backward hands nothing
    on (the gradients of the parameters are recorded too)."""

    @staticmethod
    def forward(ctx, weight, delta):
        return delta.new_zeros(1).expand(delta.shape)

    @staticmethod
    def backward(ctx, grad):
        return None, None


class RecordedLinear(nn.Linear):
    """An nn.Linear whose forward is a recorded one: it takes its input and
    gives an output whose cotangent the program then supplies."""

    delta = None

    def forward(self, x):
        return _Recorded.apply(self.weight, self.delta)


class _Attention(nn.Module):
    def __init__(self, w):
        super().__init__()
        self.q_proj, self.k_proj, self.v_proj, self.c_proj = (RecordedLinear(w, w) for _ in range(4))


class _Mlp(nn.Module):
    def __init__(self, w, m):
        super().__init__()
        self.c_fc, self.c_proj = RecordedLinear(w, m), RecordedLinear(m, w)


class _Block(nn.Module):
    def __init__(self, w, m):
        super().__init__()
        self.ln_1, self.attn, self.ln_2, self.mlp = nn.LayerNorm(w), _Attention(w), nn.LayerNorm(w), _Mlp(w, m)


def _model(case):
    w = case["width"]
    if case["layers"] == 0:
        return nn.Sequential(RecordedLinear(w, case["mlp"]))
    return nn.ModuleDict(dict(transformer=nn.ModuleDict(dict(
        wte=nn.Embedding(case["vocab"], w), wpe=nn.Embedding(case["ctx"], w),
        h=nn.ModuleList([_Block(w, case["mlp"]) for _ in range(case["layers"])]), ln_f=nn.LayerNorm(w)))))


def _flatten(parameters, dtype):
    """One buffer with the parameters as views of it (each on a 16-byte boundary)."""
    sizes = [-(-p.numel() // 8) * 8 for p in parameters]
    flat = torch.zeros(sum(sizes), dtype=dtype, device=DEVICE)
    at = 0
    for p, n in zip(parameters, sizes):
        p.data = flat[at:at + p.numel()].view(p.shape)
        at += n
    return flat


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _activation(g, rows, cols, dtype):
    """Per-channel offsets and scales a decade apart, as the layers of a GPT have them."""
    mu = torch.randn(cols, generator=g, device=DEVICE) * 0.3
    sigma = torch.exp(torch.empty(cols, device=DEVICE).uniform_(math.log(0.3), math.log(3.0), generator=g))
    return (torch.randn(rows, cols, generator=g, device=DEVICE) * sigma + mu).to(dtype)


def _cotangent(g, rows, cols, dtype):
    sigma = torch.exp(torch.empty(cols, device=DEVICE).uniform_(math.log(0.3), math.log(3.0), generator=g))
    return (torch.randn(rows, cols, generator=g, device=DEVICE) * (1e-3 * sigma)).to(dtype)


class _Call:
    """One hooked Linear of a microbatch: its module, input and cotangent."""

    __slots__ = ("module", "x", "delta")

    def __init__(self, module, x, delta):
        self.module, self.x, self.delta = module, x, delta


def _recorded(case, seed):
    """The model, its gradients and the recorded microbatches."""
    g = _generator(seed)
    low = DTYPES[case["dtype"]]
    with torch.device(DEVICE):
        model = _model(case)
    linears = [m for m in model.modules() if isinstance(m, RecordedLinear)]
    matrices = [m.weight for m in linears]
    ids = {id(p) for p in matrices}
    rest = [p for p in model.parameters() if id(p) not in ids]
    flat_m, flat_r = _flatten(matrices, low), _flatten(rest, low)
    for p in matrices + rest:
        scale = 0.02 if p.ndim == 2 else 0.0
        p.data.copy_(torch.randn(p.shape, generator=g, device=DEVICE) * scale + (0.0 if p.ndim == 2 else 0.1))
        p.grad = (torch.randn(p.shape, generator=g, device=DEVICE) * 1e-3).to(low)
    # What autocast hands the hooks: LayerNorm outputs stay fp32, the outputs
    # of attention and GELU and every cotangent are bf16; a 16-bit model's
    # are of its own dtype.
    ln, act, cot = (torch.float32, torch.bfloat16, torch.bfloat16) if low == torch.float32 else (low, low, low)
    if case["layers"] == 0:
        ln = cot = low
    micro = []
    for _ in range(case["micro"]):
        calls, r, w, m = [], case["rows"], case["width"], case["mlp"]
        if case["layers"] == 0:
            calls.append(_Call(linears[0], _activation(g, r, w, ln), _cotangent(g, r, m, cot)))
        else:
            for block in model["transformer"]["h"]:
                x = _activation(g, r, w, ln)
                for lin in (block.attn.q_proj, block.attn.k_proj, block.attn.v_proj):
                    calls.append(_Call(lin, x, _cotangent(g, r, w, cot)))
                calls.append(_Call(block.attn.c_proj, _activation(g, r, w, act), _cotangent(g, r, w, cot)))
                calls.append(_Call(block.mlp.c_fc, _activation(g, r, w, ln), _cotangent(g, r, m, cot)))
                calls.append(_Call(block.mlp.c_proj, _activation(g, r, m, act), _cotangent(g, r, w, cot)))
        micro.append(calls)
    return model, linears, matrices, rest, flat_m, flat_r, micro


# ---------------------------------------------------------------- prepare ---
def _matrices(case, seed):
    """Gaussian matrices with diagonal row and column scales a decade each way."""
    g = _generator(seed)
    b, r, c = case["batch"], case["rows"], case["cols"]
    x = torch.randn(b, r, c, generator=g, device=DEVICE)
    scale = lambda *s: torch.exp(torch.empty(*s, device=DEVICE).uniform_(-2.3, 2.3, generator=g))
    return x * scale(b, r, 1) * scale(b, 1, c), g


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        model, linears, matrices, rest, flat_m, flat_r, micro = _recorded(case, seed)
        new = RankOneAWeightedPE if case["variant"] == "rank1" else DiagonalWeightedPE
        opt = new(model, LR, s8_mode=case["mode"])
        return dict(case=case, model=model, opt=opt, linears=linears, flat=(flat_m, flat_r), micro=micro)
    if kind == "mlp":
        g = _generator(seed)
        w, m = case["width"], case["mlp"]
        with torch.device(DEVICE):
            model = _GeluMlp(w, m)
        for p in model.parameters():
            p.data.copy_(torch.randn(p.shape, generator=g, device=DEVICE) * (0.02 if p.ndim == 2 else 0.01))
        x = torch.randn(case["batch"], case["seq"], w, generator=g, device=DEVICE).requires_grad_()
        dy = (torch.randn(case["batch"], case["seq"], w, generator=g, device=DEVICE) * 1e-3).bfloat16()
        opt = RankOneAWeightedPE(model, LR)
        fused = fuse_statistics(opt, model)
        return dict(case=case, model=model, opt=opt, fused=fused, x=x, dy=dy)
    x, g = _matrices(case, seed)
    state = dict(case=case, x=x)
    if kind == "direction":
        r, c = case["rows"], case["cols"]
        rows = _activation(g, 256, r, torch.float32)
        cols = _activation(g, 256, c, torch.float32)
        state["left"] = (rows * rows).mean(0), rows.mean(0)
        state["right"] = (cols * cols).mean(0), cols.mean(0)
    return state


class _GeluMlp(nn.Module):
    def __init__(self, w, m):
        super().__init__()
        self.c_fc, self.c_proj = nn.Linear(w, m), nn.Linear(m, w)

    def forward(self, x):
        return self.c_proj(F.gelu(self.c_fc(x)))


# -------------------------------------------------------------------- run ---
def _state_outputs(opt, parameter):
    """A matrix's updated optimizer state."""
    st = opt.state[parameter]
    return {k: st[k] for k in ("momentum_buffer", "a_ema", "a_mean_ema", "b_ema") if k in st}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        opt = state["opt"]
        for calls in state["micro"]:
            outputs = []
            for call in calls:
                call.module.delta = call.delta
                outputs.append(call.module(call.x))
            torch.autograd.backward(outputs, [call.delta for call in calls])
        opt.step()
        # The updated parameters, and the optimizer state of the last block's
        # matrices (of the one matrix where there is no block).
        return {"matrices": state["flat"][0], "rest": state["flat"][1],
                "state": [_state_outputs(opt, lin.weight) for lin in state["linears"][-6:]]}
    if kind == "mlp":
        model, opt, x = state["model"], state["opt"], state["x"]
        opt.zero_grad(set_to_none=True)
        x.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = model(x)
        y.backward(state["dy"])
        opt.step()
        linears = (model.c_fc, model.c_proj)
        return {"y": y.detach(), "dx": x.grad, "grads": [p.grad for lin in linears for p in (lin.weight, lin.bias)],
                "weights": [p.detach() for lin in linears for p in (lin.weight, lin.bias)],
                "state": [_state_outputs(opt, lin.weight) for lin in linears]}
    if kind == "s8":
        return smx._s8_fp32(state["x"], case["mode"])
    left = smx.rank1_inverse_sqrt(*state["left"])
    right = smx.rank1_inverse_sqrt(*state["right"])
    white = smx.rank1_whiten(state["x"], left, right)
    polar = smx._s8_fp32(white, case["mode"])
    mapped = smx.rank1_mapback(polar, left, right)
    return {"white": white, "mapped": mapped, "direction": smx._graft_direction(mapped, case["rows"])}


# ------------------------------------------------------------------- work ---
def _shapes(case):
    w, m = case["width"], case["mlp"]
    if case["layers"] == 0:
        return [(m, w)]
    return [(w, w)] * 4 * case["layers"] + [(m, w), (w, m)] * case["layers"]


def _s8_flops(rows, cols):
    """Five stages on r x c (r <= c): a symmetric Gram and square (half of
    each) and an apply, or, for a wide matrix, the same polynomials by
    products of r x r matrices between two Grams and two applies."""
    r, c = sorted((rows, cols))
    return min(5 * (3.0 * r * r * c + r ** 3), 6.0 * r * r * c + 17.0 * r ** 3)


def work(case):
    if case["kind"] == "step":
        e = DTYPES[case["dtype"]].itemsize
        w, m, rows = case["width"], case["mlp"], case["rows"]
        if case["layers"] == 0:
            seen = rows * (w + m) * e
            rest = m
        else:
            ln, low = (4, 2) if e == 4 else (e, e)
            seen = case["layers"] * rows * (2 * w * ln + (w + m) * low + (5 * w + m) * low)
            rest = (case["vocab"] + case["ctx"] + 2) * w + case["layers"] * (9 * w + m)
        n = sum(r * c for r, c in _shapes(case))
        # matrices: gradient read, momentum and parameter read and written;
        # the rest: gradient read, two moments and parameter read and written
        return dict(bytes=case["micro"] * seen + n * (3 * e + 8) + rest * (3 * e + 16),
                    flops=sum(_s8_flops(r, c) for r, c in _shapes(case)))
    if case["kind"] == "mlp":
        w, m, rows = case["width"], case["mlp"], case["batch"] * case["seq"]
        n = 2 * w * m
        # x, dx in fp32, y and dy in bf16, and the hidden layer before and
        # after the GELU and its cotangents in bf16, each written and read;
        # the weights as in a step, their gradients written and read
        return dict(bytes=rows * (8 * w + 4 * w + 16 * m) + n * 28, flops=6.0 * rows * n + 2 * _s8_flops(w, m))
    b, r, c = case["batch"], case["rows"], case["cols"]
    if case["kind"] == "s8":
        return dict(bytes=8 * b * r * c, flops=b * _s8_flops(r, c))
    return dict(bytes=16 * b * r * c, flops=b * (_s8_flops(r, c) + 16.0 * r * c))


# -------------------------------------------------------------- tolerance ---
def tolerance(case):
    mode = case.get("mode", "comp_bf16")
    if case["kind"] == "step":
        if case["dtype"] != "f32":
            # a weight's last place: 2^-9 (bf16) or 2^-12 (f16) of it, in the
            # few whose sum lands on the other side of a rounding boundary
            return dict(rel=4e-4 if case["dtype"] == "bf16" else 1e-4, max=0.01 if case["dtype"] == "bf16" else 0.002)
        # the direction's error (below) in a weight that it changes by 2-10%
        return dict(rel={"comp_bf16": 8e-5, "mixed": 3e-4, "fp32": 4e-6}[mode])
    if case["kind"] == "mlp":
        return dict(rel=4e-3, max=0.1)  # bf16 activations and their gradients
    # four times the error against 64 bits on such matrices
    return dict(rel={"comp_bf16": 1.2e-3, "mixed": 8e-3, "fp32": 6e-5}[mode])


# ------------------------------------------------------------------ exact ---
_S8 = ((11.062126275847973, -56.051653229128085, 72.32081107619855),
       (4.100720073616268, -2.9324183165353577, 0.5339692084282731),
       (3.930310192522361, -2.873509793709714, 0.5366557527206212),
       (3.280567968245866, -2.414925589994015, 0.48635134757825227),
       (2.282741575232451, -1.6302296637355072, 0.40275720810675486))
_MARGIN = 1.35


def _polar64(x):
    """The five-stage map of a batch in 64 bits."""
    x = x.double()
    flip = x.shape[-2] > x.shape[-1]
    if flip:
        x = x.transpose(-2, -1).contiguous()
    x = x / torch.linalg.matrix_norm(x, keepdim=True)
    eye = torch.eye(x.shape[-2], dtype=x.dtype, device=x.device)
    for k, (a, b, c) in enumerate(_S8):
        g = x @ x.transpose(-2, -1).contiguous()
        g2 = g @ g
        s = _MARGIN * torch.linalg.matrix_norm(g2, keepdim=True) ** 0.25 if k == 0 else torch.ones_like(g2[..., :1, :1])
        x = (a * eye + b * g / s ** 2 + c * g2 / s ** 4) @ x / s
    return x.transpose(-2, -1) if flip else x


def _diagonal64(v):
    m = v.mean()
    return torch.rsqrt(torch.clamp(torch.maximum(v, m * 1e-6) / m, min=1e-6))


def _rank_one64(second, mean):
    q = second.mean()
    inv = torch.rsqrt(torch.clamp(torch.clamp(second - mean * mean, min=0.0) / q, min=1e-6))
    z = inv * (mean / torch.sqrt(q))
    rho = torch.sqrt(1 + (z * z).sum())
    return inv, z, -1 / (rho * (rho + 1))


def _whiten64(x, left, right):
    (li, lz, lc), (ri, rz, rc) = left, right
    v = x.double() * li[:, None] * ri
    v = v + lc * lz[:, None] * (lz[None, :] @ v)
    return v + rc * (v @ rz[:, None]) * rz


def _mapback64(v, left, right):
    (li, lz, lc), (ri, rz, rc) = left, right
    v = v + lc * lz[:, None] * (lz[None, :] @ v)
    v = v + rc * (v @ rz[:, None]) * rz
    return v * li[:, None] * ri


def _exact_step(case, seed):
    model, linears, matrices, rest, flat_m, flat_r, micro = _recorded(case, seed)
    out_m, out_r = flat_m.double(), flat_r.double()
    view = lambda flat, out, p: out[p.storage_offset():p.storage_offset() + p.numel()].view(p.shape)
    stats = {}
    for calls in micro:
        for call in calls:
            x, d = call.x.double(), call.delta.double()
            st = stats.setdefault(id(call.module), [0, 0, 0, 0])
            st[0] = st[0] + (x * x).sum(0)
            st[1] = st[1] + x.sum(0)
            st[2] = st[2] + (d * d).sum(0)
            st[3] += x.shape[0]
            del x, d
    state = []
    for lin in linears:
        sq, first, b, n = stats[id(lin)]
        second, mean = sq / n, first / n
        b_ema = b / n / (b / n).mean()
        p = lin.weight
        out, inp = p.shape
        zero = torch.zeros(out, dtype=torch.float64, device=p.device)
        one = torch.zeros((), dtype=torch.float64, device=p.device)
        left = _diagonal64(b_ema), zero, one
        if case["variant"] == "rank1":
            right = _rank_one64(second, mean)
        else:
            right = _diagonal64(second), torch.zeros_like(second), one
        grad = p.grad.double()
        momentum = grad * (1 - .8)  # the first step's
        source = momentum * .8 + grad * (1 - .8)
        u = _mapback64(_polar64(_whiten64(source, left, right)), left, right)
        view(flat_m, out_m, p).sub_(u * (LR * math.sqrt(out) / torch.linalg.vector_norm(u)))
        shared = "transformer" in model and any(lin is m for blk in model["transformer"]["h"]
                                                for m in (blk.attn.k_proj, blk.attn.v_proj))
        entry = {"momentum_buffer": momentum, "b_ema": b_ema}
        if not shared:
            entry["a_ema"] = second
            if case["variant"] == "rank1":
                entry["a_mean_ema"] = mean
        state.append(entry)
    lr = LR * .1
    for p in rest:
        gr = p.grad.double()
        w = view(flat_r, out_r, p)
        w.mul_(1 - lr * .01)
        w.sub_(lr * gr / (gr.abs() + 1e-8))  # the first step's moments, bias-corrected
    return {"matrices": out_m, "rest": out_r, "state": state[-6:]}


def _gelu64(h):
    return 0.5 * h * (1 + torch.erf(h / math.sqrt(2.0)))


def exact(case, seed):
    """``run``'s outputs in 64 bits, on the first pass of a new state."""
    with torch.no_grad():
        if case["kind"] == "step":
            return _exact_step(case, seed)
        if case["kind"] == "s8":
            return _polar64(_matrices(case, seed)[0])
        if case["kind"] == "direction":
            x, g = _matrices(case, seed)
            rows = _activation(g, 256, case["rows"], torch.float32)
            cols = _activation(g, 256, case["cols"], torch.float32)
            left = _rank_one64((rows * rows).mean(0).double(), rows.mean(0).double())
            right = _rank_one64((cols * cols).mean(0).double(), cols.mean(0).double())
            white = _whiten64(x, left, right)
            mapped = _mapback64(_polar64(white), left, right)
            return {"white": white, "mapped": mapped,
                    "direction": mapped * (math.sqrt(case["rows"]) / torch.linalg.vector_norm(mapped))}
        # The MLP: its forward and backward on the weights and inputs as bf16
        # holds them.  The update directions of step() come out of gradients
        # that bf16 has rounded and have no value of their own.
        g = _generator(seed)
        w, m = case["width"], case["mlp"]
        rnd = lambda *s: torch.randn(*s, generator=g, device=DEVICE)
        low = lambda t: t.bfloat16().double()
        w1, b1, w2, b2 = rnd(m, w) * 0.02, rnd(m) * 0.01, rnd(w, m) * 0.02, rnd(w) * 0.01
        x = rnd(case["batch"], case["seq"], w)
        dy = (rnd(case["batch"], case["seq"], w) * 1e-3).bfloat16().double()
        xl, w1l, w2l = low(x), low(w1), low(w2)
        h = xl @ w1l.t() + low(b1)
        a = _gelu64(h)
        y = a @ w2l.t() + low(b2)
        da = dy @ w2l
        pdf = torch.exp(-0.5 * h * h) / math.sqrt(2 * math.pi)
        dh = da * (0.5 * (1 + torch.erf(h / math.sqrt(2.0))) + h * pdf)
        flat = lambda t: t.reshape(-1, t.shape[-1])
        a_ema = [flat(x.double()), flat(a)]
        b_sum = [(flat(dh) ** 2).mean(0), (flat(dy) ** 2).mean(0)]
        return {"y": y, "dx": dh @ w1l,
                "grads": [flat(dh).t().contiguous() @ flat(xl), flat(dh).sum(0),
                          flat(dy).t().contiguous() @ flat(a), flat(dy).sum(0)],
                "weights": [None] * 4,
                "state": [{"momentum_buffer": None, "a_ema": (t * t).mean(0), "a_mean_ema": t.mean(0),
                           "b_ema": b / b.mean()} for t, b in zip(a_ema, b_sum)]}
