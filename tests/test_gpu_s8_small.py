"""Small matrices, whose S8 map runs whole in one block: at the edges of its
16-row tiles, its Gram split over waves (1 to 8 row tiles), its two LDS sizes
and the largest iterate that fits, against FP64.  Every product is FP32
whatever the mode (comp_bf16 and mixed round the input to BF16 hi + lo, 2^-17
of an element, first): some 1e-5 on these inputs, a third of the bound."""
import math

import pytest
import torch

from oracle import sandmuon_oracle as O
from sandmuon_amd import _native
from sandmuon_amd.optimizer import _s8_fp32

pytestmark = pytest.mark.gpu


def _small_ran(fn):
    _native.s8_timing(True)
    try:
        out = fn()
    finally:
        _native.s8_timing(False)
    return out, [p for _, p, _ in _native.s8_timing_read()] == ["run", "small"]


@pytest.mark.parametrize("mode", ["fp32", "comp_bf16", "mixed"])
@pytest.mark.parametrize("shape,small", [((1, 1, 1), True), ((2, 1, 9), True), ((3, 16, 16), True), ((2, 17, 40), True),
                                         ((70, 31, 33), True), ((2, 48, 300), True), ((2, 200, 64), True),
                                         ((1, 80, 320), True), ((1, 96, 250), True), ((2, 112, 113), True),
                                         ((2, 128, 128), True), ((1, 16, 2240), True), ((1, 16, 2241), False),
                                         ((1, 129, 129), False)])
def test_small_matrices(device, mode, shape, small):
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(shape, generator=g)
    out, ran = _small_ran(lambda: _s8_fp32(x.to(device), mode=mode).cpu())
    assert ran == small, "the rule for small matrices moved"
    want = O.s8(x.double())
    tol = 4e-5 if small else {"fp32": 1e-4, "comp_bf16": 1e-2, "mixed": 1e-2}[mode]
    assert ((out.double() - want).flatten(1).norm(dim=1) <= tol * want.flatten(1).norm(dim=1)).all()


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_small_and_large_classes_in_one_matrix_step(device, mode):
    """Small classes beside large ones, plain and transposed, with the
    rank-one term: their row sums and results reach the mapback as the chains'
    do (policy 2 runs every class in the chains)."""
    shapes = [(24, 40), (40, 24), (24, 40), (64, 200), (300, 180), (30, 1000), (16, 16), (400, 400)]

    def step(policy, dtype=torch.float32):
        g = torch.Generator().manual_seed(11)
        prev = _native.s8_tile_geometry(policy)
        try:
            descs, keep, out = [], [], []
            for r, c in shapes:
                t = lambda *s: torch.randn(*s, generator=g).to(device)
                w, gr, m = (t(r, c) * .02).to(dtype), t(r, c), t(r, c) * .1
                ir, ic, z = t(r).abs() + .5, t(c).abs() + .5, t(c) * .3
                ka = torch.tensor([-1 / (2 + math.sqrt(2))], device=device)
                keep += [gr, m, ir, ic, z, ka]
                out.append((w.clone(), w))
                descs.append(_native.MatrixDesc(
                    param=w.data_ptr(), grad=gr.data_ptr(), momentum=m.data_ptr(), inv_row=ir.data_ptr(),
                    inv_col=ic.data_ptr(), z=z.data_ptr(), kappa=ka.data_ptr(), rows=r, cols=c, lr=1e-2,
                    momentum_beta=.8, param_dtype=_native.dtype_code(dtype)))
            ws = torch.empty(_native.matrix_step_workspace_bytes(shapes, mode), dtype=torch.uint8, device=device)
            _native.matrix_step(descs, mode, ws)
            torch.cuda.synchronize()
        finally:
            _native.s8_tile_geometry(prev)
        return [(a.double() - b.double()) / 1e-2 for a, b in out]

    for a, b, (r, _) in zip(step(0), step(2), shapes):
        assert (a - b).norm() <= {0: 4e-5, 1: 2e-3, 2: 8e-3}[mode] * b.norm()
        assert abs(a.norm().item() / math.sqrt(r) - 1) <= 1e-4
    # 16-bit parameters keep their bits
    for a, b in zip(step(0, torch.bfloat16), step(2, torch.bfloat16)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mixed_parameter_types_in_one_matrix_step(device, mode, dtype):
    """An FP32 parameter's update has the same bits beside 16-bit parameters of
    its shape and others, and a 16-bit one beside FP32 ones (7 shapes in both
    types: 14 classes, more than one group); the 16-bit update is the FP32
    one's, to the mode's rounding and its own."""
    shapes = [(24, 40), (96, 48), (300, 180), (180, 400), (260, 260), (64, 500)] * 2 + [(256, 256)] * 50

    def step(dtypes):
        g = torch.Generator().manual_seed(5)
        descs, keep, out = [], [], []
        for (r, c), dt in zip(shapes, dtypes):
            t = lambda *s: torch.randn(*s, generator=g).to(device)
            w = (t(r, c) * .02).to(dtype).to(dt)  # the same values in either type
            gr, m, ir, ic = t(r, c), t(r, c) * .1, t(r).abs() + .5, t(c).abs() + .5
            keep += [gr, m, ir, ic]
            out.append((w, w.double()))
            descs.append(_native.MatrixDesc(
                param=w.data_ptr(), grad=gr.data_ptr(), momentum=m.data_ptr(), inv_row=ir.data_ptr(),
                inv_col=ic.data_ptr(), rows=r, cols=c, lr=1e-2, momentum_beta=.8, param_dtype=_native.dtype_code(dt)))
        ws = torch.empty(_native.matrix_step_workspace_bytes(shapes, mode), dtype=torch.uint8, device=device)
        _native.matrix_step(descs, mode, ws)
        torch.cuda.synchronize()
        return out

    def close(a, b, w0):
        # the update and the new weight each by half a last place of the type
        # (2^-8 or 2^-11 of the value at most; f16: 2^-25 below its normal
        # range), some FP32 roundings of both, which may cancel, and the map's
        # error in the mode
        half, least = (2 ** -8, 0.0) if dtype == torch.bfloat16 else (2 ** -11, 2 ** -25)
        u = (w0 - b).abs()
        bound = (b.abs() + u) * half + 2 * least + 2 ** -22 * b.abs().max()
        return ((a - b).abs() <= bound * (1 + half) + {0: 4e-5, 1: 2e-3, 2: 8e-3}[mode] * u.max()).all()

    n = len(shapes)
    low = [k % 2 == (k // 6) % 2 for k in range(n)]
    full, narrow = step([torch.float32] * n), step([dtype] * n)
    for (a, w0), (b, _) in zip(narrow, full):
        assert close(a.double(), b.double(), w0)
    for lo, (a, _), (b, _), (c, _) in zip(low, step([dtype if lo else torch.float32 for lo in low]), full, narrow):
        assert torch.equal(a, c if lo else b)
