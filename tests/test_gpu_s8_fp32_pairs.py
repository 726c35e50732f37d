"""The fp32 mode: FP16 pairs, and FP32 MFMAs for matrices whose rows, columns
or blocks lie far apart in scale; accuracy against the FP64 map and range.

A pair carries 22 significant bits and every product FP32 accumulation, so
the map's error is that of FP32 GEMMs: a few 1e-6 on scaled Gaussian
matrices, up to 1e-4 on steep spectra at 2048, where FP32 operands on FP32
MFMAs measured 4e-6 to 1.1e-5 and 1.5e-4.  The bounds are about three times
the pairs' own measurements."""
import math

import pytest
import torch

from oracle import sandmuon_oracle as O
from sandmuon_amd import _native
from sandmuon_amd.optimizer import _s8_fp32

pytestmark = pytest.mark.gpu


def _input(shape, kind, seed):
    g = torch.Generator().manual_seed(seed)
    b, r, c = shape
    if kind == "scaled":
        f = lambda *s: torch.exp(torch.empty(*s).uniform_(-2.3, 2.3, generator=g))
        return torch.randn(shape, generator=g) * f(b, r, 1) * f(b, 1, c)
    n = min(r, c)
    u = torch.linalg.qr(torch.randn(b, r, n, generator=g, dtype=torch.float64))[0]
    v = torch.linalg.qr(torch.randn(b, c, n, generator=g, dtype=torch.float64))[0]
    return ((u * torch.arange(1, n + 1, dtype=torch.float64) ** -2) @ v.transpose(1, 2)).float()


# X-space and Gram space, transposed, around the padding of 256
@pytest.mark.parametrize("shape", [(2, 33, 40), (3, 129, 140), (2, 256, 256), (1, 257, 600), (2, 520, 300),
                                   (1, 768, 768)])
@pytest.mark.parametrize("kind,tol", [("scaled", 3e-5), ("steep", 1e-4)])
def test_fp32_mode_against_fp64(device, shape, kind, tol):
    x = _input(shape, kind, sum(shape))
    want = O.s8(x.double())
    got = _s8_fp32(x.to(device)).cpu().double()
    err = ((got - want).flatten(1).norm(dim=1) / want.flatten(1).norm(dim=1)).max().item()
    print(f"{kind} {shape}: {err:.2e}")
    assert err <= tol


# Gaussian matrices with row and column scales a decade each way, against the
# error of FP32 MFMAs on FP32 operands on such matrices (their mean over
# seeds): alone and in a batch of 128 x 128 tiles, Gram space, few rows
@pytest.mark.parametrize("shape,fp32", [((1, 768, 768), 4.5e-6), ((30, 768, 768), 4.5e-6), ((3, 640, 1280), 1.0e-5),
                                        ((3, 64, 3000), 6.9e-6), ((3, 128, 600), 5.7e-6), ((2, 192, 1200), 5.6e-6)])
def test_fp32_mode_is_no_further_from_fp64_than_fp32_mfmas(device, shape, fp32):
    err = 0.0
    for seed in range(4):
        g = torch.Generator(device=device).manual_seed(seed)
        f = lambda *s: torch.exp(torch.empty(*s, device=device).uniform_(-2.3, 2.3, generator=g))
        x = torch.randn(shape, generator=g, device=device) * f(*shape[:2], 1) * f(shape[0], 1, shape[2])
        want = O.s8(x[:3].double().cpu())
        err += ((_s8_fp32(x)[:3].double().cpu() - want).norm() / want.norm()).item() / 4
    assert err <= fp32


@pytest.mark.parametrize("shape", [(2, 130, 150), (2, 90, 700)])
@pytest.mark.parametrize("k", [-60, -20, 30, 55])
def test_fp32_mode_ignores_powers_of_two(device, shape, k):
    # The input's exponent is folded into the scales exactly.
    x = _input(shape, "scaled", 5).to(device)
    assert torch.equal(_s8_fp32(x * math.ldexp(1.0, k)), _s8_fp32(x))


# One block, X-space, Gram space and transposed, the classes of few rows.  FP32
# MFMAs measured 3e-6 at every scale: each product carries 2^-24 of itself,
# and every term of a scaled row, column or block has its scale.  (2^-11:
# still pairs, 2^-39 of the operand's scale in every element.)
@pytest.mark.parametrize("shape", [(40, 60), (256, 256), (300, 280), (200, 700), (700, 200), (90, 600), (20, 2400)])
@pytest.mark.parametrize("scale", [2 ** -11, 2 ** -13, 1e-6, 1e-9, 1e-12, 1e-18])
def test_fp32_mode_keeps_small_rows_columns_and_blocks(device, shape, scale):
    x = torch.randn(3, *shape, generator=torch.Generator().manual_seed(sum(shape)))
    h, w = shape[0] // 2, shape[1] // 2
    x[0, 5] *= scale
    x[1, :, 9] *= scale
    x[2, :h, w:] *= scale
    x[2, h:, :w] *= scale
    want = O.s8(x.double())
    got = _s8_fp32(x.to(device)).cpu().double()
    # (a block's coupling passes through three products with it)
    for a, b, tol in ((got[0, 5], want[0, 5], 2e-5), (got[1, :, 9], want[1, :, 9], 2e-5),
                      (got[2, :h, w:], want[2, :h, w:], 2e-4), (got[2, h:, :w], want[2, h:, :w], 2e-4)):
        assert ((a - b).norm() / b.norm()).item() <= tol


@pytest.mark.parametrize("shape", [(300, 280), (200, 700), (700, 300)])
def test_fp32_mode_wide_matrices_in_a_batch(device, shape):
    """Each matrix has the bits it has alone, in every geometry."""
    x = torch.randn(12, *shape, generator=torch.Generator().manual_seed(sum(shape)))
    x[1::2, 7] *= 1e-7
    x = x.to(device)
    out = _s8_fp32(x)
    for policy in (0, 2):
        prev = _native.s8_tile_geometry(policy)
        try:
            for i in range(4):
                assert torch.equal(out[i], _s8_fp32(x[i]))
        finally:
            _native.s8_tile_geometry(prev)


def test_fp32_arithmetic_does_not_depend_on_a_narrow_neighbour(device):
    """A 16 x 2304 matrix, too wide for one block, beside a 768 x 768 one."""
    def step(shapes):
        g = torch.Generator().manual_seed(7)
        descs, keep = [], []
        for r, c in shapes:
            t = lambda *s: torch.randn(*s, generator=g).to(device)
            w, gr, m = t(r, c) * .02, t(r, c), torch.zeros(r, c, device=device)
            ir, ic = t(r).abs() + .5, t(c).abs() + .5
            keep.append((w.clone(), w, gr, m, ir, ic))
            descs.append(_native.MatrixDesc(
                param=w.data_ptr(), grad=gr.data_ptr(), momentum=m.data_ptr(), inv_row=ir.data_ptr(),
                inv_col=ic.data_ptr(), rows=r, cols=c, lr=1e-2, momentum_beta=.8))
        ws = torch.empty(_native.matrix_step_workspace_bytes(shapes, 0), dtype=torch.uint8, device=device)
        _native.matrix_step(descs, 0, ws)
        torch.cuda.synchronize()
        return keep

    alone, both = step([(768, 768)]), step([(768, 768), (16, 2304)])
    assert torch.equal(alone[0][1], both[0][1])
    for w0, w, gr, _, ir, ic in both:
        v = O.s8((gr.double() * ir.double()[:, None] * ic.double()).cpu()[None])[0].to(device)
        u = v * ir.double()[:, None] * ic.double()
        u *= 1e-2 * math.sqrt(w.shape[0]) / u.norm()
        assert ((w0.double() - w.double() - u).norm() / u.norm()).item() <= 1e-4


def test_fp32_mma_classes_record_one_product(device):
    """A class on FP32 MFMAs as a whole (16 x 2304 here) runs in launches of its
    own, one product per K: two Grams (Gram space: stages 1 and 3) of the upper
    triangle of 256 x 256 in 128 x 128 tiles or their quadrants."""
    _native.s8_timing(True)
    try:
        _s8_fp32(torch.randn(2, 16, 2304, device=device))
    finally:
        _native.s8_timing(False)
    grams = [f for _, p, f in _native.s8_timing_read() if p == "gram"]
    assert grams == [2 * 3 * 128 * 128 * 2 * 2304.0] * 2


def test_fp32_mode_keeps_non_finite_inputs_visible(device):
    x = torch.randn(2, 40, 50, device=device)
    x[1, 3, 4] = float("inf")
    out = _s8_fp32(x)
    assert torch.isfinite(out[0]).all() and not torch.isfinite(out[1]).all()
