"""The 64 x 64 tiles with K split over a block's waves, which short S8
launches take, against the other geometries (policy 2 never takes them nor
256 x 256) and FP64.  Both add the same products of the same operands, in
another order, so they agree to the mode's rounding of its operands: 2^-17
(comp_bf16), 2^-12 (mixed, stages 3-5 of square matrices) and 2^-22 (fp32),
each amplified some tenfold by the map's cancellations."""
import math

import pytest
import torch

from oracle import sandmuon_oracle as O
from sandmuon_amd import _native
from sandmuon_amd.optimizer import _s8_fp32

pytestmark = pytest.mark.gpu

AGREE = {"fp32": 2e-5, "comp_bf16": 1e-3, "mixed": 6e-3}


def _both(fn):
    out = []
    for policy in (0, 2):
        prev = _native.s8_tile_geometry(policy)
        try:
            out.append(fn())
        finally:
            _native.s8_tile_geometry(prev)
    return out


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


# K of 256, 512, 768 and 1280; one and several matrices, X-space, Gram space
# and transposed, sizes with padding; five run as two chains
@pytest.mark.parametrize("mode", ["fp32", "comp_bf16", "mixed"])
@pytest.mark.parametrize("shape", [(1, 256, 256), (3, 140, 250), (1, 500, 512), (5, 300, 260), (1, 400, 1200),
                                   (2, 1100, 200), (1, 768, 700)])
def test_split_tiles_agree(device, mode, shape):
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(shape, generator=g)
    a, b = _both(lambda: _s8_fp32(x.to(device), mode=mode).cpu())
    assert not torch.equal(a, b), "both policies ran the same geometry"
    assert _rel(a, b) <= AGREE[mode]
    assert _rel(a, O.s8(x.double())) <= {"fp32": 1e-4, "comp_bf16": 1e-2, "mixed": 1e-2}[mode]


@pytest.mark.parametrize("mode", ["fp32", "comp_bf16", "mixed"])
@pytest.mark.parametrize("rank1", [True, False])
@pytest.mark.parametrize("shape", [(256, 256), (300, 200), (200, 700), (700, 260)])
def test_split_tiles_in_the_matrix_step(device, mode, rank1, shape):
    """The stage-5 row sums (plain and transposed parameters).  A 16-bit
    parameter's step keeps its bits: no split tiles, no FP16 pairs."""
    rows, cols = shape
    g = torch.Generator().manual_seed(rows + 3 * cols)
    vec = lambda n: (torch.rand(n, generator=g) + .5).to(device)
    inv_row, inv_col = vec(rows), vec(cols)
    z = (torch.randn(cols, generator=g) * .3).to(device)
    kappa = torch.tensor([-1 / (2 + math.sqrt(2))], device=device)
    w0 = (torch.randn(rows, cols, generator=g) * .02).to(device)
    grad = torch.randn(rows, cols, generator=g).to(device)

    def step(dtype):
        w, m = w0.to(dtype, copy=True), torch.zeros(rows, cols, device=device)
        d = _native.MatrixDesc(param=w.data_ptr(), grad=grad.data_ptr(), momentum=m.data_ptr(),
                               inv_row=inv_row.data_ptr(), inv_col=inv_col.data_ptr(), rows=rows, cols=cols, lr=1e-2,
                               momentum_beta=.8, param_dtype=_native.dtype_code(dtype))
        if rank1:
            d.z, d.kappa = z.data_ptr(), kappa.data_ptr()
        code = _native.S8_MODES[mode]
        ws = torch.empty(_native.matrix_step_workspace_bytes([shape], code), dtype=torch.uint8, device=device)
        _native.matrix_step([d], code, ws)
        torch.cuda.synchronize()
        return w.float()

    a, b = _both(lambda: step(torch.float32))
    assert not torch.equal(a, b)
    assert _rel(w0 - a, w0 - b) <= AGREE[mode]
    assert abs(((w0 - a).double().norm() / 1e-2 / math.sqrt(rows)).item() - 1) <= 1e-4
    for dtype in (torch.bfloat16, torch.float16):
        a, b = _both(lambda: step(dtype))
        assert torch.equal(a, b)
