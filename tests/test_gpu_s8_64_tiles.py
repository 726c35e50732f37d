"""The 64 x 64 tiles that short S8 launches take: the bits of the 128 x 128
tiles (policy 2 never takes 64 x 64 nor 256 x 256 ones), so that a matrix's
result does not depend on what else is in its launch."""
import math

import pytest
import torch

from oracle import sandmuon_oracle as O
from sandmuon_amd import _native
from sandmuon_amd.optimizer import _s8_fp32

pytestmark = pytest.mark.gpu


def _both(fn):
    out, tiles = [], []
    for policy in (0, 2):
        prev = _native.s8_tile_geometry(policy)
        _native.s8_timing(True)
        try:
            out.append(fn())
        finally:
            _native.s8_timing(False)
            _native.s8_tile_geometry(prev)
        tiles.append({t[1:] for t in _native.s8_timing_tiles()})
    assert tiles == [{(64, 64)}, {(128, 128)}]
    return out


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


# K of 256, 512, 768 and 1280; one and several matrices, X-space, Gram space
# and transposed, sizes with padding; five run as two chains
@pytest.mark.parametrize("mode", ["fp32", "comp_bf16", "mixed"])
@pytest.mark.parametrize("shape", [(1, 256, 256), (3, 140, 250), (1, 500, 512), (5, 300, 260), (1, 400, 1200),
                                   (2, 1100, 200), (1, 768, 700)])
def test_64_tiles_have_the_bits_of_128_tiles(device, mode, shape):
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(shape, generator=g)
    a, b = _both(lambda: _s8_fp32(x.to(device), mode=mode).cpu())
    assert torch.equal(a, b)
    assert _rel(a, O.s8(x.double())) <= {"fp32": 1e-4, "comp_bf16": 1e-2, "mixed": 1e-2}[mode]


@pytest.mark.parametrize("mask", [0x03, 0x1a])
def test_64_tiles_in_plain_bf16_stages(device, mask):
    x = torch.randn(2, 300, 700, generator=torch.Generator().manual_seed(3)).to(device)
    prev = _native.s8_comp_mask(mask)
    try:
        a, b = _both(lambda: _s8_fp32(x, mode="comp_bf16"))
    finally:
        _native.s8_comp_mask(prev)
    assert torch.equal(a, b)


@pytest.mark.parametrize("mode", ["fp32", "comp_bf16", "mixed"])
@pytest.mark.parametrize("shape", [(42, 512, 512), (30, 768, 500), (28, 300, 900)])
def test_a_matrix_of_a_batch_has_the_bits_it_has_alone(device, mode, shape):
    # the batch's launches take 128 x 128 tiles, a single matrix's 64 x 64
    x = torch.randn(shape, generator=torch.Generator().manual_seed(sum(shape))).to(device)
    out = _s8_fp32(x, mode=mode)
    for i in (0, shape[0] // 2, shape[0] - 1):
        assert torch.equal(out[i], _s8_fp32(x[i], mode=mode))


@pytest.mark.parametrize("mode", ["fp32", "comp_bf16", "mixed"])
@pytest.mark.parametrize("rank1", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", [(256, 256), (300, 200), (200, 700), (700, 260)])
def test_64_tiles_in_the_matrix_step(device, mode, rank1, dtype, shape):
    """The stage-5 row sums, plain and transposed: one matrix on 64 x 64 tiles,
    on 128 x 128 tiles, and among 90 others of its shape (128 x 128 tiles)."""
    rows, cols = shape
    g = torch.Generator().manual_seed(rows + 3 * cols)
    vec = lambda n: (torch.rand(n, generator=g) + .5).to(device)
    inv_row, inv_col = vec(rows), vec(cols)
    z = (torch.randn(cols, generator=g) * .3).to(device)
    kappa = torch.tensor([-1 / (2 + math.sqrt(2))], device=device)
    w0 = (torch.randn(rows, cols, generator=g) * .02).to(device)
    grads = torch.randn(91, rows, cols, generator=g).to(device)

    def step(n):
        descs, keep = [], []
        for grad in grads[:n]:
            w, m = w0.to(dtype, copy=True), torch.zeros(rows, cols, device=device)
            keep.append((w, m))
            d = _native.MatrixDesc(param=w.data_ptr(), grad=grad.data_ptr(), momentum=m.data_ptr(),
                                   inv_row=inv_row.data_ptr(), inv_col=inv_col.data_ptr(), rows=rows, cols=cols,
                                   lr=1e-2, momentum_beta=.8, param_dtype=_native.dtype_code(dtype))
            if rank1:
                d.z, d.kappa = z.data_ptr(), kappa.data_ptr()
            descs.append(d)
        code = _native.S8_MODES[mode]
        ws = torch.empty(_native.matrix_step_workspace_bytes([shape] * n, code), dtype=torch.uint8, device=device)
        _native.matrix_step(descs, code, ws)
        torch.cuda.synchronize()
        return keep[0][0].float()

    a, b = _both(lambda: step(1))
    assert torch.equal(a, b)
    assert torch.equal(a, step(91))
    if dtype == torch.float32:
        assert abs(((w0 - a).double().norm() / 1e-2 / math.sqrt(rows)).item() - 1) <= 1e-4
