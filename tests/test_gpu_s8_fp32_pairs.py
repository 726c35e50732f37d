"""The fp32 mode's FP16 pairs: accuracy against the FP64 map and range.

A pair carries 22 significant bits and every product FP32 accumulation, so
the map's error is that of FP32 GEMMs: a few 1e-6 on scaled Gaussian
matrices, up to 1e-4 on steep spectra at 2048, where FP32 operands on FP32
MFMAs measured 4e-6 to 1.1e-5 and 1.5e-4.  The bounds are about three times
the pairs' own measurements."""
import math

import pytest
import torch

from oracle import sandmuon_oracle as O
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


@pytest.mark.parametrize("shape", [(2, 130, 150), (2, 90, 700)])
@pytest.mark.parametrize("k", [-60, -20, 30, 55])
def test_fp32_mode_ignores_powers_of_two(device, shape, k):
    # The input's exponent is folded into the scales exactly.
    x = _input(shape, "scaled", 5).to(device)
    assert torch.equal(_s8_fp32(x * math.ldexp(1.0, k)), _s8_fp32(x))


def test_fp32_mode_keeps_non_finite_inputs_visible(device):
    x = torch.randn(2, 40, 50, device=device)
    x[1, 3, 4] = float("inf")
    out = _s8_fp32(x)
    assert torch.isfinite(out[0]).all() and not torch.isfinite(out[1]).all()
