"""How smx_s8 reads its input and leaves its result: the vector and the
element-wise load and store, and the result written straight to `out` by the
last stage, must all give the same bits."""
import pytest
import torch

from oracle import sandmuon_oracle as O
from sandmuon_amd import _native

pytestmark = pytest.mark.gpu


def _s8(x, out, mode):
    b, r, c = x.shape
    ws = torch.empty(int(_native.lib().smx_s8_workspace_bytes(b, r, c, mode)), dtype=torch.uint8, device=x.device)
    rc = _native.lib().smx_s8(x.data_ptr(), out.data_ptr(), b, r, c, *x.stride(), mode, ws.data_ptr(), ws.numel(),
                              _native.stream_of(x.device))
    assert rc == 0
    torch.cuda.synchronize()
    return out


# Padded sizes (the result goes straight to `out`: X-space, Gram space,
# transposed), sizes with padding, and odd columns (element-wise load).
@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("shape", [(2, 256, 256), (1, 256, 768), (5, 512, 256), (2, 260, 132), (1, 70, 301),
                                   (4, 301, 70), (3, 1, 5)])
def test_every_load_and_store_gives_the_same_bits(device, mode, shape):
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(shape, generator=g).to(device)
    want = _s8(x, torch.empty_like(x), mode)
    ref = O.s8(x.cpu())
    err = (want.cpu() - ref).flatten(1).norm(dim=1) / ref.flatten(1).norm(dim=1)
    assert err.max() <= (1e-4 if mode == 0 else 1e-2)
    # in place (a result never goes straight to an `out` that overlaps x)
    y = x.clone()
    assert torch.equal(_s8(y, y, mode), want)
    # rows 1, 2 and 4 elements apart from the next boundary
    for pad in (1, 2, 4):
        wide = torch.zeros(shape[0], shape[1], shape[2] + pad, device=device)
        wide[..., :shape[2]] = x
        res = torch.full_like(wide, 7.0)
        assert torch.equal(_s8(wide[..., :shape[2]], res[..., :shape[2]], mode)[..., :shape[2]], want)
        assert (res[..., shape[2]:] == 7.0).all()
    # column-major
    xt = x.transpose(1, 2).contiguous().transpose(1, 2)
    assert torch.equal(_s8(xt, torch.empty_like(xt), mode), want)
    # an `out` that starts 4 bytes off a boundary
    flat = torch.empty(x.numel() + 1, device=device)
    assert torch.equal(_s8(x, flat[1:].view(shape), mode), want)
