"""smx_rank1_apply at the edges of its column tiles (32), row groups (32, four
rows in flight) and row loops (rounds of eight columns for each of a row's 64
or 256 lanes: 512 or 2048 columns), against the same formula in float64.  The bound: FP64 sums, so an element carries the few
FP32 roundings of its own expression (eps32 = 6e-8 each)."""
import pytest
import torch

from oracle import sandmuon_oracle as O
from sandmuon_amd.optimizer import rank1_mapback, rank1_whiten

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-6), (torch.float64, 1e-13)])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 2, 33), (2, 31, 32), (1, 33, 65), (2, 128, 255), (1, 129, 257),
                                   (1, 300, 1025), (70, 5, 7)])
def test_rank1_apply_edges(device, dtype, tol, shape):
    b, r, c = shape
    g = torch.Generator().manual_seed(b + 10 * r + 100 * c)
    x = torch.randn(shape, generator=g, dtype=dtype)
    fac = lambda n: (torch.rand(b, n, generator=g, dtype=dtype) + .5, torch.randn(b, n, generator=g, dtype=dtype) * .3,
                     -torch.rand(b, generator=g, dtype=dtype) * .5)
    left, right = fac(r), fac(c)
    up = lambda f: tuple(t.double() for t in f)
    got = rank1_whiten(x.to(device), left, right)
    want = O.rank1_whiten(x.double(), up(left), up(right))
    assert got.dtype == dtype and (got.cpu().double() - want).norm() <= tol * want.norm()
    got = rank1_mapback(x.to(device), left, right).cpu().double()
    for k in range(b):
        one = lambda f: tuple(t[k].double() for t in f)
        want = O.rank1_mapback(x[k].double(), one(left), one(right))
        assert (got[k] - want).norm() <= tol * want.norm()


# Rows of several rounds, which are read again for the output: four waves per
# row from 2049 columns on, one wave (more than 65536 rows) from 513
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-6), (torch.float64, 1e-13)])
@pytest.mark.parametrize("shape", [(2, 6, 2047), (2, 6, 2048), (2, 6, 2049), (2, 5, 4100), (1, 65537, 512),
                                   (1, 65537, 513)])
def test_rank1_apply_long_rows(device, dtype, tol, shape):
    b, r, c = shape
    g = torch.Generator().manual_seed(r + c)
    x = torch.randn(shape, generator=g, dtype=dtype)
    fac = lambda n: (torch.rand(b, n, generator=g, dtype=dtype) + .5,
                     torch.randn(b, n, generator=g, dtype=dtype) / n ** .5, -torch.rand(b, generator=g, dtype=dtype) * .5)
    left, right = fac(r), fac(c)
    for fn, oracle in ((rank1_whiten, O.rank1_whiten), (rank1_mapback, O.rank1_mapback)):
        got = fn(x.to(device), left, right).cpu().double()
        for k in range(b):
            one = lambda f: tuple(t[k].double() for t in f)
            want = oracle(x[k].double(), one(left), one(right))
            assert (got[k] - want).norm() <= tol * want.norm()
            # the last round's columns by themselves
            assert (got[k, :, -1] - want[:, -1]).norm() <= 10 * tol * want[:, -1].norm()


@pytest.mark.parametrize("shared", ["left", "right", "both"])
@pytest.mark.parametrize("shape", [(3, 33, 65), (2, 5, 256), (4, 7, 2048), (2, 6, 2049), (2, 65537, 257)])
def test_factors_shared_by_the_batch_equal_expanded_ones(device, shape, shared):
    # A row on one wave and on four, on one round of columns and on two: the
    # same values are read, so the bits are the same.
    b, r, c = shape
    g = torch.Generator().manual_seed(b + 10 * r + 100 * c)
    x = torch.randn(shape, generator=g).to(device)
    one = lambda n: tuple(t.to(device) for t in (torch.rand(n, generator=g) + .5, torch.randn(n, generator=g) * .3 / n ** .5,
                                                 torch.tensor(-.25)))
    many = lambda f: (f[0].expand(b, -1).contiguous(), f[1].expand(b, -1).contiguous(), f[2].expand(b).contiguous())
    left, right = one(r), one(c)
    lf = left if shared != "right" else many(left)
    rf = right if shared != "left" else many(right)
    for fn in (rank1_whiten, rank1_mapback):
        got, want = fn(x, lf, rf), fn(x, many(left), many(right))
        assert torch.equal(got, want)
    k = b - 1
    ref = O.rank1_whiten(x[k].double().cpu(), *[tuple(t.double().cpu() for t in f) for f in (left, right)])
    assert (rank1_whiten(x, left, right)[k].double().cpu() - ref).norm() <= 1e-6 * ref.norm()
