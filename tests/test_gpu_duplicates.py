"""Bins listed more than once in a staged back projection, far apart and three
times over: every row counts once, as with float atomics.

Tolerance: the parity bar 1e-5 of the image's largest value, as between the two
ways in general (float32 sums of the same positive terms in another order)."""
import pytest

from test_gpu_crossings import back, rows_of

pytestmark = pytest.mark.gpu
BAR = 1e-5


@pytest.mark.parametrize('nb', [1, 2])
@pytest.mark.parametrize('n,per', [(1800, 1800), (3300, 1600)])
def test_bins_listed_more_than_once(params, n, per, nb):
    import torch

    from nipet_amd import _lib as lib
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, n, 71)
    rows[0] = rows[700] = rows[1500]      # three times, in blocks of their own
    rows[n - 1] = rows[3]                 # in the first and the last pass
    rows[300:364] = rows[900:964]         # a whole wave of pairs
    g = torch.Generator(device='cuda').manual_seed(7)
    y = torch.rand((n, geom.nsn) + ((nb,) if nb > 1 else ()), generator=g, device='cuda')
    ref = back(torch, lib, geom, y, rows, None, nb).double()
    got = back(torch, lib, geom, y, rows, per, nb)
    assert float((got - ref).abs().max()) < BAR * float(ref.max())
    assert torch.equal(got == 0, ref == 0)
    # the repeated rows alone: as many times their own image
    few = torch.full_like(rows, -1)
    few[[0, 700, 1500]] = rows[0]
    y[700], y[1500] = y[0], y[0]
    one = back(torch, lib, geom, y[:1].contiguous(), rows[:1].contiguous(), None, nb).double()
    got = back(torch, lib, geom, y, few, per, nb).double()
    assert float((got - 3 * one).abs().max()) < BAR * float(one.max())
