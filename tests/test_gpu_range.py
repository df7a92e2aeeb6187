"""Projections of values that span the whole range of float32: small values keep
their precision beside large ones, huge finite values overflow only where they
must, and non-finite ones reach only what they touch, with float atomics and
staged, one image and two.

Tolerance: every value against the sum of its own terms' magnitudes, 1e-5 (at
most a hundred float32 additions of 6e-8). What large values touch, or miss by
less than a plane, is left out: there their own rounding rules."""
import numpy as np
import pytest

from test_gpu_crossings import back, exact, exact_back, project, rows_of

pytestmark = pytest.mark.gpu
BAR = 1e-5


@pytest.fixture(scope='module')
def torch():
    import torch
    assert torch.cuda.is_available(), 'GPU tests need a HIP device'
    return torch


@pytest.fixture(scope='module')
def lib():
    from nipet_amd import _lib
    return _lib


def near(torch, hit):
    """Voxels of ``hit`` and those on the planes next to them."""
    n = hit.clone()
    n[..., 1:] |= hit[..., :-1]
    n[..., :-1] |= hit[..., 1:]
    return n


def own(got, ref, free):
    """Largest error of ``got`` (all terms positive) relative to each value;
    where the reference is 0 the value has to be 0."""
    got, ref = got[free].double(), ref[free].double()
    assert bool((got[ref == 0] == 0).all())
    pos = ref > 0
    return float(((got - ref).abs()[pos] / ref[pos]).max())


# ------------------------------------------------------------ back projection
def rays(torch, geom, n, bright, faint, seed):
    """Sinogram of values about ``faint`` with a few of ``bright``, and those alone."""
    g = torch.Generator(device='cuda').manual_seed(seed)
    y = faint * (0.5 + torch.rand((n, geom.nsn), generator=g, device='cuda'))
    big = torch.zeros_like(y)
    big[:, 700:710] = bright
    big[::3] = 0.0
    return torch.where(big > 0, big, y), big


@pytest.mark.parametrize('bright,faint', [(1e6, 1e-12), (3.4e38, 1.0), (1.0, 1e-6), (1.0, 3e-7),
                                          (1.0, 1e-7), (1e30, 1e-30)])
def test_back_projection_small_beside_large(torch, lib, params, bright, faint):
    """Float atomics against the FP64 oracle."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 23, 51)
    y, big = rays(torch, geom, len(rows), bright, faint, 1)
    hit = near(torch, exact_back(torch, params, (big > 0).float(), rows) > 0)
    ref = exact_back(torch, params, y, rows)
    assert bool(hit.any()) and bool((ref[~hit] > 0).any())
    assert own(back(torch, lib, geom, y, rows), ref, ~hit) < BAR


@pytest.mark.parametrize('nb', [1, 2])
@pytest.mark.parametrize('bright,faint', [(1e6, 1e-12), (3.4e38, 1.0), (1.0, 1e-6)])
def test_staged_small_beside_large(torch, lib, params, bright, faint, nb):
    """Staged sums against float atomics of each image; a second image at
    another scale altogether."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 1601, 52)
    y, big = rays(torch, geom, len(rows), bright, faint, 2)
    hit = near(torch, back(torch, lib, geom, (big > 0).float(), rows) > 0)
    ref = [back(torch, lib, geom, y, rows)]
    if nb == 2:
        other = 1e-22 * torch.rand_like(y)
        ref.append(back(torch, lib, geom, other, rows))
        y = torch.stack([y, other], 2).contiguous()
    got = back(torch, lib, geom, y, rows, len(rows), nb)
    assert own(got[..., 0] if nb == 2 else got, ref[0], ~hit) < BAR
    if nb == 2:
        assert own(got[..., 1], ref[1], torch.ones_like(hit)) < BAR


@pytest.mark.parametrize('bad', [float('inf'), float('nan')])
def test_staged_non_finite_pair(torch, lib, params, bad):
    """Staged, two images: a non-finite value reaches the voxels of its LORs in
    its own image."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 1537, 53)
    y = torch.rand((len(rows), geom.nsn, 2), device='cuda')
    one = torch.zeros_like(y[..., 0])
    one[700, 400] = 1.0
    hit = back(torch, lib, geom, one, rows) > 0
    ref = [back(torch, lib, geom, (y[..., b] * (1 - one)) if b == 0 else y[..., b].contiguous(),
                rows) for b in range(2)]
    y[700, 400, 0] = bad
    got = back(torch, lib, geom, y, rows, len(rows), 2)
    assert bool(hit.any()) and not bool(torch.isfinite(got[..., 0][hit]).any())
    assert own(got[..., 0], ref[0], ~hit) < BAR
    assert own(got[..., 1], ref[1], torch.ones_like(hit)) < BAR


# --------------------------------------------------------- forward projection
def voxels(torch, geom, rows, bright, faint, seed):
    """Image of values about ``faint`` with a few voxels of ``bright`` on the
    first bins' rays, and the voxels within a plane of those."""
    g = torch.Generator(device='cuda').manual_seed(seed)
    img = faint * (0.5 + torch.rand((320, 320, 127), generator=g, device='cuda'))
    off, col, _, _ = geom.tx_lists()
    big = torch.zeros(img.shape, dtype=torch.bool, device='cuda')
    for k, aw in enumerate(rows[:8].tolist()):
        c = int(col[(off[aw] + off[aw + 1]) // 2])
        big[c // 320, c % 320, 30 + 8 * k] = True
    return torch.where(big, torch.full_like(img, bright), img), near(torch, big)


@pytest.mark.parametrize('bright,faint', [(1e6, 1e-12), (3.4e38, 1.0), (1.0, 1e-6), (1e30, 1e-30)])
def test_forward_projection_small_beside_large(torch, lib, params, bright, faint):
    """LORs that do not touch the large voxels, against the FP64 oracle; in a
    batch as alone, bit for bit."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 24, 54)
    img, big = voxels(torch, geom, rows, bright, faint, 3)
    hit = exact(torch, params, big.float(), rows) > 0
    got, ref = project(torch, lib, 'nipet_fprj', geom, img, rows), exact(torch, params, img, rows)
    assert bool(hit.any()) and bool((ref[~hit] > 0).any())
    assert own(got, ref, ~hit) < BAR
    assert bool((got[hit] > 0).all())
    two = torch.stack([torch.rand_like(img), img], 3).contiguous()
    assert torch.equal(project(torch, lib, 'nipet_fprj_b', geom, two, rows, nb=2)[..., 1], got)


@pytest.mark.parametrize('bright', [1e7, 3.4e38])
def test_attenuation_beside_large(torch, lib, params, bright):
    """Attenuation factors of LORs that do not touch the large voxels."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 24, 55)
    mu, big = voxels(torch, geom, rows, bright, 0.01, 4)
    hit = exact(torch, params, big.float(), rows) > 0
    got = project(torch, lib, 'nipet_fprj', geom, mu, rows, 1)
    assert own(got, exact(torch, params, mu, rows, 1), ~hit) < BAR
    assert bool((got[hit] < 1).all())


@pytest.mark.parametrize('bright,faint,add', [(1e6, 1e-5, 0.0), (3.4e38, 1e-2, 0.0),
                                              (1e6, 1e-5, 1e-3), (1e6, 1e-5, 1e2)])
def test_ratio_beside_large(torch, lib, params, bright, faint, add):
    """The OSEM ratio of LORs that do not touch the large voxels, without and with
    an additive term."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 24, 56)
    img, big = voxels(torch, geom, rows, bright, faint, 5)
    hit = exact(torch, params, big.float(), rows) > 0
    prompts = torch.full((geom.naw, geom.nsn), 3, dtype=torch.int32, device='cuda').to(torch.uint16)
    rho = torch.full((geom.naw, geom.nsn), add, device='cuda')
    mask = torch.ones((320, 320, 127), dtype=torch.uint8, device='cuda')
    sens, wimg = torch.ones((320, 320, 127), device='cuda'), torch.empty_like(img)
    got, upd = torch.zeros((len(rows), geom.nsn), device='cuda'), img.clone()
    lib.check(lib.lib().nipet_osem_subset(
        geom.handle, lib.ptr(upd), lib.ptr(prompts), lib.ptr(rho), lib.ptr(sens),
        lib.ptr(mask), None, lib.ptr(rows), len(rows), lib.ptr(got), lib.ptr(wimg),
        lib.stream_handle()), 'nipet_osem_subset')
    ref = exact(torch, params, img, rows).double() + add
    assert float(ref[~hit].min()) > 1e-5  # (far from the guard)
    assert own(got, 3.0 / ref, ~hit) < BAR


@pytest.mark.parametrize('bad', [float('inf'), float('nan')])
def test_forward_non_finite_pair(torch, lib, params, bad):
    """Two images: a non-finite voxel changes nothing in the other image, and in
    its own the LORs that touch it."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 24, 57)
    img, big = voxels(torch, geom, rows, bad, 1.0, 6)
    hit = exact(torch, params, big.float(), rows) > 0
    clean = torch.where(torch.isfinite(img), img, torch.zeros_like(img))
    two = torch.stack([img, torch.rand_like(img)], 3).contiguous()
    got = project(torch, lib, 'nipet_fprj_b', geom, two, rows, nb=2)
    assert torch.equal(got[..., 1], project(torch, lib, 'nipet_fprj', geom,
                                            two[..., 1].contiguous(), rows))
    assert own(got[..., 0], exact(torch, params, clean, rows), ~hit) < BAR
    touch = exact(torch, params, (~torch.isfinite(img)).float(), rows) > 0
    assert not bool(torch.isfinite(got[..., 0][touch]).any())
