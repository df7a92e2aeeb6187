"""The forward projector by z crossings (k_fprj) where it can go wrong, against
the FP64 oracle: non-finite voxels, signed images, bins that miss the object,
odd and strided batches, segment windows and single bins.

Tolerance: the parity bar of the projectors, 1e-5 of each value with values
below 1e-6 of the largest held to that floor; the kernel rounds to float32
(6e-8) and keeps a boundary's distance into its segment to 2^-32 of it."""
import ctypes as ct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BAR, FLOOR = 1e-5, 1e-6


@pytest.fixture(scope='module')
def torch():
    import torch
    assert torch.cuda.is_available(), 'GPU tests need a HIP device'
    return torch


@pytest.fixture(scope='module')
def lib():
    from nipet_amd import _lib
    return _lib


def close(torch, got, ref):
    got = got.double()
    ref = (torch.from_numpy(ref).cuda() if isinstance(ref, np.ndarray) else ref).double()
    fin = torch.isfinite(ref)
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(torch.isfinite(got), fin)
    top = float(ref[fin].abs().max())
    err = (got[fin] - ref[fin]).abs() / ref[fin].abs().clamp(min=FLOOR * max(top, 1e-30))
    assert float(err.max()) < BAR, float(err.max())


def project(torch, lib, name, geom, img, rows, att=0, nb=1):
    """``name`` over ``rows`` of device image(s) img; [rows, nsn(, nb)]."""
    out = torch.full((len(rows), geom.nsn) + ((nb,) if nb > 1 else ()), 7.0, device='cuda')
    args = [geom.handle, lib.ptr(out), lib.ptr(img), lib.ptr(rows), len(rows)]
    args += [nb] if name.endswith('_b') else []
    lib.check(getattr(lib.lib(), name)(*args, att, lib.stream_handle()), name)
    return out


def exact(torch, params, img, rows, att=0):
    from oracle import oracle as O
    return torch.from_numpy(np.asarray(O.fprj(params, img.cpu().numpy(), rows.cpu().numpy(),
                                              att=bool(att)))).cuda()


def rows_of(torch, n, seed=0):
    r = np.random.default_rng(seed).choice(68516, n, replace=False).astype(np.int32)
    return torch.from_numpy(r).cuda()


def image(torch, seed=3):
    from nipet_amd.prj.mmrsim import ellipsoid_phantom
    return torch.from_numpy(ellipsoid_phantom(seed)).cuda()


@pytest.mark.parametrize('kind', ['signed', 'zero', 'one voxel', 'faint'])
@pytest.mark.parametrize('n', [1, 97])
def test_images(torch, lib, params, kind, n):
    """Signed values, an empty image (exact zeros), one voxel (LORs that miss it
    exactly 0), and a weak background beside hot spheres."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, n)
    img = image(torch)
    if kind == 'signed':
        img = img * torch.sign(torch.rand(img.shape, device='cuda') - 0.3)
    elif kind == 'zero':
        img.zero_()
    elif kind == 'one voxel':
        img.zero_()
        img[160, 160, 63] = 1e4
    else:
        img = torch.where(img > 1, img, 1e-3 * img)
    got = project(torch, lib, 'nipet_fprj', geom, img, rows)
    ref = exact(torch, params, img, rows)
    if kind == 'signed':   # sums of both signs: to the size of their terms
        top = exact(torch, params, img.abs(), rows)
        assert float(((got - ref).abs() / top.clamp(min=1e-3)).max()) < BAR
    else:
        assert torch.equal(got == 0, ref == 0)
        close(torch, got, ref)


@pytest.mark.parametrize('bad', [float('inf'), float('-inf'), float('nan')])
@pytest.mark.parametrize('att', [0, 1])
def test_non_finite_voxels(torch, lib, params, bad, att):
    """Only the LORs that touch a non-finite voxel see it."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 64, 5)
    img = image(torch) * (0.01 if att else 1.0)
    off, col, _, _ = geom.tx_lists()
    aw = int(rows[0])
    c = int(col[(off[aw] + off[aw + 1]) // 2])  # a column on the first bin's ray
    at = (c // 320, c % 320, 60)
    img[at] = bad
    got = project(torch, lib, 'nipet_fprj', geom, img, rows, att)
    img2 = img.clone()
    img2[at] = 0.0
    clean = exact(torch, params, img2, rows, att)
    img2.zero_()
    img2[at] = 1.0
    hit = exact(torch, params, img2, rows) > 0
    assert bool(hit.any()) and not bool(hit.all())
    close(torch, got[~hit], clean[~hit])
    if att and bad == float('inf'):
        assert bool(torch.isfinite(got[hit]).all())
    else:
        assert not bool(torch.isfinite(got[hit]).any()) or (att and bad < 0)


@pytest.mark.parametrize('nb', [2, 3, 5])
@pytest.mark.parametrize('shift', [0, 1])
def test_batches(torch, lib, params, nb, shift):
    """Odd batches (pairs and a strided single) and images off their alignment;
    every image as projected alone, bit for bit."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 33, 9)
    one = image(torch)
    buf = torch.zeros(one.numel() * nb + 1, device='cuda')
    img = buf[shift:shift + one.numel() * nb].view(320, 320, 127, nb)
    for b in range(nb):
        img[..., b] = one * (b + 1) if b % 2 else one.flip(2)
    got = project(torch, lib, 'nipet_fprj_b', geom, img, rows, nb=nb)
    for b in range(nb):
        ref = project(torch, lib, 'nipet_fprj', geom, img[..., b].contiguous(), rows)
        assert torch.equal(got[..., b], ref), b


@pytest.mark.parametrize('span', [11, 1])
def test_window_is_the_masked_image(torch, lib, params, span):
    """The OSEM ratio over a mask's segment windows equals the one over whole
    rays for an image that is zero outside the mask."""
    from nipet_amd.geom import get_geom
    from nipet_amd.prj.osem import mask_window
    p = params if span == 11 else dict(params, Cnt=dict(params['Cnt'], SPN=1))
    geom, rows = get_geom(p), rows_of(torch, 41, 11)
    y, x = np.ogrid[:320, :320]
    disc = torch.from_numpy(((y - 150)**2 + (x - 170)**2 < 55**2)).cuda()
    mask = disc[:, :, None].expand(320, 320, 127).to(torch.uint8).contiguous()
    img = (image(torch) + 0.1) * mask
    win = mask_window(geom, mask)
    g = torch.Generator(device='cuda').manual_seed(1)
    prompts = torch.randint(0, 50, (geom.naw, geom.nsn), generator=g, device='cuda',
                            dtype=torch.int32).to(torch.uint16)
    rho = torch.full((geom.naw, geom.nsn), 0.5, device='cuda')
    sens = torch.ones((320, 320, 127), device='cuda')
    outs = []
    for w in (None, win):
        work, wimg, im = (torch.zeros((len(rows), geom.nsn), device='cuda'),
                          torch.zeros_like(img), img.clone())
        lib.check(lib.lib().nipet_osem_subset(
            geom.handle, lib.ptr(im), lib.ptr(prompts), lib.ptr(rho), lib.ptr(sens),
            lib.ptr(mask), lib.ptr(w), lib.ptr(rows), len(rows), lib.ptr(work), lib.ptr(wimg),
            lib.stream_handle()), 'nipet_osem_subset')
        outs.append(work)
    close(torch, outs[1], outs[0])
    assert isinstance(geom.handle, ct.c_void_p)


# ------------------------------------------------------------ back projection
def back(torch, lib, geom, sino, rows, scratch_rows=None, nb=1):
    """``nipet_bprj_b`` without scratch (atomics), or staged with room for
    ``scratch_rows`` bins a pass."""
    img = torch.full((320, 320, 127) + ((nb,) if nb > 1 else ()), 3.0, device='cuda')
    buf = None
    if scratch_rows:
        full = lib.lib().nipet_bprj_scratch(geom.handle, len(rows), nb)
        one = lib.lib().nipet_bprj_scratch(geom.handle, 2001, nb) - \
            lib.lib().nipet_bprj_scratch(geom.handle, 2000, nb)
        n = full - (len(rows) - min(scratch_rows, len(rows))) * one
        buf = torch.full((n,), 255, dtype=torch.uint8, device='cuda')
    with lib.scratch(buf):
        lib.check(lib.lib().nipet_bprj_b(geom.handle, lib.ptr(img), lib.ptr(sino), lib.ptr(rows),
                                         len(rows), nb, lib.stream_handle()), 'nipet_bprj_b')
    return img


def exact_back(torch, params, sino, rows):
    from oracle import oracle as O
    return torch.from_numpy(O.bprj(params, sino.cpu().numpy(), rows.cpu().numpy())).cuda()


@pytest.mark.parametrize('kind', ['signed', 'one bin', 'huge beside small'])
def test_back_projection_sums_return_to_zero(torch, lib, params, kind):
    """The plane sums along a ray hold what enters and leaves: voxels that no
    LOR with a value touches get exactly 0, and small values beside huge ones
    keep their precision (a sum of a voxel's own terms bounds its error)."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 1 if kind == 'one bin' else 23, 21)
    g = torch.Generator(device='cuda').manual_seed(2)
    y = torch.rand((len(rows), geom.nsn), generator=g, device='cuda')
    y = y * (torch.rand(y.shape, generator=g, device='cuda') < 0.05)
    if kind == 'signed':
        y = y * torch.sign(torch.rand(y.shape, generator=g, device='cuda') - 0.5)
    elif kind != 'one bin':
        y[:, ::3] *= 1e6
    got = back(torch, lib, geom, y, rows).double()
    ref, top = exact_back(torch, params, y, rows), exact_back(torch, params, y.abs(), rows)
    assert bool((got[top == 0] == 0).all())
    assert float(((got - ref).abs() / top.clamp(min=1e-3 if kind != 'one bin' else 1e-4)).max()) < BAR


@pytest.mark.parametrize('bad', [float('inf'), float('nan')])
def test_back_projection_non_finite(torch, lib, params, bad):
    """A non-finite sinogram value reaches the voxels of its LORs and no others."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 9, 22)
    y = torch.rand((len(rows), geom.nsn), device='cuda')
    one = torch.zeros_like(y)
    one[4, 400] = 1.0
    hit = exact_back(torch, params, one, rows) > 0
    clean = y.clone()
    clean[4, 400] = 0.0
    y[4, 400] = bad
    got = back(torch, lib, geom, y, rows)
    assert not bool(torch.isfinite(got[hit]).any())
    close(torch, got[~hit], exact_back(torch, params, clean, rows)[~hit])


@pytest.mark.parametrize('nb', [1, 2, 3])
@pytest.mark.parametrize('n,per', [(1536, 1536), (1700, 1537), (3400, 1600)])
def test_staged_equals_atomics(torch, lib, params, n, per, nb):
    """Staged rows gathered in one or several passes against float atomics:
    duplicated and invalid bins, odd batches, twice the same bits."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, n, 23)
    rows[7], rows[n // 2], rows[n - 1] = rows[11], -1, 68516
    g = torch.Generator(device='cuda').manual_seed(4)
    y = torch.rand((n, geom.nsn) + ((nb,) if nb > 1 else ()), generator=g, device='cuda')
    ref = back(torch, lib, geom, y, rows, None, nb).double()
    got = back(torch, lib, geom, y, rows, per, nb)
    assert torch.equal(got, back(torch, lib, geom, y, rows, per, nb))
    assert float((got - ref).abs().max()) < BAR * float(ref.max())
    assert torch.equal(got == 0, ref == 0)
    if nb > 1:
        for b in range(nb):
            one = back(torch, lib, geom, y[..., b].contiguous(), rows, n)
            assert float((got[..., b] - one).abs().max()) < 1e-6 * float(one.max())


@pytest.mark.parametrize('dmax', [0, 1, 7])
def test_few_ring_differences(torch, lib, params, dmax):
    """Michelograms of the first ring differences only (none of them crosses a
    plane at dmax 0): the projections by segments, and the adjoint of them."""
    from nipet_amd.geom import DeviceGeom
    ax = params['axLUT']
    sel = np.abs(ax['li2rng'][:, 0] - ax['li2rng'][:, 1]) < (dmax + 0.5) * params['Cnt']['AXR']
    few = dict(params, axLUT=dict(ax, **{k: ax[k][sel] for k in ('li2rng', 'li2sn', 'li2nos')}))
    geom, rows = DeviceGeom(few, torch.cuda.current_device()), rows_of(torch, 40, 31)
    g = torch.Generator(device='cuda').manual_seed(6)
    img = torch.rand((320, 320, 127), generator=g, device='cuda')
    out = [torch.full((len(rows), geom.nsn), 9.0, device='cuda') for _ in range(2)]
    for o, name in zip(out, ('nipet_fprj', 'nipet_fprj_seg')):
        lib.check(getattr(lib.lib(), name)(geom.handle, lib.ptr(o), lib.ptr(img), lib.ptr(rows),
                                           len(rows), 0, lib.stream_handle()), name)
    assert float((out[0] - out[1]).abs().max()) < BAR * float(out[1].max())
    y = torch.rand((len(rows), geom.nsn), generator=g, device='cuda')
    dot = float((back(torch, lib, geom, y, rows).double() * img).sum())
    assert abs(dot / float((out[0].double() * y).sum()) - 1) < 1e-6


def test_scratch_nests(torch, lib, params):
    """Leaving an inner scratch context gives the outer one back: staged sums
    (the same bits) and not atomics; without room there is no buffer."""
    from nipet_amd.geom import get_geom
    geom, rows = get_geom(params), rows_of(torch, 2000, 41)
    y = torch.rand((len(rows), geom.nsn), device='cuda')
    outer = lib.bprj_scratch(geom, len(rows))
    imgs = [torch.zeros((320, 320, 127), device='cuda') for _ in range(2)]
    with lib.scratch(outer):
        for im in imgs:
            with lib.scratch(None):
                pass
            outer.fill_(255)
            lib.check(lib.lib().nipet_bprj_b(geom.handle, lib.ptr(im), lib.ptr(y), lib.ptr(rows),
                                             len(rows), 1, lib.stream_handle()), 'nipet_bprj_b')
            assert not bool((outer == 255).all())  # the rows went there
    assert torch.equal(*imgs)
