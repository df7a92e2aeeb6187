"""Geometries of the same rays share the ray tables: a second span or parameter
set takes little device memory, each lives on when the other goes, and the
last one gives the memory back."""
import copy

import pytest

pytestmark = pytest.mark.gpu
MB = 1 << 20


def test_same_rays_share_tables(params):
    import torch

    from nipet_amd.geom import DeviceGeom, get_geom
    from test_gpu_crossings import back, project, rows_of
    from nipet_amd import _lib as lib
    dev = torch.cuda.current_device()

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info(dev)[0]

    # rays that no other test's geometry has (their own field of view)
    Cnt = dict(params['Cnt'], TFOV2=880.0)
    a11, rows = dict(params, Cnt=Cnt), rows_of(torch, 40, 61)
    again = dict(copy.deepcopy(dict(params)), Cnt=dict(Cnt))
    img = torch.rand((320, 320, 127), device='cuda')
    project(torch, lib, 'nipet_fprj', get_geom(params), img, rows)  # (modules loaded)
    f0 = free()
    g1 = DeviceGeom(a11, dev)
    f1 = free()
    assert f0 - f1 > 3000 * MB
    g2 = DeviceGeom(dict(a11, Cnt=dict(Cnt, SPN=1)), dev)
    g3 = DeviceGeom(again, dev)
    assert f1 - free() < 64 * MB
    ref = project(torch, lib, 'nipet_fprj', g1, img, rows)
    s1 = project(torch, lib, 'nipet_fprj', g2, img, rows)
    y = torch.rand_like(s1)
    b1 = back(torch, lib, g2, y, rows)
    del g1
    assert torch.equal(project(torch, lib, 'nipet_fprj', g3, img, rows), ref)
    assert torch.equal(project(torch, lib, 'nipet_fprj', g2, img, rows), s1)
    assert float((back(torch, lib, g2, y, rows) - b1).abs().max()) <= 1e-5 * float(b1.max())
    assert g2.nseg == g3.nseg and g2.tx_lists()[0][-1] == g3.nseg
    # other rays do not share: one ring difference less
    ax = params['axLUT']
    r = ax['li2rno']
    few = abs(r[:, 0].astype(int) - r[:, 1]) < abs(r[:, 0].astype(int) - r[:, 1]).max()
    g4 = DeviceGeom(dict(again, axLUT=dict(ax, **{k: ax[k][few] for k in
                                                 ('li2rng', 'li2sn', 'li2nos')})), dev)
    out4 = project(torch, lib, 'nipet_fprj', g4, img, rows)
    assert bool((out4 <= ref * (1 + 1e-6)).all()) and not torch.equal(out4, ref)
    del g2, g3, g4, ref, s1, y, b1, out4
    torch.cuda.empty_cache()
    assert f0 - free() < 64 * MB
