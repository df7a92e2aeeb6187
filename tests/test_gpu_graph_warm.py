"""Before a batch's graph is captured, everything that it captures has been
launched once: the same entry points, batch sizes, and staged or direct back
projections; the replays then give the eager images."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('psf', [False, True])
def test_capture_launches_nothing_new(params, monkeypatch, psf):
    import torch

    import nipet_amd as nip
    from nipet_amd import _lib
    from nipet_amd.prj.batch import OsemGraph
    from nipet_amd.prj.osem import osem_prepare_batch, osem_run_batch
    subs = [np.asarray(nip.get_subsets14(0, params)[0], np.int32)]
    subs.append(np.asarray(nip.get_subsets14(1, params)[0][:200], np.int32))  # not staged
    g = torch.Generator(device='cuda').manual_seed(5)
    one = torch.ones((68516, 837), device='cuda')
    krnl = nip.psf_config(4.5, params['Cnt']) if psf else None
    states, sens = [], None
    for nb in (3, 3, 1):
        p = torch.randint(0, 9, (68516, 837, nb), generator=g, device='cuda', dtype=torch.int32)
        states.append(osem_prepare_batch(params, p.to(torch.uint16), one, one, one, subsets=subs,
                                         sens=sens, psf=krnl))
        sens = states[0].sens
    ref = [osem_run_batch(st, 1) for st in states]
    warm, captured, L = set(), set(), _lib.lib()

    class Lib:  # the library, its subset updates noted down
        def __getattr__(self, name):
            f = getattr(L, name)
            if not name.startswith('nipet_osem_subset'):
                return f

            def noted(*args):
                nprj, nb = args[10], args[11]
                staged = _lib._scratch.buf is not None and \
                    L.nipet_bprj_scratch(args[0], nprj, nb) > 0
                (captured if torch.cuda.is_current_stream_capturing() else warm).add(
                    (name, nb, staged))
                return f(*args)
            return noted

    monkeypatch.setattr(_lib, 'lib', Lib)
    graph = OsemGraph(states, 1)
    monkeypatch.undo()
    assert len(captured) == 4 and captured <= warm, (captured, warm)
    for _ in range(3):
        for im, r in zip(graph.run_groups(), ref):
            assert float((im - r).abs().max()) <= 1e-5 * float(r.max())
        torch.cuda.synchronize()
        assert torch.isfinite(osem_run_batch(states[2], 1)).all()
