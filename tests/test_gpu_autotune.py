"""The batch autotuner times what a batch launches: its own strided images, each
different way of splitting them once, and leaves settings that no kernel reads
alone."""
import ctypes as ct

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nb,times', [(4, {'fprj': [4, 1], 'bprj': [4, 1]}),
                                      (1, {'fprj': [4], 'bprj': [4]})])
def test_times_the_batch_itself(params, monkeypatch, nb, times):
    import torch

    from nipet_amd import _lib
    from nipet_amd.prj import batch
    from nipet_amd.prj.osem import osem_prepare_batch
    monkeypatch.setattr(batch, '_TUNED', {})
    shape = (68516, 837)
    one = torch.ones(shape, device='cuda')
    st = osem_prepare_batch(params, torch.ones(shape + (nb,), dtype=torch.int32,
                                               device='cuda').to(torch.uint16), one, one)
    calls, L = [], _lib.lib()

    class Lib:  # the library, its batched projections noted down
        def __getattr__(self, name):
            f = getattr(L, name)
            if name not in ('nipet_fprj_b', 'nipet_bprj_b'):
                assert name != 'nipet_tune_set_run'
                return f
            w, kernel = ct.c_int(), _lib.PROF_FPRJ if name == 'nipet_fprj_b' else _lib.PROF_BPRJ
            _lib.check(L.nipet_tune_get(kernel, ct.byref(w)))

            def noted(*args):
                calls.append((name[6:10], w.value, args[5]))
                return f(*args)
            return noted

    monkeypatch.setattr(_lib, 'lib', Lib)
    res = batch.autotune(st, repeats=2)
    monkeypatch.undo()
    assert all(n == nb for _, _, n in calls)  # whole batches, as they lie
    for name, widths in times.items():
        assert [w for k, w, _ in calls if k == name] == [w for w in widths for _ in range(3)]
        assert res[name] in widths
        keys = [k[1] for k in res['ms'] if k[0] == name]
        assert keys == widths and res[name] == min(
            keys, key=lambda w: [v for k, v in res['ms'].items() if k[:2] == (name, w)][0])
    for k in (_lib.PROF_FPRJ, _lib.PROF_BPRJ):
        _lib.check(_lib.lib().nipet_tune_set(k, 4))
