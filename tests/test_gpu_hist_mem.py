"""List-mode sessions in the caller's memory: the same counts as in memory of
their own, on another stream, in chunks of growing size; too little memory is
refused."""
import ctypes as ct

import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def words(params):
    from nipet_amd.lm.lmsim import synth_lm
    return synth_lm(params, 4, 300, seed=5)


@pytest.mark.parametrize('span,btp,nrep', [(11, 0, 1), (1, 0, 1), (11, 2, 3), (0, 1, 1)])
def test_callers_memory_equals_own(params, words, span, btp, nrep):
    import torch

    from nipet_amd import _lib
    from nipet_amd.lm.mmrhist import LmHistogram, tag_range
    tf, tl = tag_range(words)
    kw = dict(span=span, btp=btp, nrep=nrep, seed=3)
    cuts = [0, 8192, 3 * 8192, len(words)]
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        side.wait_stream(torch.cuda.default_stream())
        a = LmHistogram(params, tf, (tl - tf + 999) // 1000, **kw)
        for i, j in zip(cuts, cuts[1:]):
            a.add(words[i:j])
        a.finish()
    side.synchronize()
    b = LmHistogram(params, tf, (tl - tf + 999) // 1000, **kw)
    L, own = _lib.lib(), ct.c_void_p()
    cfg = _lib.NipetLmConfig(tf, b.nitag, 0, b.nitag, span, btp, b.btprt, 3, nrep, 0,
                             *[k.ctypes.data for k in b._keep])
    _lib.check(L.nipet_lm_create(ct.byref(cfg), ct.byref(own)))
    for i, j in zip(cuts, cuts[1:]):
        w = words[i:j].contiguous()
        _lib.check(L.nipet_lm_chunk(own, w.data_ptr(), len(w), ct.byref(b._o),
                                    _lib.stream_handle()))
    _lib.check(L.nipet_lm_finish(own, ct.byref(b._o), _lib.stream_handle()))
    torch.cuda.synchronize()
    for k in a.out:
        assert torch.equal(a.out[k], b.out[k]), k
    n, bad, ovf = ct.c_int64(), ct.c_uint(), ct.c_uint()
    _lib.check(L.nipet_lm_status(own, ct.byref(n), ct.byref(bad), ct.byref(ovf)))
    assert (n.value, bad.value, ovf.value) == a.status() and n.value == len(words)
    L.nipet_lm_destroy(own)
    need = L.nipet_lm_work_bytes(a.handle, len(words))
    mem = torch.empty(need, dtype=torch.uint8, device='cuda')
    assert L.nipet_lm_chunk_in(a.handle, words.data_ptr(), len(words), ct.byref(a._o),
                               mem.data_ptr(), need - 1, _lib.stream_handle()) != 0
    size = L.nipet_lm_bytes(ct.byref(cfg))
    assert L.nipet_lm_create_in(ct.byref(cfg), mem.data_ptr(), size - 1, _lib.stream_handle(),
                                ct.byref(own)) != 0


@pytest.mark.parametrize('span', [11, 0])
def test_outputs_at_odd_addresses(params, words, span):
    """Outputs that are not aligned to 16 bytes, in two chunks: the same counts."""
    import torch

    from nipet_amd.lm.mmrhist import LmHistogram, tag_range
    tf, tl = tag_range(words)
    outs = []
    for shift in (0, 1):
        h = LmHistogram(params, tf, (tl - tf + 999) // 1000, span=span)
        for k in ('psino', 'dsino', 'ssr'):
            t = h.out[k]
            h.out[k] = torch.zeros(t.numel() + shift, dtype=t.dtype,
                                   device='cuda')[shift:].view(t.shape)
            setattr(h._o, k, h.out[k].data_ptr())
        h.add(words[:5 * 8192])
        h.add(words[5 * 8192:])
        h.finish()
        outs.append(h.out)
    for k in outs[0]:
        assert torch.equal(outs[0][k], outs[1][k]), k
