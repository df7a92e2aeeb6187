"""A list-mode session that is made on one stream, used on another and dropped
at once: its memory is not given out again while the other stream's kernels
still use it, and the outputs kept from it are whole."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('drop_out', [False, True])
def test_session_on_another_stream(params, drop_out):
    import torch

    from nipet_amd.lm.lmsim import synth_lm
    from nipet_amd.lm.mmrhist import LmHistogram, tag_range
    words = synth_lm(params, 4, 300, seed=8)
    tf, tl = tag_range(words)

    def session():
        return LmHistogram(params, tf, (tl - tf + 999) // 1000)

    ref = session()
    ref.add(words)
    ref.finish()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    a = torch.rand((4096, 4096), device='cuda')
    h = session()
    sizes = {k: v.numel() for k, v in h.out.items()}
    ptrs = {h._mem.data_ptr(): '_mem', **{v.data_ptr(): k for k, v in h.out.items()}}
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(64):  # the histogram's kernels wait behind these
            a @ a
        h.add(words)
        h.finish()
    keep = {} if drop_out else {k: h.out[k] for k in ('psino', 'fan', 'ssr')}
    del h
    # blocks of the session's sizes on the first stream, while the side stream works
    busy = not side.query()
    new = [torch.full((n,), -7, dtype=torch.int64 if k in ('zR', 'zM') else torch.int32,
                      device='cuda') for k, n in sizes.items()]
    given = [ptrs[t.data_ptr()] for t in new if t.data_ptr() in ptrs]
    assert not busy or not given, given
    torch.cuda.synchronize()
    assert all(bool((t == -7).all()) for t in new)
    for k, v in keep.items():
        assert torch.equal(v, ref.out[k]), k
