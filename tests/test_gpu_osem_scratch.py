"""A reconstruction keeps scratch for two images only while sensitivity images are
pending, also where another stream than the state's own runs the iteration."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('how', ['iteration', 'other stream', 'property'])
def test_scratch_for_two_images_is_given_back(params, how):
    import torch

    import nipet_amd as nip
    from nipet_amd import _lib
    from nipet_amd.prj.osem import osem_iteration, osem_prepare
    subs = [np.asarray(nip.get_subsets14(k, params)[0], np.int32) for k in range(2)]
    g = torch.Generator(device='cuda').manual_seed(5)
    one = torch.ones((68516, 837), device='cuda')
    p = torch.randint(0, 9, (68516, 837), generator=g, device='cuda', dtype=torch.int32)

    def state():
        return osem_prepare(params, p.to(torch.uint16), one, one, one, subsets=subs)

    st = state()
    n = max(len(s) for s in subs)
    sizes = [_lib.lib().nipet_bprj_scratch(st.geom.handle, n, nb) for nb in (1, 2)]
    assert st.scratch.numel() == sizes[1] > 1.9 * sizes[0]
    img = torch.ones((320, 320, 127), device='cuda')
    if how == 'property':
        sens = st.sens
        assert bool((sens > 0).any())
    else:
        stream = torch.cuda.Stream() if how == 'other stream' else torch.cuda.current_stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            osem_iteration(st, img)
            # blocks of the buffer's size, while the stream may still work
            with torch.cuda.stream(torch.cuda.default_stream()):
                torch.empty(sizes[1], dtype=torch.uint8, device='cuda').fill_(255)
            osem_iteration(st, img, first_full=False)
        torch.cuda.current_stream().wait_stream(stream)
        ref, want = state(), torch.ones_like(img)
        ref.sens  # (one image at a time)
        for k in range(2):
            osem_iteration(ref, want, first_full=k == 0)
        assert float((img - want).abs().max()) <= 1e-4 * float(want.max())
    assert st.scratch.numel() == sizes[0] and not st.pending
