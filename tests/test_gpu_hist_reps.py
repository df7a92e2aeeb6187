"""Replicate histograms: lane groups of every size against one-replicate
sessions, with chunks that start at any place of a word quad (exact)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('btp', [0, 2])
@pytest.mark.parametrize('nrep,cuts', [(2, (0, 1, 70001)), (3, (0, 2)), (4, (0, 3, 8195)),
                                       (16, (0, 8192)), (17, (0, 63, 64)), (33, (0, 4097))])
def test_replicates_equal_single_sessions(params, nrep, cuts, btp):
    import torch

    from nipet_amd.lm.lmsim import synth_lm
    from nipet_amd.lm.mmrhist import LmHistogram, tag_range
    w = synth_lm(params, 3, 60, seed=9)
    tf, tl = tag_range(w)
    nitag = (tl - tf + 999) // 1000

    def run(n, rep0, at):
        h = LmHistogram(params, tf, nitag, btp=btp, seed=77, nrep=n, rep0=rep0)
        for i, j in zip(at, at[1:] + (len(w),)):
            h.add(w[i:j])
        h.finish()
        return h.out

    big = run(nrep, 5, cuts)
    for r in {0, 1, nrep // 2, nrep - 1}:
        one = run(1, 5 + r, (0,))
        for k in ('psino', 'dsino', 'phc', 'dhc'):
            assert torch.equal(big[k][:, r], one[k][:, 0]), (r, k)
        if r == 0:
            for k in ('ssr', 'zR', 'zM', 'pvs', 'fan', 'bck'):
                assert torch.equal(big[k], one[k]), k
