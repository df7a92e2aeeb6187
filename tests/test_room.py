"""A library call whose device allocation failed is tried once more after torch
has given back the memory that it only keeps; other codes are returned as
they are."""
import pytest

from nipet_amd import _lib


@pytest.mark.parametrize('codes,rc,calls,emptied', [([0], 0, 1, 0), ([-3, 0], 0, 2, 1),
                                                    ([-3, -3], -3, 2, 1), ([-1], -1, 1, 0)])
def test_with_room(monkeypatch, codes, rc, calls, emptied):
    import torch
    seen = []
    monkeypatch.setattr(torch.cuda, 'empty_cache', lambda: seen.append(len(done)))
    done = []

    def call():
        done.append(codes[len(done)])
        return done[-1]

    assert _lib.with_room(call) == rc and len(done) == calls and len(seen) == emptied
    assert seen in ([], [1])
