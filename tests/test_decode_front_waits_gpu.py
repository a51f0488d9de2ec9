"""Workgroups of the one-launch attention half (decode_front.hip) that wait in vain: what other launches on the GPU keep from being started
is made by whoever waits for it, with the same bits."""
import threading

import numpy as np
import pytest
import torch

from test_decode_front_gpu import _layers, ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,nh,nkv,hd,B,lens", [
    (2048, 32, 4, 64, 16, [600]),                                   # two parts, one row: the output tiles look past the caches only
    (2048, 32, 4, 64, 16, [2048, 0, 1025, 1537, 128, 257, 512, 2]),   # four parts, parts without tokens, a padding row, eight rows
    (320, 5, 1, 64, 8, [449, 1, 448]),                               # odd group, K slices of unequal length
    (64, 2, 2, 64, 24, [100, 23]),                                   # one query head a KV head, a product of one unit of K
    (256, 7, 1, 128, 32, [1, 640, 33]),
    (512, 8, 1, 128, 16, [1100, 20]),                                # the most query heads of 128: every wave rotates q, the last two k and v too
])
def test_made_by_who_waits(ops, H, nh, nkv, hd, B, lens):
    """No wait at all: attention workgroups that come before q make it, output tiles make everything.  Every bit of the stream, of what the norm
    leaves and of the pages is as without."""
    run, _, _ = _layers(ops, H, nh, nkv, hd, B, lens, 3, seed=H + hd + len(lens), scaled_first=len(lens) % 2 == 0)
    want = run(True)
    assert all(np.isfinite(a).all() for a in want)
    for polls in (0, 1):
        assert all(np.array_equal(a, b) for a, b in zip(run(True, polls), want)), polls


def test_two_streams_at_once(ops):
    """Two threads with a stream each launch attention halves whose waiting workgroups fill the GPU together: the results are those of one alone."""
    cases = [(2048, 32, 4, 64, 16, [2048, 700, 1025, 1537, 128, 257, 512, 2]), (4096, 32, 8, 128, 16, [900, 3, 1200, 77])]
    runs = [_layers(ops, *c, 4, seed=7 + i)[0] for i, c in enumerate(cases)]
    wants = [run(True) for run in runs]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for n in range(12):
                got = runs[i](True)
                if not all(np.array_equal(a, b) for a, b in zip(got, wants[i])):
                    bad.append((i, n))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_many_short_heads_keep_three_launches(ops):
    """Heads of 64 with more than 192 pairs of a row and a KV head, in more than one part each: the one launch was up to 5 % slower."""
    parts = ops.decode_front_parts
    assert parts(8, 2048, 32, 32, 64, 16, 513) == 0 and parts(7, 2048, 32, 32, 64, 16, 2048) == 0
    assert parts(8, 2048, 32, 32, 64, 16, 512) == 1 and parts(6, 2048, 32, 32, 64, 16, 2048) == 4
    assert parts(8, 4096, 32, 32, 128, 16, 2048) == 4 and parts(8, 2048, 32, 16, 64, 16, 2048) == 4
