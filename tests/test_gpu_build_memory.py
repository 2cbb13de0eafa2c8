"""The working memory that the index builder keeps: bounded, given back on request, never shared by two builds."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from galn_amd import native as nv

pytestmark = pytest.mark.gpu


def _codes(seed, n):
    return np.random.default_rng(seed).integers(0, 4, n).astype(np.uint8)


def test_a_finished_build_keeps_one_arena_until_it_is_given_back():
    import torch
    print("case build memory", flush=True)
    nv.build_bwt(_codes(1, 1000), 0)  # (the library's own static memory is there from its first kernel on)
    nv.build_trim()
    free0 = torch.cuda.mem_get_info()[0]
    for n in (2_000_000, 3_000_000, 1_000_000):
        m, words, _, _ = nv.build_bwt(_codes(1, n), 0)
    held = free0 - torch.cuda.mem_get_info()[0]
    assert held < 40 * 6_000_000, held  # the largest build's alone, 34 bytes a suffix (free memory counts whole pages)
    with nv.Index(words, m, 0):  # (opening an index frees nothing: that time would be the caller's)
        assert nv.build_trim() >= 34 * 6_000_000
        assert nv.build_trim() == 0
    assert free0 - torch.cuda.mem_get_info()[0] < 32 << 20
    nv.build_bwt(_codes(2, 20_000_000), 0)  # 1.36 GB: too large to be kept
    assert nv.build_trim() == 0


def test_builds_side_by_side_equal_builds_alone():
    print("case builds side by side", flush=True)
    sizes = [3_000, 900_001, 2_500_000, 50_000, 2_500_001, 1_200_000]
    alone = [nv.build_bwt(_codes(i, n), 0, want_sa=True) for i, n in enumerate(sizes)]
    got = [[None] * len(sizes) for _ in range(3)]

    def run(t):
        for k in range(len(sizes)):
            i = (k + 2 * t) % len(sizes)
            got[t][i] = nv.build_bwt(_codes(i, sizes[i]), 0, want_sa=True)
            if t == 2:
                nv.build_trim()

    threads = [threading.Thread(target=run, args=(t,)) for t in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for row in got:
        for a, b in zip(alone, row):
            assert int(a[0].primary) == int(b[0].primary)
            np.testing.assert_array_equal(a[1], b[1])
            np.testing.assert_array_equal(a[2], b[2])
