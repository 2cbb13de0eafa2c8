"""The autotuner searches only with settings that act on the search."""
from __future__ import annotations

import numpy as np
import pytest

from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth

pytestmark = pytest.mark.gpu


def test_no_trials_of_the_lanes_settings_where_no_lane_runs(capfd, monkeypatch):
    print("case autotune 2000 reads", flush=True)
    rng = np.random.default_rng(12)
    ref = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, 300_000)]
    prim, last = ix.bwt_from_forward(ix.encode_forward(ref))
    L2, words = ix.pack_bwt(last)
    meta = {"primary": prim, "L2": list(L2), "seq_len": int(last.size), "bwt_size": int(words.size)}
    n = 2000
    lens = np.full(n, 100, np.int32)
    reads = ref[rng.integers(0, ref.size - 100, n)[:, None] + np.arange(100)].copy()
    reads[np.arange(n), rng.integers(0, 100, n)] = ord("A")
    q, qoff = synth.encode_queries(reads, lens)
    batch = np.zeros(n, np.int32)
    bopts, nst, md = nv.prepare_batches(nv.gap_opt_from_args([]), lens, batch)
    monkeypatch.setenv("GALN_HIP_VERBOSE", "1")
    with nv.Index(words, meta, 0) as idx:
        rs = nv.ReadSet(idx, q, qoff, lens, md, batch, bopts, nst)
        rs.search()
        before = rs.results()
        capfd.readouterr()
        tuned = rs.autotune()
        trials = capfd.readouterr().err.count("autotune: cutoff")
        if tuned["heavy_pops"] == 1:  # every read to the wave engine: eight cutoffs and no more
            assert trials == 8
            assert tuned["block_threads"] == 64 and tuned["waves_per_cu"] == tuned["rec_per_lane"] == tuned["chunks_per_lane"] == 0
        else:
            assert trials == 15
        rs.search(nv.FORM_BATCHED, 0, nv.Tune(sort_by_cost=1, heavy_pops=1))
        # the field of the former variant of five waves is accepted, and the search is the same one
        one = rs.results()
        rs.search(nv.FORM_BATCHED, 0, nv.Tune(sort_by_cost=1, heavy_pops=1, heavy_waves_per_simd=5))
        five = rs.results()
        rs.search()
        after = rs.results()
        for got in (one, five, after):
            np.testing.assert_array_equal(got.n_aln, before.n_aln)
            np.testing.assert_array_equal(got.pops, before.pops)
            np.testing.assert_array_equal(got.rec, before.rec)
        rs.close()
