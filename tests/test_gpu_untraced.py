"""The untraced kernels, which run the steps of exact descents side by side, against the traced ones, which do
not: the same records, pops and byte counts on reads of all lengths, and again when run again."""
from __future__ import annotations

import numpy as np
import pytest

from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def genome():
    ref = synth.adna_reference(11, 3_000_000)
    f2 = ix.encode_forward(ref)
    m, words, _, _ = nv.build_bwt(f2, 0)
    with nv.Index(words, m, 0) as idx:
        yield ref, idx


@pytest.mark.parametrize("opts", [[], ["-l", "1024", "-n", "0.01", "-o", "2"], ["-n", "0.04", "-o", "2", "-e", "6", "-k", "2"],
                                  ["-n", "3", "-o", "1", "-e", "3", "-l", "20", "-k", "1", "-M", "5", "-O", "5", "-E", "5"],
                                  ["-n", "4", "-o", "2", "-l", "1024", "-m", "300"]])
def test_untraced_equals_traced_and_itself(opts, genome):
    print(f"case untraced {opts}", flush=True)
    ref, idx = genome
    rng = np.random.default_rng(len(opts))
    n, longest = 30_000, 200
    lens = rng.integers(25, longest + 1, n).astype(np.int32)
    reads = np.asarray(ref)[rng.integers(0, len(ref) - longest, n)[:, None] + np.arange(longest)].copy()
    hit = rng.random(reads.shape) < 0.015
    reads[hit] = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, int(hit.sum()))]
    q, qoff = synth.encode_queries(reads, lens)
    batch = np.zeros(n, np.int32)
    bopts, nst, md = nv.prepare_batches(nv.gap_opt_from_args(opts), lens, batch)
    rs = nv.ReadSet(idx, q, qoff, lens, md, batch, bopts, nst)
    rs.search(nv.FORM_BATCHED, nv.GALN_HIP_TRACE)
    exp = rs.results(want_bytes=True)
    for form, flags in ((nv.FORM_BATCHED, 0), (nv.FORM_BATCHED, 0), (nv.FORM_BATCHED, nv.GALN_HIP_GRAPH), (nv.FORM_PLAIN, 0)):
        rs.search(form, flags)
        got = rs.results(want_bytes=True)
        np.testing.assert_array_equal(got.n_aln, exp.n_aln)
        np.testing.assert_array_equal(got.pops, exp.pops)
        np.testing.assert_array_equal(got.occ_bytes, exp.occ_bytes)
        np.testing.assert_array_equal(got.rec, exp.rec)
    rs.close()
