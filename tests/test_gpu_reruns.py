"""Reads with more records than a wave's slots: the re-runs give 16 times more, so a search takes as many
re-runs as that needs and no record count is too many."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as orc
from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu

# reads of 10 bp with 4 mismatches have some 6,500 records on this genome, those of 12 bp some 1,100: past
# the 256 slots of the first launch, on either side of the 4,096 of the first re-run
REF_BP = 200_000


@pytest.fixture(scope="module")
def genome():
    ref = np.frombuffer(b"ACGT", np.uint8)[np.random.default_rng(5).integers(0, 4, REF_BP)]
    prim, last = ix.bwt_from_forward(ix.encode_forward(ref))
    L2, words = ix.pack_bwt(last)
    meta = {"primary": prim, "L2": list(L2), "seq_len": int(last.size), "bwt_size": int(words.size)}
    with nv.Index(words, meta, 0) as idx:
        yield ref, words, meta, idx


@pytest.mark.parametrize("lengths", [(12,), (10,), (10, 12)])
@pytest.mark.parametrize("form", [nv.FORM_PLAIN, nv.FORM_BATCHED])
def test_reads_of_thousands_of_records(lengths, form, genome):
    print(f"case records {lengths} form {form}", flush=True)
    ref, words, meta, idx = genome
    rng = np.random.default_rng(9)
    n = 12
    lens = np.array([lengths[i % len(lengths)] for i in range(n)], np.int32)
    reads = np.stack([ref[a:a + 12] for a in rng.integers(0, REF_BP - 12, n)])
    q, qoff = synth.encode_queries(reads, lens)
    batch = np.zeros(n, np.int32)
    opts = ["-n", "4", "-o", "0", "-N"]
    o = orc.parse_aln_opts(opts)
    bo, ns, md = orc.batch_options(o, lens, batch)
    exp = orc.search(words, meta, q, qoff, lens, md, batch, bo, ns, o["seed_len"], 8)
    assert exp.n_aln.min() > 256 and (exp.n_aln.max() > 24 * 256) == (10 in lengths)
    bopts, nst, mdx = nv.prepare_batches(nv.gap_opt_from_args(opts), lens, batch)
    rs = nv.ReadSet(idx, q, qoff, lens, mdx, batch, bopts, nst)
    rs.search(form)
    got = rs.results(want_pops=True)
    tiers = [ln["tier"] for ln in rs.launches()]
    rs.close()
    np.testing.assert_array_equal(got.n_aln, exp.n_aln)
    np.testing.assert_array_equal(got.pops, exp.pops)
    for i in range(n):
        np.testing.assert_array_equal(got.records(i), exp.records(i))
    # 256 slots, then 4,096, then 65,536; and once more where the output arena (65,536 records) was full
    reruns = 1 + int(exp.n_aln.max() > 4096) + int(exp.n_aln.sum() > 65536)
    assert [t for t in tiers if t > 10] == [11 + i for i in range(reruns)]


def test_noalloc_gives_a_read_the_record_slots_that_fit(monkeypatch):
    """122k records in an array cut to 40 MB, where 65,536 slots are too few and 16 times more do not fit."""
    print("case 122k records", flush=True)
    monkeypatch.setenv("GALN_HIP_TEST_NA_BYTES", str(40 << 20))
    ref = np.frombuffer(b"ACGT", np.uint8)[np.random.default_rng(5).integers(0, 4, 4_000_000)]
    m, words, _, _ = nv.build_bwt(ix.encode_forward(ref), 0)
    lens = np.array([11, 40], np.int32)
    reads = np.stack([ref[a:a + 40] for a in (1000, 2000)])
    q, qoff = synth.encode_queries(reads, lens)
    batch = np.array([0, 1], np.int32)
    sets = [["-n", "5", "-o", "0", "-N", "-l", "1024"], []]
    meta = {"primary": int(m.primary), "L2": [int(v) for v in m.L2], "seq_len": int(m.seq_len), "bwt_size": int(words.size)}
    o = orc.parse_aln_opts(sets[0])
    bo, ns, md = orc.batch_options(o, lens[:1], batch[:1])
    exp = orc.search(words, meta, q[:11], qoff[:1], lens[:1], md, batch[:1], bo, ns, o["seed_len"], 8)
    assert 65536 < exp.n_aln[0] < 1 << 20
    per = [nv.prepare_batches(nv.gap_opt_from_args(s), lens[i:i + 1], np.zeros(1, np.int32)) for i, s in enumerate(sets)]
    bopts = (nv.SearchOpt * 2)(per[0][0][0], per[1][0][0])
    nst, mdx = (np.concatenate([p[k] for p in per]) for k in (1, 2))
    with nv.Index(words, m, 0) as idx:
        rc, n_rec, got = _noalloc(idx, (q, qoff, lens, mdx, batch, bopts, nst), 0, rec_cap=1 << 18)
        assert rc == 0, nv.last_error()
        np.testing.assert_array_equal(got.records(0), exp.records(0))
        assert got.n_aln[1] >= 1 and n_rec == got.n_aln.sum() and got.pops[0] == exp.pops[0]
