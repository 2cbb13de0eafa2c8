"""The untraced kernels of indexes of 2^32 symbols or more, which an ordinary search of such an index runs
(GALN_HIP_TEST_EPOCH counts a small index in epochs): every form gives the reference's .sai and pops, and
the byte counts of the search of the same index without epochs."""
from __future__ import annotations

import numpy as np
import pytest

import fixtures as fx
from conftest import golden_inputs, load_reads, run_opts
from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth
from test_zz_no_alloc import _in_order, _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("epoch", ["1", "5"])
@pytest.mark.parametrize("name,key", [("adna_mixed", "adna_1"), ("deep_repeats", "deep_1"), ("serving_mix", "default_1"),
                                      ("options", "max_entries_m300_1"), ("human_like", "adna_1")])
def test_untraced_search_on_an_index_of_many_epochs(name, key, epoch, golden_dir, monkeypatch):
    print(f"case untraced epochs {name}/{key} epoch={epoch}", flush=True)
    w = golden_inputs(name, golden_dir)
    opts, mate = run_opts(w["meta"], key)
    r = load_reads(w["reads"][mate])
    o = nv.gap_opt_from_args(opts)
    bopts, nst, md = nv.prepare_batches(o, r["qlen"], r["batch"])
    arrays = (r["query"], r["qoff"], r["qlen"], md, r["batch"], bopts, nst)
    meta, words = ix.read_bwt(w["bwt"])
    exp = w["expected"]
    with nv.Index(words, meta, 0) as idx:
        rs = nv.ReadSet(idx, *arrays)
        rs.search(nv.FORM_BATCHED)
        narrow = rs.results(want_bytes=True)
        rs.close()
    monkeypatch.setenv("GALN_HIP_TEST_EPOCH", epoch)
    with nv.Index(words, meta, 0) as idx:
        rs = nv.ReadSet(idx, *arrays)
        # (64: k_search hands reads over with their widths; parked after one pop, the four-wave kernel goes on with every read)
        for form, flags, cutoff, park in ((nv.FORM_PLAIN, 0, None, None), (nv.FORM_BATCHED, 0, None, None), (nv.FORM_BATCHED, 0, 64, None),
                                          (nv.FORM_BATCHED, 0, -1, None), (nv.FORM_BATCHED, 0, 1, "1"), (nv.FORM_BATCHED, 0, 64, "100"),
                                          (nv.FORM_BATCHED, nv.GALN_HIP_GRAPH, 1, "40"), (nv.FORM_BATCHED, nv.GALN_HIP_GRAPH, 64, "40")):
            print(f"  form {form} flags {flags} cutoff {cutoff} park {park}", flush=True)
            with monkeypatch.context() as m:
                if park:
                    m.setenv("GALN_HIP_TEST_PARK_POPS", park)
                rs.search(form, flags, None if cutoff is None else nv.Tune(sort_by_cost=1, heavy_pops=cutoff))
            got = rs.results(want_bytes=True)
            np.testing.assert_array_equal(got.n_aln, exp[key + "_n_aln"])
            np.testing.assert_array_equal(got.pops, exp[key + "_pops"])
            np.testing.assert_array_equal(got.occ_bytes, narrow.occ_bytes)
            np.testing.assert_array_equal(got.rec, narrow.rec)
            assert fx.md5_bytes(nv.sai_bytes(o, got.n_aln, got.rec_off, got.rec)) == w["meta"]["runs"][key]["sai_md5"]
        rs.close()
        rc, _, got = _noalloc(idx, arrays, 0)
        assert rc == 0, nv.last_error()
        off, rec = _in_order(got, r["qlen"].size)
        np.testing.assert_array_equal(got.pops, exp[key + "_pops"])
        assert fx.md5_bytes(nv.sai_bytes(o, got.n_aln, off, rec)) == w["meta"]["runs"][key]["sai_md5"]


@pytest.mark.parametrize("length", [40, 64, 100])
def test_many_unseeded_reads_with_and_without_epochs(length, monkeypatch):
    """65,536 unseeded reads and more get fewer waves, above 2^32 symbols by their mean length: the same results."""
    print(f"case many unseeded reads of {length}", flush=True)
    rng = np.random.default_rng(length)
    ref = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, 400_000)]
    m, words, _, _ = nv.build_bwt(ix.encode_forward(ref), 0)
    n = 70_000
    lens = np.full(n, length, np.int32)
    lens[::7] -= 1
    reads = ref[rng.integers(0, ref.size - length, n)[:, None] + np.arange(length)].copy()
    reads[np.arange(n), rng.integers(0, length - 1, n)] = ord("C")
    q, qoff = synth.encode_queries(reads, lens)
    batch = np.zeros(n, np.int32)
    bopts, nst, md = nv.prepare_batches(nv.gap_opt_from_args(["-l", "1024", "-n", "2", "-o", "1"]), lens, batch)
    got = []
    for epoch in ("", "5"):
        monkeypatch.setenv("GALN_HIP_TEST_EPOCH", epoch)
        with nv.Index(words, m, 0) as idx:
            rs = nv.ReadSet(idx, q, qoff, lens, md, batch, bopts, nst)
            rs.search(nv.FORM_BATCHED)
            got.append(rs.results(want_bytes=True))
            rs.close()
    a, b = got
    for x, y in ((a.n_aln, b.n_aln), (a.pops, b.pops), (a.occ_bytes, b.occ_bytes), (a.rec, b.rec)):
        np.testing.assert_array_equal(x, y)
