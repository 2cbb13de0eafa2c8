"""The wave engine's launches, at the settings where their seams are: reads parked by the one-wave launch
and gone on with by workgroups of four waves (GALN_HIP_TEST_PARK_POPS parks them after that many pops)
give the reference's .sai, pops, traces and the oracle-checked byte counts.
"""
from __future__ import annotations

import numpy as np
import pytest

import fixtures as fx
import oracle as orc
from conftest import golden_inputs, load_reads, run_opts
from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth

pytestmark = pytest.mark.gpu


def _readset(index, w, key):
    opts, mate = run_opts(w["meta"], key)
    r = load_reads(w["reads"][mate])
    o = nv.gap_opt_from_args(opts)
    bopts, nst, md = nv.prepare_batches(o, r["qlen"], r["batch"])
    return o, nv.ReadSet(index, r["query"], r["qoff"], r["qlen"], md, r["batch"], bopts, nst)


@pytest.mark.parametrize("park", ["1", "40", "700"])
@pytest.mark.parametrize("name,key", [("adna_mixed", "adna_1"), ("deep_repeats", "deep_1"), ("serving_mix", "default_1"),
                                      ("options", "max_entries_m300_1"), ("human_like", "adna_1")])
def test_parked_reads_give_the_golden_results(name, key, park, golden_dir, monkeypatch):
    print(f"case park {name}/{key} after {park}", flush=True)
    w = golden_inputs(name, golden_dir)
    meta, words = ix.read_bwt(w["bwt"])
    tune = nv.Tune(sort_by_cost=1, heavy_pops=1)
    exp = w["expected"]
    with nv.Index(words, meta, 0) as idx:
        o, rs = _readset(idx, w, key)
        monkeypatch.setenv("GALN_HIP_TEST_PARK_POPS", "0")
        rs.search(nv.FORM_BATCHED, 0, tune)
        whole = rs.results(want_pops=True, want_bytes=True)
        monkeypatch.setenv("GALN_HIP_TEST_PARK_POPS", park)
        for flags in (0, nv.GALN_HIP_TRACE, nv.GALN_HIP_GRAPH, nv.GALN_HIP_GRAPH):
            rs.search(nv.FORM_BATCHED, flags, tune)
            trace = flags == nv.GALN_HIP_TRACE
            res = rs.results(want_pops=True, want_bytes=True, want_trace=trace)
            np.testing.assert_array_equal(res.n_aln, exp[key + "_n_aln"])
            np.testing.assert_array_equal(res.pops, exp[key + "_pops"])
            np.testing.assert_array_equal(res.occ_bytes, whole.occ_bytes)
            np.testing.assert_array_equal(res.rec, whole.rec)
            if trace:
                np.testing.assert_array_equal(res.trace, exp[key + "_trace"])
        assert fx.md5_bytes(nv.sai_bytes(o, res.n_aln, res.rec_off, res.rec)) == w["meta"]["runs"][key]["sai_md5"]
        rs.close()


def _search_both(refseq, reads, lens, opts, form=nv.FORM_BATCHED, flags=0):
    """The batched form's results of ASCII reads, and the oracle's."""
    prim, last = ix.bwt_from_forward(ix.encode_forward(refseq))
    L2, words = ix.pack_bwt(last)
    meta = {"primary": prim, "L2": list(L2), "seq_len": int(last.size), "bwt_size": int(words.size)}
    q, qoff = synth.encode_queries(reads, lens)
    n = lens.size
    batch = np.zeros(n, np.int32)
    o = orc.parse_aln_opts(opts)
    bo, ns, md = orc.batch_options(o, lens, batch)
    exp = orc.search(words, meta, q, qoff, lens, md, batch, bo, ns, o["seed_len"], 8)
    bopts, nst, mdx = nv.prepare_batches(nv.gap_opt_from_args(opts), lens, batch)
    with nv.Index(words, meta, 0) as idx:
        rs = nv.ReadSet(idx, q, qoff, lens, mdx, batch, bopts, nst)
        rs.search(form, flags)
        got = rs.results(want_pops=True, want_bytes=True)
        rs.close()
    return got, exp


# the root chain's kept steps (127) and a round's (60) with one more and one fewer, the smallest reads, an N
# at either end and inside the descent, pushes that fill a bucket's ranks (equal penalties)
@pytest.mark.parametrize("length", [1, 2, 59, 61, 62, 126, 127, 128, 129, 190, 260])
@pytest.mark.parametrize("opts", [["-n", "2", "-o", "1", "-l", "1024", "-M", "5", "-O", "5", "-E", "5", "-d", "0", "-i", "0"],
                                  ["-n", "0", "-o", "0", "-l", "20"], ["-n", "2", "-o", "1", "-l", "20", "-k", "1", "-m", "40"]])
@pytest.mark.parametrize("cap", ["", "128"])
def test_root_chain_and_walked_descents(length, opts, cap, monkeypatch):
    print(f"case root {length} {opts} cap {cap}", flush=True)
    if cap:
        monkeypatch.setenv("GALN_HIP_TEST_PUSH_CAP", cap)
    rng = np.random.default_rng(length)
    ref = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, 12_000)]
    n = 40
    at = rng.integers(0, ref.size - length, n)
    reads = np.stack([ref[a:a + length] for a in at])
    for i in range(n):
        for p in rng.integers(0, length, i % 4):
            reads[i, p] = ord("ACGT"[int(rng.integers(0, 4))])
    reads[3, 0] = reads[7, length - 1] = reads[11, length // 2] = ord("N")
    lens = np.full(n, length, np.int32)
    got, exp = _search_both(ref, reads, lens, opts)
    np.testing.assert_array_equal(got.n_aln, exp.n_aln)
    np.testing.assert_array_equal(got.pops, exp.pops)
    np.testing.assert_array_equal(got.occ_bytes, exp.occ_bytes)
    for i in range(n):
        np.testing.assert_array_equal(got.records(i), exp.records(i))
