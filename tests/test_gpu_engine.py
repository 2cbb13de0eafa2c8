"""The wave engine's launches, at the settings where their seams are: reads parked by the one-wave launch
and gone on with by workgroups of four waves (GALN_HIP_TEST_PARK_POPS parks them after that many pops)
give the reference's .sai, pops, traces and the oracle-checked byte counts.
"""
from __future__ import annotations

import numpy as np
import pytest

import fixtures as fx
from conftest import golden_inputs, load_reads, run_opts
from galn_amd import index as ix
from galn_amd import native as nv

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
