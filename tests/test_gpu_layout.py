"""The device index layout at its edges, and indexes counted in epochs.

* An index of 2^32 symbols or more keeps 32-bit counts per epoch of blocks; GALN_HIP_TEST_EPOCH makes
  the epochs a few blocks long, so that the fixtures' indexes span many of them: searches give the
  reference's .sai, pops and traces, in every engine.
* Texts whose lengths fall on and around the layout's word and block edges: positions of every row equal
  the suffix array, with and without epochs.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import fixtures as fx
from conftest import golden_inputs, load_reads, run_opts
from galn_amd import index as ix
from galn_amd import native as nv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heavy_pops", [-1, 0, 1])
@pytest.mark.parametrize("name,key", [("adna_mixed", "adna_1"), ("deep_repeats", "deep_1"), ("serving_mix", "default_1"),
                                      ("options", "max_entries_m300_1")])
def test_search_on_an_index_of_many_epochs(name, key, heavy_pops, golden_dir, monkeypatch):
    print(f"case epochs {name}/{key} heavy_pops={heavy_pops}", flush=True)
    monkeypatch.setenv("GALN_HIP_TEST_EPOCH", "5")  # 4096 symbols
    w = golden_inputs(name, golden_dir)
    opts, mate = run_opts(w["meta"], key)
    r = load_reads(w["reads"][mate])
    o = nv.gap_opt_from_args(opts)
    bopts, nst, md = nv.prepare_batches(o, r["qlen"], r["batch"])
    meta, words = ix.read_bwt(w["bwt"])
    with nv.Index(words, meta, 0) as idx:
        rs = nv.ReadSet(idx, r["query"], r["qoff"], r["qlen"], md, r["batch"], bopts, nst)
        rs.search(nv.FORM_BATCHED, nv.GALN_HIP_TRACE, nv.Tune(sort_by_cost=1, heavy_pops=heavy_pops))
        res = rs.results(want_pops=True, want_trace=True)
        rs.close()
    exp = w["expected"]
    np.testing.assert_array_equal(res.n_aln, exp[key + "_n_aln"])
    np.testing.assert_array_equal(res.pops, exp[key + "_pops"])
    np.testing.assert_array_equal(res.trace, exp[key + "_trace"])
    assert fx.md5_bytes(nv.sai_bytes(o, res.n_aln, res.rec_off, res.rec)) == w["meta"]["runs"][key]["sai_md5"]


@pytest.mark.parametrize("epoch", ["", "1"])
@pytest.mark.parametrize("L", [1, 15, 16, 17, 63, 64, 65, 127, 128, 192, 4096])
def test_positions_at_word_and_block_edges(L, epoch, monkeypatch):
    print(f"case layout L={L} epoch={epoch}", flush=True)
    monkeypatch.setenv("GALN_HIP_TEST_EPOCH", epoch)
    f2 = np.random.default_rng(100 + L).integers(0, 4, L).astype(np.uint8)
    m, words, sa, _ = nv.build_bwt(f2, 0, want_sa=True)
    f = torch.as_tensor(f2, dtype=torch.uint8)
    ref = ix.suffix_array(torch.cat([f, (3 - f).flip(0)])).numpy().astype(np.uint64)
    with nv.Index(words, m, 0) as index:
        index.set_sa(sa)
        pos = index.sa_positions(np.arange(int(m.seq_len) + 1))
    np.testing.assert_array_equal(pos, np.concatenate([[np.uint64(2**64 - 1)], ref]))
