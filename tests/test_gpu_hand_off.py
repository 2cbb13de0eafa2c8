"""The hand-off slots of the wave engine: a slot holds a root chain only where a read can have one, and
reads without a chain or without a slot give the same results."""
from __future__ import annotations

import numpy as np
import pytest

import fixtures as fx
from conftest import golden_inputs, load_reads, run_opts
from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("share", [0.9, 0.5, 0.1, 0.0])
@pytest.mark.parametrize("name,key", [("adna_mixed", "adna_1"), ("plain_small", "default_1"), ("serving_mix", "default_1")])
def test_golden_results_with_fewer_slots(name, key, share, golden_dir, monkeypatch):
    print(f"case hand-off {name}/{key} share {share}", flush=True)
    w = golden_inputs(name, golden_dir)
    opts, mate = run_opts(w["meta"], key)
    r = load_reads(w["reads"][mate])
    o = nv.gap_opt_from_args(opts)
    bopts, nst, md = nv.prepare_batches(o, r["qlen"], r["batch"])
    meta, words = ix.read_bwt(w["bwt"])
    n, most = int(r["qlen"].size), int(r["qlen"].max())
    # of what slots with root chains take at most: all without chains, or some of the reads
    monkeypatch.setenv("GALN_HIP_TEST_HAND_BYTES", str(int(share * n * (4 + 2 * (most + 1) + min(most, 127)) * 8)))
    exp = w["expected"]
    with nv.Index(words, meta, 0) as idx:
        rs = nv.ReadSet(idx, r["query"], r["qoff"], r["qlen"], md, r["batch"], bopts, nst)
        for form, flags, cutoff in ((nv.FORM_BATCHED, 0, None), (nv.FORM_PLAIN, 0, None), (nv.FORM_BATCHED, 0, 64),
                                    (nv.FORM_BATCHED, nv.GALN_HIP_GRAPH, 1)):
            rs.search(form, flags, None if cutoff is None else nv.Tune(sort_by_cost=1, heavy_pops=cutoff))
            res = rs.results()
            np.testing.assert_array_equal(res.n_aln, exp[key + "_n_aln"])
            np.testing.assert_array_equal(res.pops, exp[key + "_pops"])
            assert fx.md5_bytes(nv.sai_bytes(o, res.n_aln, res.rec_off, res.rec)) == w["meta"]["runs"][key]["sai_md5"]
        rs.close()


def test_slots_of_short_reads_hold_no_root_chain():
    """Device memory that a search takes for each further read: the slot (97 words for 60 bp and a seed of 32
    with no chain, 60 more with one), a few bytes of scan space beside it."""
    import torch
    print("case hand-off bytes a read", flush=True)
    rng = np.random.default_rng(6)
    ref = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, 100_000)]
    prim, last = ix.bwt_from_forward(ix.encode_forward(ref))
    L2, words = ix.pack_bwt(last)
    meta = {"primary": prim, "L2": list(L2), "seq_len": int(last.size), "bwt_size": int(words.size)}
    n = 600_000
    lens = np.full(n, 60, np.int32)
    reads = ref[rng.integers(0, ref.size - 60, n)[:, None] + np.arange(60)]
    q, qoff = synth.encode_queries(reads, lens)
    bopts, nst, md = nv.prepare_batches(nv.gap_opt_from_args(["-n", "1", "-o", "0"]), lens, np.zeros(n, np.int32))
    with nv.Index(words, meta, 0) as idx:
        def taken(m):
            rs = nv.ReadSet(idx, q[:60 * m], qoff[:m], lens[:m], md[:m], np.zeros(m, np.int32), bopts, nst)
            free = torch.cuda.mem_get_info()[0]
            rs.search(nv.FORM_BATCHED)
            free -= torch.cuda.mem_get_info()[0]
            assert (rs.results().n_aln >= 1).all()
            rs.close()
            return free

        taken(n)  # (the index's stack pool)
        per_read = (taken(n) - taken(n // 2)) / (n - n // 2)
    slot = (1 + 61 + 33 + 2) * 8
    assert slot * 0.9 < per_read < slot + 32, per_read
