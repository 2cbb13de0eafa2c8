"""A .bwt body's trailing words: the totals after the last block with symbols are the header's, whatever the
body holds there or whether it holds them at all (texts that fill their last block, where a position at the
text's end is counted past it)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as orc
from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("epoch", ["", "1", "3"])
@pytest.mark.parametrize("bp", [64, 192, 8192 + 64])
def test_positions_and_searches_do_not_depend_on_the_trailing_words(bp, epoch, monkeypatch):
    print(f"case tail {bp} bp epoch={epoch}", flush=True)
    monkeypatch.setenv("GALN_HIP_TEST_EPOCH", epoch)
    rng = np.random.default_rng(bp)
    ref = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, bp)]
    m, words, sa, _ = nv.build_bwt(ix.encode_forward(ref), 0, want_sa=True)
    n, length = 40, 36
    reads = ref[rng.integers(0, bp - length, n)[:, None] + np.arange(length)].copy()
    reads[::3, 11] = ord("A")
    lens = np.full(n, length, np.int32)
    q, qoff = synth.encode_queries(reads, lens)
    batch = np.zeros(n, np.int32)
    opts = ["-n", "2", "-o", "1", "-l", "1024"]
    o = orc.parse_aln_opts(opts)
    bo, ns, md = orc.batch_options(o, lens, batch)
    meta = {"primary": int(m.primary), "L2": [int(v) for v in m.L2], "seq_len": int(m.seq_len), "bwt_size": int(words.size)}
    exp = orc.search(words, meta, q, qoff, lens, md, batch, bo, ns, o["seed_len"], 4)
    bopts, nst, mdx = nv.prepare_batches(nv.gap_opt_from_args(opts), lens, batch)
    rows = np.arange(2 * bp + 1)
    pos = None
    for body in (words, words[:-8], words[:-4], np.concatenate([words[:-8], np.full(8, 0xffffffff, np.uint32)])):
        meta["bwt_size"] = int(body.size)
        with nv.Index(body, meta, 0) as idx:
            idx.set_sa(sa)
            got = idx.sa_positions(rows)
            if pos is None:
                pos = got
                assert (np.sort(got[1:]) == np.arange(2 * bp, dtype=np.uint64)).all()
            np.testing.assert_array_equal(got, pos)
            rs = nv.ReadSet(idx, q, qoff, lens, mdx, batch, bopts, nst)
            for tune in (None, nv.Tune(sort_by_cost=1, heavy_pops=-1)):
                rs.search(nv.FORM_BATCHED, 0, tune)
                res = rs.results(want_bytes=True)
                np.testing.assert_array_equal(res.n_aln, exp.n_aln)
                np.testing.assert_array_equal(res.pops, exp.pops)
                np.testing.assert_array_equal(res.occ_bytes, exp.occ_bytes)
                for i in range(n):
                    np.testing.assert_array_equal(res.records(i), exp.records(i))
            rs.close()
