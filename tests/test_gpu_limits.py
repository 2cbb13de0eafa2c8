"""What lies outside the kernels' limits is refused read by read, the same in every form and engine."""
from __future__ import annotations

import numpy as np
import pytest

from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("field,value", [("max_gape", -1), ("max_gapo", 127), ("max_gape", 256)])
def test_options_beyond_the_limits_are_refused_in_every_form(field, value):
    print(f"case limits {field}={value}", flush=True)
    rng = np.random.default_rng(3)
    ref = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, 5000)]
    prim, last = ix.bwt_from_forward(ix.encode_forward(ref))
    L2, words = ix.pack_bwt(last)
    meta = {"primary": prim, "L2": list(L2), "seq_len": int(last.size), "bwt_size": int(words.size)}
    n = 70
    lens = np.full(n, 40, np.int32)
    reads = np.stack([ref[a:a + 40] for a in rng.integers(0, ref.size - 40, n)])
    q, qoff = synth.encode_queries(reads, lens)
    # two batches: the second one's options are ordinary
    batch = (np.arange(n) >= 35).astype(np.int32)
    bopts, nst, md = nv.prepare_batches(nv.gap_opt_from_args([]), lens, batch)
    setattr(bopts[0], field, value)
    arrays = (q, qoff, lens, md, batch, bopts, nst)
    with nv.Index(words, meta, 0) as idx:
        rs = nv.ReadSet(idx, *arrays)
        for form, tune in ((nv.FORM_PLAIN, None), (nv.FORM_BATCHED, None), (nv.FORM_BATCHED, nv.Tune(sort_by_cost=1, heavy_pops=64)),
                           (nv.FORM_BATCHED, nv.Tune(sort_by_cost=1, heavy_pops=-1))):
            for flags in (0, nv.GALN_HIP_TRACE):
                rs.search(form, flags, tune)
                got = rs.results().n_aln
                assert (got[:35] == -5).all() and (got[35:] >= 1).all()
        rs.close()
        rc, _, got = _noalloc(idx, arrays, 0)
        assert rc == 0, nv.last_error()
        assert (got.n_aln[:35] == -5).all() and (got.n_aln[35:] >= 1).all()
