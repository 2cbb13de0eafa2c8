"""A server slot allocates for a full launch before its first one: later launches of other reads and options
allocate nothing that shows."""
from __future__ import annotations

import numpy as np
import pytest

from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth

pytestmark = pytest.mark.gpu


# the first launch: unseeded reads, enough of them that fewer waves run than seeded reads get; or a few short ones
@pytest.mark.parametrize("first", [(70_000, 30, ["-l", "1024", "-n", "0.01", "-o", "2"]), (2_000, 30, []), (1, 36, ["-n", "1", "-o", "0"])])
def test_later_launches_fit_what_the_first_one_reserved(first):
    import torch
    print(f"case server memory {first[:2]}", flush=True)
    rng = np.random.default_rng(4)
    ref = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, 200_000)]
    prim, last = ix.bwt_from_forward(ix.encode_forward(ref))
    L2, words = ix.pack_bwt(last)
    meta = {"primary": prim, "L2": list(L2), "seq_len": int(last.size), "bwt_size": int(words.size)}

    def request(n, length, opts):
        reads = ref[rng.integers(0, ref.size - length, n)[:, None] + np.arange(length)]
        lens = np.full(n, length, np.int32)
        q, qoff = synth.encode_queries(reads, lens)
        batch = np.zeros(n, np.int32)
        bopts, nst, md = nv.prepare_batches(nv.gap_opt_from_args(opts), lens, batch)
        return q, qoff, lens, md, batch, bopts, nst

    with nv.Index(words, meta, 0) as idx, nv.Server(idx, max_launch_reads=70_000, slots=1) as srv:
        free = []
        for r in (first, (6_000, 250, []), (6_000, 256, ["-n", "3", "-o", "2", "-e", "20", "-l", "1024"]), (70_000, 100, [])):
            rid = srv.submit(*request(*r))
            srv.wait(rid)
            res, _ = srv.result(rid)
            assert (res.n_aln >= 1).all()
            free.append(torch.cuda.mem_get_info()[0])
    assert free[0] - min(free) < 64 << 20, [f >> 20 for f in free]
