"""Many read sets at once, made and freed by several threads (each with an index of its own): what a search
reads back belongs to its read set."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth

pytestmark = pytest.mark.gpu


def test_read_sets_of_several_threads_keep_their_results():
    print("case read sets, 3 threads", flush=True)
    rng = np.random.default_rng(21)
    ref = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, 60_000)]
    m, words, _, _ = nv.build_bwt(ix.encode_forward(ref), 0)

    def reads(n, length, opts):
        r = ref[rng.integers(0, ref.size - length, n)[:, None] + np.arange(length)].copy()
        r[np.arange(n), rng.integers(0, length, n)] = ord("G")
        lens = np.full(n, length, np.int32)
        q, qoff = synth.encode_queries(r, lens)
        batch = np.zeros(n, np.int32)
        return (q, qoff, lens, *(lambda p: (p[2], batch, p[0], p[1]))(nv.prepare_batches(nv.gap_opt_from_args(opts), lens, batch)))

    # (reads of 10 bp outgrow their record slots: re-runs, counted by what is read back)
    sets = [reads(200, 50, []), reads(3, 10, ["-n", "3", "-o", "0", "-N"]), reads(1, 80, []), reads(700, 36, ["-l", "1024", "-n", "2"])]
    bad = []

    def run(t):
        with nv.Index(words, m, 0) as idx:
            alone = []
            for s in sets:
                rs = nv.ReadSet(idx, *s)
                rs.search(nv.FORM_BATCHED)
                alone.append((rs.results(want_bytes=True), sum(x["algo_bytes"] for x in rs.launches())))
                rs.close()
            for rep in range(4):
                live = [nv.ReadSet(idx, *sets[(i + t) % 4]) for i in range(12)]
                for rs in live:
                    rs.search(nv.FORM_BATCHED)
                for i, rs in enumerate(live):
                    exp, algo = alone[(i + t) % 4]
                    got = rs.results(want_bytes=True)
                    same = all(np.array_equal(getattr(got, k), getattr(exp, k)) for k in ("n_aln", "pops", "occ_bytes", "rec"))
                    if not same or sum(x["algo_bytes"] for x in rs.launches()) != algo:
                        bad.append((t, rep, i))
                    rs.close()

    threads = [threading.Thread(target=run, args=(t,)) for t in range(3)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad, bad
