"""The stack pool of an index's first search: as large as a full grid of waves can take on a repeat-rich genome,
since a pool that runs dry while the reads run costs that search several times its time."""
from __future__ import annotations

import numpy as np
import pytest

from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth

pytestmark = pytest.mark.gpu


def test_the_first_search_allocates_512_granules_for_each_wave():
    import torch
    print("case first pool", flush=True)
    rng = np.random.default_rng(8)
    ref = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, 50_000)]
    m, words, _, _ = nv.build_bwt(ix.encode_forward(ref), 0)
    nv.build_trim()
    n = 6000
    lens = np.full(n, 36, np.int32)
    reads = ref[rng.integers(0, ref.size - 36, n)[:, None] + np.arange(36)]
    q, qoff = synth.encode_queries(reads, lens)
    batch = np.zeros(n, np.int32)
    bopts, nst, md = nv.prepare_batches(nv.gap_opt_from_args(["-l", "1024", "-n", "1", "-o", "0"]), lens, batch)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    with nv.Index(words, m, 0) as idx:
        for k in (16, n):  # (a small request takes a small pool)
            rs = nv.ReadSet(idx, q[:36 * k], qoff[:k], lens[:k], md[:k], batch[:k], bopts, nst)
            free = torch.cuda.mem_get_info()[0]
            rs.search(nv.FORM_BATCHED)
            taken = free - torch.cuda.mem_get_info()[0]
            assert (rs.results().n_aln >= 1).all()
            rs.close()
            waves = min(k, 12 * cus)  # at least 12 a CU
            assert taken >= waves * 512 * 16384 and (k > 16 or taken < 1 << 30), taken
