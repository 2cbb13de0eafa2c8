"""The stack pool of an index's first search: as many granules as the searches of so many reads can take on a
repeat-rich genome (a pool that runs dry while the reads run costs that search several times its time), and few for
few reads, and for seeded ones (handing out and taking back tens of gigabytes costs seconds in some phases)."""
from __future__ import annotations

import numpy as np
import pytest

from galn_amd import index as ix
from galn_amd import native as nv
from galn_amd import synth

pytestmark = pytest.mark.gpu

GIB = 1 << 30


@pytest.fixture(scope="module")
def small():
    rng = np.random.default_rng(8)
    ref = np.frombuffer(b"ACGT", np.uint8)[rng.integers(0, 4, 50_000)]
    m, words, _, _ = nv.build_bwt(ix.encode_forward(ref), 0)
    nv.build_trim()
    return ref, m, words


# granules of 16 KB (and 260 bytes of links): 32 a wave and 4 for each read more; the scratch of a full grid is 1.1 GB
@pytest.mark.parametrize("args,n,least,most", [
    (["-l", "1024"], 1, 1 << 10, GIB),
    (["-l", "1024"], 16, 1 << 10, GIB),
    (["-l", "1024"], 6000, 6000 * 4 + 3072 * 28, 7 * GIB),
    (["-l", "1024"], 600_000, 1 << 21, 40 * GIB),
    ([], 2000, 1 << 16, 3 * GIB),
    ([], 600_000, 1 << 19, 13 * GIB),
    (["-k", "4"], 600_000, 1 << 21, 40 * GIB),  # (its seeds hold nothing back)
    (["-l", "33"], 600_000, 1 << 21, 40 * GIB),
])
def test_a_first_search_takes_a_pool_by_its_reads(small, args, n, least, most):
    import torch
    print("case first pool", args, n, flush=True)
    ref, m, words = small
    rng = np.random.default_rng(9)
    lens = np.full(n, 36, np.int32)
    reads = ref[rng.integers(0, ref.size - 36, n)[:, None] + np.arange(36)]
    q, qoff = synth.encode_queries(reads, lens)
    batch = np.zeros(n, np.int32)
    bopts, nst, md = nv.prepare_batches(nv.gap_opt_from_args(["-n", "1", "-o", "0"] + args), lens, batch)
    with nv.Index(words, m, 0) as idx:
        rs = nv.ReadSet(idx, q, qoff, lens, md, batch, bopts, nst)
        free = torch.cuda.mem_get_info()[0]
        rs.search(nv.FORM_BATCHED)
        taken = free - torch.cuda.mem_get_info()[0]
        assert (rs.results().n_aln >= 1).all()
        rs.close()
        assert least * 16384 <= taken < most, taken
