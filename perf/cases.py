"""The calls whose time matters to a user of this framework, from one small request to a block of
two million reads, through the public entry points of `galn_amd.native`.

A case is one call (or one request's few calls) on one genome with one kind of reads:

  path    what is called
            request     reload the reads of a read set, search (batched form), results: new reads
                        each time, as a program that answers requests does
            batched     search (batched form) and results of reads already on the device
            replay      the same with the captured graph and a tuning found before, as a program
                        does that searches read set after read set of one kind
            plain       search (plain form) and results of reads already on the device
            device      the search that allocates nothing, on the caller's device tensors
            serve       requests of several sizes, lengths and options through the serving loop
            positions   text positions of BWT rows (the step after the search)
            build       the .bwt and SA samples of a new genome
  genome  uniform (i.i.d. bases), adna (41% GC, a tenth duplicated, runs of N), repeats (45%
          interspersed repeats of 50 families), copies (8 diverged copies of one sequence)
  bp, n   bases of the genome; reads (rows for positions)
  lo, hi  read lengths: lognormal of median 45 within [lo, hi] with `lens` "adna", else uniform
  opts    aln options: default, adna (-l 1024 -n 0.01 -o 2), deep (-n 0.04 -o 2 -e 6 -k 2)

A genome is fixed by its kind and size and is indexed once, as a program keeps its index open; the
reads are drawn from the seed. Outputs are whole numbers (record counts, records, pop counts, text
positions, index words): they are right or wrong, there is no rounding to allow for.
"""
from __future__ import annotations

import collections
import ctypes as C
import math

import numpy as np
import torch

from galn_amd import native as nv

OPTS = {"default": [], "adna": ["-l", "1024", "-n", "0.01", "-o", "2"], "deep": ["-n", "0.04", "-o", "2", "-e", "6", "-k", "2"]}
BATCH = 0x40000  # reads of one bwa batch
RECORDS = 4      # records a read that the callers' arrays have room for


def _case(name, path, genome, bp, n, lo=100, hi=100, lens="uniform", opts="default"):
    c = {"path": path, "genome": genome, "bp": bp, "n": n, "lo": lo, "hi": hi, "lens": lens, "opts": opts}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one small request on a small genome: launches, copies and one read's own latency
        _case("request_16", "request", "uniform", 5_000_000, 16),
        # the plain small workload (5 Mbp, 100k reads of 100 bp, bwa's default options), both forms
        _case("plain_100k", "plain", "uniform", 5_000_000, 100_000),
        _case("batched_100k", "batched", "uniform", 5_000_000, 100_000),
        # the same reads where the caller may not allocate; an odd count
        _case("device_30k", "device", "uniform", 5_000_000, 30_011),
        # a new genome of that size: what `galn index` does
        _case("build_5M", "build", "uniform", 5_000_000, 1),
        # ancient DNA on 100 Mbp: a request of an odd size, one bwa batch, and a large read set searched
        # the way the benchmark searches it
        _case("request_4k_adna", "request", "adna", 100_000_000, 4001, 30, 150, "adna", "adna"),
        _case("batched_262k_adna", "batched", "adna", 100_000_000, BATCH, 30, 150, "adna", "adna"),
        _case("replay_2M_adna", "replay", "adna", 100_000_000, 2_000_000, 30, 150, "adna", "adna"),
        # the rows of a large .sai to text positions
        _case("positions_1M", "positions", "adna", 100_000_000, 1_000_000),
        # requests of 1k to 32k reads of 30 to 250 bp, default and ancient DNA options in turn
        _case("serve_6", "serve", "adna", 100_000_000, 65_000, 30, 250),
        # long pairs against a genome of near copies: deep backtracking with gaps
        _case("batched_pairs", "batched", "copies", 100_000_000, 100_000, 150, 150, "uniform", "deep"),
        # an index far beyond the caches, repeats, reads of all lengths
        _case("batched_repeats", "batched", "repeats", 700_000_000, 100_003, 30, 150, "uniform", "adna"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["request", "request", "batched", "batched", "batched", "replay", "plain", "device", "positions", "build"])
    if path == "build":
        return _case(None, path, "uniform", _log(rng, 50_000, 20_000_000), 1)
    if path == "positions":
        return _case(None, path, rng.choice(["uniform", "adna"]), _log(rng, 1_000_000, 100_000_000), _log(rng, 1000, 4_000_000))
    if path in ("plain", "device"):  # one thread per read to its end: reads that do not backtrack for long
        length = rng.randint(36, 125)
        return _case(None, path, "uniform", _log(rng, 1_000_000, 50_000_000), _log(rng, 100, 100_000), length, length)
    kind = rng.choice(["uniform", "adna", "adna", "copies", "repeats"])
    bp = _log(rng, 1_000_000, 100_000_000)
    n = _log(rng, 1, 10_000) if path == "request" else _log(rng, 10_000, BATCH)
    if kind == "copies":
        return _case(None, path, kind, bp, min(n, 100_000), 100, 150, "uniform", "deep")
    if kind == "uniform":
        length = rng.randint(36, 150)
        return _case(None, path, kind, bp, n, length, length)
    if rng.random() < 0.3:
        return _case(None, path, kind, bp, n, 30, rng.randint(100, 150), "uniform", "default")
    return _case(None, path, kind, bp, n, 30, rng.randint(100, 150), "adna", "adna")


# --------------------------------------------------------------------------
# genomes, as 2-bit codes on the device (4 = N), and their indexes


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _bases(g, n, gc):
    out = torch.empty(n, dtype=torch.uint8, device="cuda")
    for s in range(0, n, 1 << 27):
        u = torch.rand(min(1 << 27, n - s), generator=g, device="cuda")
        out[s:s + u.numel()] = (u >= (1 - gc) / 2).byte() + (u >= 0.5).byte() + (u >= 1 - (1 - gc) / 2).byte()
    return out


def _substitute(g, s, rate):
    """Each base replaced by another one with probability `rate` (a number, or one per base)."""
    hit = torch.rand(s.numel(), generator=g, device="cuda") < rate
    shift = torch.randint(1, 4, (s.numel(),), generator=g, device="cuda", dtype=torch.uint8)
    return torch.where(hit & (s < 4), (s + shift) & 3, s)


def _adna_genome(g, bp):
    s = _bases(g, bp, 0.41)
    rng = np.random.default_rng(bp)
    done = 0
    while done < bp // 10:  # duplicated segments of 300 bp to 5 kb at 0-5% divergence
        seg = int(rng.integers(300, 5001))
        src, dst = (int(x) for x in rng.integers(0, bp - seg, 2))
        s[dst:dst + seg] = _substitute(g, s[src:src + seg].clone(), float(rng.uniform(0, 0.05)))
        done += seg
    done = 0
    while done < bp // 100:  # runs of N
        run = int(rng.integers(100, 5001))
        at = int(rng.integers(0, bp - run))
        s[at:at + run] = 4
        done += run
    return s


def _repeats_genome(g, bp):
    """Unique sequence and copies of 50 repeat families at 2-20% divergence, in turn; 45% repeats."""
    rng = np.random.default_rng(bp)
    fam_len = rng.integers(300, 6001, 50)
    fam_at = np.concatenate([[0], np.cumsum(fam_len)[:-1]])
    fam = _bases(g, int(fam_len.sum()), 0.41)
    out = torch.empty(bp, dtype=torch.uint8, device="cuda")
    for s in range(0, bp, 1 << 25):
        m = min(1 << 25, bp - s)
        k = m // 2000 + 16
        f = rng.integers(0, 50, k)
        cut = (rng.random(k) * fam_len[f] / 3).astype(np.int64)
        rep = fam_len[f] - cut
        gap = np.maximum(rng.exponential(rep.mean() * 55 / 45, k).astype(np.int64), 1)
        size = torch.from_numpy(np.stack([gap, rep], 1).reshape(-1)).cuda()
        start = torch.cumsum(size, 0) - size
        seg = torch.repeat_interleave(torch.arange(size.numel(), device="cuda"), size)[:m]
        if seg.numel() < m:  # (the drawn segments fell short of the piece: unique sequence to its end)
            seg = torch.cat([seg, torch.zeros(m - seg.numel(), dtype=seg.dtype, device="cuda")])
        off = torch.arange(m, device="cuda") - start[seg]
        base = torch.from_numpy(np.stack([np.full(k, -1), fam_at[f] + cut], 1).reshape(-1)).cuda()
        rate = torch.from_numpy(np.stack([np.zeros(k), rng.uniform(0.02, 0.2, k)], 1).reshape(-1).astype(np.float32)).cuda()
        at = base[seg]
        piece = torch.where(at < 0, _bases(g, m, 0.41), fam[torch.where(at < 0, 0, at + off).clamp_(0, fam.numel() - 1)])
        out[s:s + m] = _substitute(g, piece, rate[seg])
    return out


def _copies_genome(g, bp):
    """8 copies of a random sequence at 1-3% substitutions and 0.2% indels of 1-3 bp."""
    rng = np.random.default_rng(bp)
    base = _bases(g, bp // 8, 0.5)
    parts = []
    for _ in range(8):
        s = _substitute(g, base, float(rng.uniform(0.01, 0.03)))
        u = torch.rand(s.numel(), generator=g, device="cuda")
        more = torch.randint(1, 4, (s.numel(),), generator=g, device="cuda")
        times = torch.where(u < 0.001, 0, torch.where(u < 0.002, 1 + more, 1))
        c = torch.repeat_interleave(s, times)
        new = torch.repeat_interleave(u >= 0.001, times) & (torch.repeat_interleave(u, times) < 0.002)
        parts.append(torch.where(new, _bases(g, c.numel(), 0.5), c))
    return torch.cat(parts)


def _genome(kind, bp):
    g = _gen(bp)
    if kind == "adna":
        return _adna_genome(g, bp)
    if kind == "repeats":
        return _repeats_genome(g, bp)
    return _copies_genome(g, bp) if kind == "copies" else _bases(g, bp, 0.5)


def _forward(codes):
    """2-bit codes for the builder: N becomes a fixed pseudo-random base."""
    fill = _bases(_gen(11), codes.numel(), 0.5)
    return torch.where(codes > 3, fill, codes).cpu().numpy()


class _Genome:
    """A genome's bases on the device and its open index (and, once asked for, a server on an index
    of its own: a server owns its index)."""

    def __init__(self, kind, bp):
        self.codes = _genome(kind, bp)
        self.meta, self.words, sa, _ = nv.build_bwt(_forward(self.codes), 0, want_sa=True)
        self.index = nv.Index(self.words, self.meta, 0)
        self.index.set_sa(sa)
        self._server = None

    def server(self):
        if self._server is None:
            self._server = nv.Server(nv.Index(self.words, self.meta, 0))
        return self._server


_OPEN = collections.OrderedDict()  # the genomes used last: (kind, bp) -> _Genome


def _open(kind, bp):
    if (kind, bp) not in _OPEN:
        while len(_OPEN) >= 2:
            _OPEN.popitem(last=False)
        _OPEN[kind, bp] = _Genome(kind, bp)
    _OPEN.move_to_end((kind, bp))
    return _OPEN[kind, bp]


# --------------------------------------------------------------------------
# reads


def _reads(codes, seed, n, lo, hi, lens, opts):
    """What a ReadSet takes: queries (the reads' reverse complements), offsets, lengths, and the
    options derived from them. Reads come from both strands. Those searched with the ancient DNA
    options are deaminated at both ends and hold 0.5% substitutions (with "adna" lengths one in twenty
    is unrelated to the genome); the others hold 1% (2% with the deep options) substitutions and, one
    time in ten, an indel of 1 to 3 bp."""
    rng = np.random.default_rng([seed, n])
    g = _gen(seed * 1_000_003 + n)
    if lens == "adna":
        qlen = np.clip(np.rint(np.exp(rng.normal(math.log(45), 0.45, n))), lo, hi).astype(np.int32)
    else:
        qlen = rng.integers(lo, hi + 1, n).astype(np.int32)
    parts = []
    for s in range(0, n, 1 << 18):
        ql = torch.from_numpy(qlen[s:s + (1 << 18)].astype(np.int64)).cuda()
        m = ql.numel()
        start = (torch.rand(m, generator=g, device="cuda", dtype=torch.float64) * (codes.numel() - hi - 8)).long()
        col = torch.arange(hi, device="cuda").expand(m, hi)
        off = col
        if opts != "adna":  # an indel: the bases from a random place on come from 1 to 3 bp further on, or back
            u = torch.rand(m, 2, generator=g, device="cuda")
            size = torch.randint(1, 4, (m,), generator=g, device="cuda") * torch.where(u[:, 0] < 0.05, 1, torch.where(u[:, 0] < 0.1, -1, 0))
            off = col + torch.where(col >= (u[:, 1] * ql).long()[:, None], size[:, None], 0)
        r = codes[(start[:, None] + off).clamp_(0, codes.numel() - 1)]
        r = _substitute(g, r.reshape(-1), 0.005 if opts == "adna" else 0.02 if opts == "deep" else 0.01).reshape(m, hi)
        flip = torch.rand(m, generator=g, device="cuda") < 0.5
        back = (ql[:, None] - 1 - col).clamp_(0)
        rc = r.gather(1, back)
        r = torch.where(flip[:, None], torch.where(rc > 3, rc, 3 - rc), r)
        if opts == "adna":
            other = torch.rand(m, generator=g, device="cuda") < (0.05 if lens == "adna" else 0.0)
            r = torch.where(other[:, None], _bases(g, m * hi, 0.41).reshape(m, hi), r)
            p5 = 0.3 * 0.5 ** col.float()
            r = torch.where((r == 1) & (torch.rand(m, hi, generator=g, device="cuda") < p5), torch.full_like(r, 3), r)
            p3 = 0.3 * 0.5 ** (ql[:, None] - 1 - col).clamp_(0).float()
            r = torch.where((r == 2) & (torch.rand(m, hi, generator=g, device="cuda") < p3), torch.zeros_like(r), r)
        q = r.gather(1, back)  # the query: the read reversed and complemented
        q = torch.where(q > 3, q, 3 - q)
        parts.append(q[col < ql[:, None]].cpu().numpy())
    qoff = np.zeros(n, np.uint64)
    qoff[1:] = np.cumsum(qlen[:-1])
    batch = (np.arange(n) // BATCH).astype(np.int32)
    bopts, nst, md = nv.prepare_batches(nv.gap_opt_from_args(OPTS[opts]), qlen, batch)
    return np.concatenate(parts), qoff, qlen, md, batch, bopts, nst


def _pinned(shape, dtype):
    size = int(np.prod(shape)) * np.dtype(dtype).itemsize
    return torch.zeros(size, dtype=torch.uint8, pin_memory=True).numpy().view(dtype).reshape(shape)


# --------------------------------------------------------------------------
# the calls


def prepare(case, seed):
    s = {"path": case["path"]}
    if case["path"] == "build":
        s["fwd"] = _forward(_bases(_gen(seed), case["bp"], 0.5))
        return s
    G = s["genome"] = _open(case["genome"], case["bp"])
    if case["path"] == "positions":
        rng = np.random.default_rng([seed, case["n"]])
        s["rows"] = rng.integers(0, int(G.meta.seq_len) + 1, case["n"]).astype(np.uint64)
        s["ref_len"] = rng.integers(30, 151, case["n"]).astype(np.int32)
        return s
    if case["path"] == "serve":
        s["server"] = G.server()
        sizes = [max(1, round(case["n"] * 2.0 ** -(k + 1))) for k in range(6)]
        s["requests"] = [_reads(G.codes, seed * 8 + k, n, case["lo"], min(case["hi"], 100 if k % 2 else 250), "adna" if k % 2 else "uniform",
                                "adna" if k % 2 else "default") for k, n in enumerate(sizes)]
        return s
    reads = _reads(G.codes, seed, case["n"], case["lo"], case["hi"], case["lens"], case["opts"])
    if case["path"] == "device":
        put = lambda a, t: torch.from_numpy(a.view(t)).cuda()  # noqa: E731
        q, qoff, qlen, md, batch, bopts, nst = reads
        n = case["n"]
        s["in"] = [put(q, np.uint8), put(qoff, np.int64), put(qlen, np.int32), put(md, np.int32), put(batch, np.int32)]
        s["n_aln"] = torch.zeros(n, dtype=torch.int32, device="cuda")
        s["off"] = torch.zeros(n, dtype=torch.int64, device="cuda")
        s["pops"] = torch.zeros(n, dtype=torch.int64, device="cuda")
        s["rec"] = torch.zeros((RECORDS * n + 4096, 3), dtype=torch.int64, device="cuda")
        s["out"] = torch.zeros_like(s["rec"])
        s["opts"] = (bopts, nst)
        return s
    s["reads"] = reads
    s["set"] = nv.ReadSet(G.index, *reads)
    s["out"] = s["set"].result_buffers(want_pops=True, rec_cap=RECORDS * case["n"] + 4096, alloc=_pinned)
    if case["path"] == "replay":  # the tuning that the autotuner picks for ancient DNA read sets
        s["tune"] = nv.Tune(sort_by_cost=1, heavy_pops=1)
    return s


def _device_search(s):
    R, O = nv.Reads(), nv.Out()
    bopts, nst = s["opts"]
    R.n_reads, R.n_batches = s["n_aln"].numel(), nst.size
    R.query, R.qoff, R.qlen, R.max_diff, R.batch = (t.data_ptr() for t in s["in"])
    R.bopts, R.n_stacks = C.cast(bopts, C.c_void_p), nst.ctypes.data
    O.n_aln, O.rec_off, O.n_pops = s["n_aln"].data_ptr(), s["off"].data_ptr(), s["pops"].data_ptr()
    O.rec, O.rec_cap = s["rec"].data_ptr(), s["rec"].shape[0]
    rc = nv.hip_lib().galn_hip_search_device_noalloc(s["genome"].index.h, C.byref(R), C.byref(O), 0)
    if rc != 0:
        raise nv.GalnError(f"search_device_noalloc failed ({rc}): {nv.last_error()}")
    # reads' records lie in no set order: put them in read order
    count = s["n_aln"].clamp(min=0).long()
    total = int(O.n_rec)
    first = torch.cumsum(count, 0) - count
    at = torch.repeat_interleave(s["off"] - first, count, output_size=total) + torch.arange(total, device="cuda")
    s["out"][:total] = s["rec"][at]
    return [s["n_aln"], s["pops"], s["out"]]


def run(s):
    path = s["path"]
    if path == "build":
        meta, words, sa, _ = nv.build_bwt(s["fwd"], 0, want_sa=True)
        return [int(meta.primary), words.view(np.int32), sa.view(np.int64)]
    if path == "positions":
        pos, strand = s["genome"].index.sa_positions(s["rows"], s["ref_len"])
        return [pos.view(np.int64), strand]
    if path == "device":
        return _device_search(s)
    if path == "serve":
        srv = s["server"]
        ids = [srv.submit(*r) for r in s["requests"]]
        out = []
        for i in ids:
            srv.wait(i)
            r = srv.result(i)[0]
            rec = np.zeros((RECORDS * r.n_aln.size + 4096, 3), np.int64)
            rec[:len(r.rec)] = r.rec.view(np.int64)
            out.append([r.n_aln, r.pops.view(np.int64), rec])
        return out
    rs = s["set"]
    if path == "request":
        rs.reload(*s["reads"])
    if path == "plain":
        rs.search(nv.FORM_PLAIN)
    elif path == "replay":
        rs.search(nv.FORM_BATCHED, nv.GALN_HIP_GRAPH, s["tune"])
    else:
        rs.search(nv.FORM_BATCHED)
    r = rs.results(out=s["out"])
    # (the whole record array, zeros after the last record: one shape for any reads)
    return [r.n_aln, r.pops.view(np.int64), s["out"]["rec"].view(np.int64)]


def work(case):
    """Index bytes of the occurrence queries that bwa's search performs for these reads (64 for each
    distinct block of a query; the library counts them), beside the reads and records. Positions: the
    LF steps to a sampled row, 15.5 blocks on average. A build: its input and output. No
    floating-point work."""
    n = case["n"]
    if case["path"] == "build":
        return {"bytes": case["bp"] * (1 + 2 / 4 + 2 / 4), "flops": 0}
    if case["path"] == "positions":
        return {"bytes": n * (15.5 * 64 + 8 + 8 + 8 + 4 + 4), "flops": 0}
    s = prepare(dict(case, path="batched"), 1) if case["path"] != "serve" else prepare(case, 1)
    G = s["genome"]
    total = 0
    for reads in s.get("requests") or [s["reads"]]:
        rs = nv.ReadSet(G.index, *reads)
        rs.search(nv.FORM_BATCHED)
        r = rs.results(want_bytes=True)
        total += int(r.occ_bytes.sum()) + reads[0].size + 36 * rs.n + 24 * len(r.rec)
        rs.close()
    return {"bytes": total, "flops": 0}


def exact(case, seed):
    """No floating outputs: every value is a whole number, the same or wrong."""
    return None
