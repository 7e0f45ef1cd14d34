"""Timed cases of the k-mer hot path, through the package's public entry points.

Every case is one call chain that a program using the package makes: a
normalization job of one sample, a count with its histogram or dump, a
coverage pass, a read-to-component vote, a batch of components, an Inchworm
run, a fixed k-mer set count, a burst of service jobs.  Reads come from the
package's seeded transcriptome model and lie on the GPU as ASCII (the service
and the single component take host memory, as their callers hold it).  The
context and the reuse of freed device blocks are the program's own, made once.

Sizes: the smallest component of a run holds a few dozen reads, a sample 0.05
to 20 M pairs of 36 to 250 nt.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from trinityrnaseq_amd import api, synth

_CTX = None


def _ctx():
    """The program's one context; jobs take the blocks that earlier jobs freed."""
    global _CTX
    if _CTX is None:
        _CTX = api.Context(0)
        api.thread_cache(96 << 30)
    return _CTX


def listed():
    return [
        # phase 2: one Chrysalis component on its own, the smallest call there is
        {"name": "component_200", "kind": "component", "reads": 200, "read_len": 150, "transcripts": 2},
        # the small single-end sample: 500 transcripts, 200k 76-nt reads, strand unknown
        {"name": "job_se_200k", "kind": "job", "paired": False, "units": 200_000, "read_len": 76,
         "transcripts": 500, "sub_rate": 0.005, "trim": 0.0, "k": 25, "canonical": True},
        # an ordinary paired sample, trimmed by quality: ragged reads
        {"name": "job_pe_2M", "kind": "job", "paired": True, "units": 2_000_003, "read_len": 150,
         "transcripts": 50_000, "sub_rate": 0.01, "trim": 0.15, "k": 25, "canonical": True},
        # the large paired sample
        {"name": "job_pe_20M", "kind": "job", "paired": True, "units": 20_000_000, "read_len": 150,
         "transcripts": 50_000, "sub_rate": 0.01, "trim": 0.0, "k": 25, "canonical": True},
        # jellyfish count + histo of a mid-size sample of 100-nt reads
        {"name": "count_histo_3M", "kind": "count", "units": 1_500_001, "read_len": 101, "transcripts": 50_000,
         "sub_rate": 0.01, "trim": 0.1, "k": 25, "canonical": True, "dump": 0},
        # the same with a strand-specific library and its dump (-L 2) to the host
        {"name": "count_dump_ss_1M", "kind": "count", "units": 500_000, "read_len": 125, "transcripts": 20_000,
         "sub_rate": 0.01, "trim": 0.0, "k": 25, "canonical": False, "dump": 2},
        # fastaToKmerCoverageStats on 2x250 reads: more than 128 windows a read
        {"name": "stats_250nt", "kind": "stats", "units": 600_000, "read_len": 250, "transcripts": 30_000,
         "sub_rate": 0.01, "trim": 0.2, "k": 25, "canonical": True},
        # ReadsToTranscripts: skewed expression, 1.5 % errors, overlapping contig pieces
        {"name": "vote_6M", "kind": "vote", "units": 3_000_000, "read_len": 150, "transcripts": 40_000,
         "sub_rate": 0.015, "trim": 0.0, "k": 25, "canonical": True},
        # phase 2 in one launch: components of power-law sizes
        {"name": "batch_1500", "kind": "batch", "components": 1500, "max_reads": 60_000, "read_len": 150},
        # Inchworm: dictionary load, entropy prune, greedy contigs
        {"name": "inchworm_120k", "kind": "inchworm", "units": 120_000, "read_len": 100, "transcripts": 2000,
         "sub_rate": 0.005},
        # GraphFromFasta's weld 48-mers counted in the reads
        {"name": "welds_2M", "kind": "welds", "units": 1_000_000, "read_len": 150, "transcripts": 50_000,
         "sub_rate": 0.01, "keys": 300_000},
        # the resident service: a burst of uneven samples from pageable host memory
        {"name": "serve_6", "kind": "serve", "samples": 6, "min_pairs": 50_000, "max_pairs": 1_000_000,
         "read_len": 150, "slots": 4},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["component", "job", "job", "job", "count", "count", "stats", "vote", "batch", "inchworm",
                       "welds", "serve"])
    if kind == "component":
        return {"kind": kind, "reads": _logint(rng, 30, 5000), "read_len": rng.randint(60, 151),
                "transcripts": rng.randint(1, 6)}
    if kind == "batch":
        return {"kind": kind, "components": _logint(rng, 20, 2000), "max_reads": _logint(rng, 2000, 60_000),
                "read_len": rng.choice([76, 100, 101, 150])}
    if kind == "serve":
        lo = _logint(rng, 20_000, 200_000)
        return {"kind": kind, "samples": rng.randint(2, 8), "min_pairs": lo, "max_pairs": lo * rng.randint(2, 6),
                "read_len": rng.choice([76, 101, 150]), "slots": rng.randint(2, 5)}
    if kind == "inchworm":
        return {"kind": kind, "units": _logint(rng, 5000, 150_000), "read_len": rng.randint(76, 150),
                "transcripts": _logint(rng, 50, 3000), "sub_rate": round(rng.uniform(0.002, 0.01), 4)}
    c = {"kind": kind, "read_len": rng.randint(50, 151), "transcripts": _logint(rng, 1000, 50_000),
         "sub_rate": round(rng.uniform(0.004, 0.015), 4), "trim": rng.choice([0.0, 0.1, 0.3])}
    if kind == "welds":
        del c["trim"]
        c.update(read_len=rng.randint(76, 151), units=_logint(rng, 20_000, 1_500_000), keys=_logint(rng, 10_000, 500_000))
        return c
    c.update(k=rng.choice([21, 25, 25, 25, 25, 31]), canonical=rng.choice([True, True, True, False]))
    if kind == "job":
        c.update(paired=rng.random() < 0.8, units=_logint(rng, 30_000, 16_000_000))
    elif kind == "count":
        c.update(units=_logint(rng, 30_000, 1_200_000), dump=0)
        if c["units"] < 300_000:
            c["dump"] = rng.choice([0, 1, 2])
    elif kind == "stats":
        c.update(units=_logint(rng, 20_000, 3_000_000), read_len=rng.choice([rng.randint(50, 151), rng.randint(200, 301)]))
        if c["read_len"] > 151:
            c["units"] = min(c["units"], 1_000_000)
    else:  # vote
        c.update(units=_logint(rng, 20_000, 4_000_000))
    return c


# ---------------------------------------------------------------- inputs
_CHUNK = 1 << 20


def _transcriptome(case, seed):
    """Lognormal lengths (median 1.2 kb), a tenth sharing exons with a partner;
    the vote's sample has the skewed expression of the stressed one."""
    return synth.Transcriptome(seed, case["transcripts"], 1, 1200.0, 0.6, 200, 15000, share_frac=0.10,
                               expr_sigma=2.5 if case["kind"] == "vote" else 1.5)


def _ascii_pairs(tx, case, seed):
    """Paired reads on the GPU, (2n, read_len) bytes: left reads, then right reads."""
    n, length = case["units"], case["read_len"]
    out = torch.empty((2 * n, length), dtype=torch.uint8, device="cuda")
    host = np.empty(2 * min(n, _CHUNK) * length, np.uint8)
    for first in range(0, n, _CHUNK):
        m = min(_CHUNK, n - first)
        left, right, _ = synth.pe_reads(tx, m, length, seed=seed, frag_mu=2.0 * length, frag_sd=length / 3.0,
                                        sub_rate=case["sub_rate"], first=first, out=host[:2 * m * length])
        out[first:first + m] = torch.from_numpy(left.reshape(m, length))
        out[n + first:n + first + m] = torch.from_numpy(right.reshape(m, length))
    return out


def _ascii_single(tx, case, seed):
    n, length = case["units"], case["read_len"]
    seq, _ = synth.se_reads(tx, n, length, seed=seed, sub_rate=case["sub_rate"])
    return torch.from_numpy(seq.reshape(n, length)).cuda()


def _trimmed(rows, share, seed):
    """Concatenated reads and their offsets; `share` of the reads cut at their
    3' end, down to a few bases."""
    n, length = rows.shape
    lens = torch.full((n,), length, dtype=torch.int64, device="cuda")
    if share:
        g = torch.Generator(device="cuda").manual_seed(seed)
        cut = torch.rand(n, generator=g, device="cuda") < share
        lens = torch.where(cut, torch.randint(10, length + 1, (n,), generator=g, device="cuda"), lens)
        at = torch.arange(length, device="cuda")
        parts = [rows[i:i + _CHUNK][at < lens[i:i + _CHUNK, None]] for i in range(0, n, _CHUNK)]
        seq = torch.cat(parts)
    else:
        seq = rows.reshape(-1)
    off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(lens, 0, out=off[1:])
    return seq, off


def _sample(case, seed):
    tx = _transcriptome(case, seed)
    rows = _ascii_pairs(tx, case, seed) if case.get("paired", True) else _ascii_single(tx, case, seed)
    seq, off = _trimmed(rows, case.get("trim", 0.0), seed)
    return tx, {"seq": seq, "off": off, "n": rows.shape[0]}


def _reads(s):
    return api.Reads.from_device(_ctx(), s["seq"].data_ptr(), s["off"].data_ptr(), s["n"])


def _count(reads, case):
    est = api.estimate_distinct(_ctx(), reads, case["k"], case["canonical"])
    table = api.Table(_ctx(), case["k"], case["canonical"], int(est * 1.05) + 4096, 0.5)
    table.count(reads)
    return table


def _pieces(tx, per_transcript=3):
    """Contig-like pieces: overlapping thirds of each transcript, and its index."""
    out, comp = [], []
    for i in range(tx.n):
        sq = tx.seq(i)
        for j in range(per_transcript):
            p = sq[j * len(sq) // 3:min(len(sq), (j + 2) * len(sq) // 3)]
            out.append(p)
            comp.append(i)
    return out, np.array(comp, np.uint32)


def _components(case, seed):
    """Reads per component ~ power law (alpha 1.8) from 10 reads up; 1-20
    transcripts of 300-5000 nt; contigs = pieces of each transcript, at most 50."""
    rng = np.random.default_rng(seed)
    n, a, lo, hi = case["components"], 1.8, 10.0, float(case["max_reads"])
    u = np.random.default_rng(n).random(n)  # the sizes are the case's, the sequences the seed's
    sizes = np.maximum(10, ((lo ** (1 - a) + u * (hi ** (1 - a) - lo ** (1 - a))) ** (1 / (1 - a))).astype(np.int64))
    sizes[0] = case["max_reads"]
    reads, contigs, n_contigs = [], [], []
    for c in range(n):
        tx = synth.Transcriptome(seed * 100_003 + c, int(rng.integers(1, 21)), 0, 300, 5000)
        reads.append(synth.se_reads(tx, int(sizes[c]), case["read_len"], seed=seed * 7 + c, sub_rate=0.01)[0])
        mine = []
        for j in range(tx.n):
            t, b0 = tx.seq(j), 0
            for x in sorted(rng.integers(50, max(51, len(t) - 50), size=int(rng.integers(0, 3)))) + [len(t)]:
                if x - b0 >= 30:
                    mine.append(t[b0:x])
                b0 = x
        mine = mine[:50] or [tx.seq(0)]
        contigs += mine
        n_contigs.append(len(mine))
    seq = np.concatenate(reads)
    off = np.arange(int(sizes.sum()) + 1, dtype=np.uint64) * np.uint64(case["read_len"])
    cum = lambda v: np.concatenate([[0], np.cumsum(v)]).astype(np.uint64)  # noqa: E731
    return seq, off, cum(sizes), contigs, cum(n_contigs)


def _weld_keys(tx, n, seed):
    """Distinct canonical 48-mers of the transcripts, as (lo, hi) words."""
    rng = np.random.default_rng(seed)
    lut = np.zeros(256, np.uint8)
    lut[list(b"ACGT")] = range(4)
    rows = []
    for j in rng.permutation(tx.n)[:max(1, n // 48)]:
        t = lut[np.frombuffer(tx.seq(int(j)).encode(), np.uint8)]
        starts = rng.integers(0, len(t) - 47, size=64)
        rows.append(t[starts[:, None] + np.arange(48)])
    c = torch.from_numpy(np.concatenate(rows)).cuda().to(torch.int64)

    def words(x):
        lo = torch.zeros(len(x), dtype=torch.int64, device="cuda")
        hi = torch.zeros_like(lo)
        for i in range(16):
            hi = (hi << 2) | x[:, i]
        for i in range(16, 48):
            lo = (lo << 2) | x[:, i]
        return lo.cpu().numpy().view(np.uint64), hi.cpu().numpy().view(np.uint64)

    (lo, hi), (rlo, rhi) = words(c), words(3 - c.flip(1))
    rc = (rhi < hi) | ((rhi == hi) & (rlo < lo))
    pairs = np.unique(np.stack([np.where(rc, rhi, hi), np.where(rc, rlo, lo)], axis=1), axis=0)
    rng.shuffle(pairs)
    return np.ascontiguousarray(pairs[:n, ::-1])


def prepare(case, seed):
    kind = case["kind"]
    seed = int(seed) % 1_000_003 + 1
    s = {"case": case}
    if kind == "component":
        tx = synth.Transcriptome(seed, case["transcripts"], 0, 300, 5000)
        s["seq"], s["off"] = synth.se_reads(tx, case["reads"], case["read_len"], seed=seed, sub_rate=0.01)
        s["seq"] = s["seq"].tobytes()
        s["contigs"], s["comp"] = _pieces(tx)
        s["cseq"], s["coff"] = api.pack_sequences(s["contigs"])
    elif kind in ("job", "count"):
        _, x = _sample(case, seed)
        s.update(x)
        if kind == "count" and case["dump"]:
            # the program's own arrays for the dictionary: room for a key per window
            room = s["n"] * max(1, case["read_len"] - case["k"] + 1)
            if case["dump"] > 1:
                room = room // 2 + 1
            s["keys"], s["counts"] = np.zeros(room, np.int64), np.zeros(room, np.int32)
        if kind == "job":
            s["stats"] = torch.empty((s["n"], 4), dtype=torch.int64, device="cuda")
            s["selected"] = torch.empty(case["units"], dtype=torch.uint8, device="cuda")
    elif kind == "stats":
        _, x = _sample(case, seed)
        s.update(x)
        s["stats"] = torch.empty((s["n"], 4), dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
        counted = _reads(s)
        s["table"] = _count(counted, case)
        counted.free()
    elif kind == "vote":
        tx, x = _sample(case, seed)
        s.update(x)
        pieces, s["comp"] = _pieces(tx)
        s["contigs"] = api.Reads.from_list(_ctx(), pieces)
        s["votes"] = torch.empty((s["n"], 3), dtype=torch.int32, device="cuda")
    elif kind == "batch":
        seq, off, read_off, contigs, contig_off = _components(case, seed)
        s["reads"] = api.Reads(_ctx(), seq, off)
        s["contigs"] = api.Reads.from_list(_ctx(), contigs)
        s["batch"] = api.Batch(_ctx(), s["reads"], read_off, s["contigs"], contig_off, use_graph=True)
        n = len(off) - 1
        s["stats"] = torch.empty((n, 4), dtype=torch.int64, device="cuda")
        s["votes"] = torch.empty((n, 3), dtype=torch.int32, device="cuda")
    elif kind == "inchworm":
        tx = _transcriptome(case, seed)
        seq, off = synth.se_reads(tx, case["units"], case["read_len"], seed=seed, sub_rate=case["sub_rate"])
        reads = api.Reads(_ctx(), seq, off)
        table = _count(reads, {"k": 25, "canonical": True})
        s["keys"], s["counts"] = table.dump()
        table.free()
        reads.free()
        s["keep"], s["seed_keep"] = _keep(1.0), _keep(1.5)
        # the program's own arrays for the contigs, with room for what the reads' windows can give
        windows = case["units"] * (case["read_len"] - 24)
        s["bases"], s["contigs"] = np.zeros(2 * windows, np.uint8), np.zeros((windows // 4, 3), np.int64)
    elif kind == "welds":
        tx, x = _sample(case, seed)
        s.update(x)
        s["keys"] = _weld_keys(tx, case["keys"], seed)
    else:  # serve
        lo, hi = math.log(case["min_pairs"]), math.log(case["max_pairs"])
        sizes = np.exp(np.linspace(lo, hi, case["samples"])).astype(np.int64)
        np.random.default_rng(case["samples"]).shuffle(sizes)
        s["samples"] = []
        tx = synth.large_transcriptome(seed, 20_000)
        for j, n in enumerate(int(v) for v in sizes):
            buf = np.empty(2 * n * case["read_len"], np.uint8)
            synth.pe_reads(tx, n, case["read_len"], seed=seed + j, out=buf)
            s["samples"].append((buf, np.arange(2 * n + 1, dtype=np.uint64) * np.uint64(case["read_len"]), n))
        s["server"] = api.Server(slots=case["slots"], max_cov=50, hbm_budget_bytes=32 << 30)
    torch.cuda.synchronize()
    return s


_KEEP: dict = {}


def _keep(entropy):
    """The entropy filter's composition table: the same for every sample, built once by the program."""
    if entropy not in _KEEP:
        _KEEP[entropy] = api.entropy_keep_table(25, entropy)
    return _KEEP[entropy]


# ---------------------------------------------------------------- one pass
def _as_int(a):
    """A record array of stats or votes as plain integers, one row per read."""
    word = np.int64 if a.dtype == api.READ_STAT_DTYPE else np.int32
    return a.view(word).reshape(len(a), -1)


def run(state):
    case, ctx = state["case"], _ctx()
    kind = case["kind"]
    if kind == "component":
        reads = api.Reads(ctx, state["seq"], state["off"])
        est = api.estimate_distinct(ctx, reads, 25, True)
        table = api.Table(ctx, 25, True, int(est * 1.05) + 64, 0.5)
        table.count(reads)
        stats = api.read_cov_stats(ctx, table, reads)
        contigs = api.Reads(ctx, state["cseq"], state["coff"])
        ctable = api.CTable(ctx, contigs, state["comp"], 25, True)
        votes = ctable.vote(reads)
        for o in (ctable, contigs, table, reads):
            o.free()
        return {"stats": _as_int(stats), "votes": _as_int(votes)}
    if kind == "job":
        k, n = case["k"], case["units"]
        reads = _reads(state)
        table = _count(reads, case)
        at = state["stats"].data_ptr()
        api.read_cov_stats_d(ctx, table, reads, at, min_count=2)
        out = {"stats": state["stats"]}
        if case["paired"]:
            out["n_selected"] = api.select_pairs_d(ctx, at, at + 32 * n, n, 50, 1, 10000,
                                                   max(0, case["read_len"] - k + 1), state["selected"].data_ptr())
            out["selected"] = state["selected"]
        table.free()
        reads.free()
        return out
    if kind == "count":
        reads = _reads(state)
        table = _count(reads, case)
        out = {"histo": table.histo().view(np.int64)}
        if case["dump"]:
            keys, counts = table.dump(case["dump"])
            state["keys"][:len(keys)], state["counts"][:len(keys)] = keys.view(np.int64), counts.view(np.int32)
            out["n"], out["keys"], out["counts"] = len(keys), state["keys"], state["counts"]
        table.free()
        reads.free()
        return out
    if kind == "stats":
        reads = _reads(state)
        api.read_cov_stats_d(ctx, state["table"], reads, state["stats"].data_ptr(), min_count=2)
        reads.free()
        return state["stats"]
    if kind == "vote":
        reads = _reads(state)
        ctable = api.CTable(ctx, state["contigs"], state["comp"], case["k"], case["canonical"])
        ctable.vote_d(reads, state["votes"].data_ptr())
        ctable.free()
        reads.free()
        return state["votes"]
    if kind == "batch":
        state["batch"].run_d(state["stats"].data_ptr(), state["votes"].data_ptr())
        return {"stats": state["stats"], "votes": state["votes"]}
    if kind == "inchworm":
        table = api.Table(ctx, 25, True, len(state["keys"]), 0.5)
        table.load(state["keys"], state["counts"])
        kept = table.prune(1, state["keep"])
        contigs, sums, seeds, _ = api.inchworm(ctx, table, 2, state["seed_keep"])
        table.free()
        bases, rows, n = np.frombuffer("".join(contigs).encode(), np.uint8), state["contigs"], len(contigs)
        state["bases"][:len(bases)] = bases
        rows[:n, 0], rows[:n, 1], rows[:n, 2] = [len(c) for c in contigs], sums.view(np.int64), seeds.view(np.int64)
        return {"kept": kept, "n": n, "bases": state["bases"], "contigs": rows}
    if kind == "welds":
        reads = _reads(state)
        ks = api.KSet(ctx, state["keys"])
        counts = ks.count(reads, 48, True)
        ks.free()
        reads.free()
        return counts.view(np.int64)
    server = state["server"]
    ids = [server.submit(buf, off, n) for buf, off, n in state["samples"]]
    return [server.wait(j)[1] for j in ids]


def work(case):
    """Bytes: the reads' bases and offsets in, the results out."""
    kind = case["kind"]
    if kind == "component":
        n = case["reads"]
        return {"bytes": n * (case["read_len"] + 8 + 32 + 12) + case["transcripts"] * 2 * 2650, "flops": 0}
    if kind == "batch":
        hi, lo, a = float(case["max_reads"]), 10.0, 1.8
        mean = (a - 1) / (2 - a) * (hi ** (2 - a) - lo ** (2 - a)) / (lo ** (1 - a) - hi ** (1 - a))
        n = case["components"] * mean
        # packed reads (0.375 B a base), packed contigs (10.5 transcripts of 2650 nt)
        return {"bytes": n * (0.375 * case["read_len"] + 12 + 32 + 12) + case["components"] * 10.5 * 2650 * 0.375,
                "flops": 0}
    if kind == "serve":
        lo, hi = math.log(case["min_pairs"]), math.log(case["max_pairs"])
        n = sum(int(v) for v in np.exp(np.linspace(lo, hi, case["samples"])))
        return {"bytes": 2 * n * (case["read_len"] + 8) + n, "flops": 0}
    if kind == "inchworm":
        # the dictionary in (12 B a k-mer: the transcripts' and those that errors made)
        windows = case["read_len"] - 24
        kmers = 1200 * case["transcripts"] + case["units"] * windows * (1 - (1 - case["sub_rate"]) ** 25)
        return {"bytes": 12 * kmers, "flops": 0}
    n = case["units"] * (2 if case.get("paired", True) else 1)
    length = case["read_len"] * (1 - case.get("trim", 0.0) / 2)
    each = length + 8
    if kind in ("job", "stats"):
        each += 32
    if kind == "vote":
        each += 12
    extra = 0
    if kind == "job" and case["paired"]:
        extra = case["units"]
    elif kind == "welds":
        extra = 24 * case["keys"]
    elif kind == "vote":
        extra = case["transcripts"] * 3 * 900 * 0.375
    return {"bytes": n * each + extra, "flops": 0}


def exact(case, seed):
    """None: every output is a whole number, and is compared as such."""
    return None
