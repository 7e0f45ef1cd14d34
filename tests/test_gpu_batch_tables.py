"""Component tables of a batch at the sizes where their regions and the LDS
build begin and end, against the oracle (GPU)."""
from __future__ import annotations

import numpy as np
import pytest

from data import concat
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from trinityrnaseq_amd import api as A
    return A


def _contigs(rng, k, windows, piece):
    """Contigs of `windows` windows in all, `piece` bases each, the last the rest;
    some repeat an earlier contig, some are empty or hold an N."""
    out, left = [], windows
    while left:
        n = min(left, piece)
        s = rng.choice(list("ACGT"), size=n + k - 1)
        left -= n
        if len(out) > 3 and rng.random() < 0.1:
            s[:min(len(s), len(out[0]))] = list(out[0])[:len(s)]
        if rng.random() < 0.02:
            s[int(rng.integers(len(s)))] = "N"
        out.append("".join(s))
        if rng.random() < 0.02:
            out.append("")
    return out


@pytest.mark.parametrize("packed", ["1", "0"])
@pytest.mark.parametrize("k,canonical", [(25, True), (25, False), (31, True), (13, True)])
def test_batch_table_regions(api, ctx, monkeypatch, k, canonical, packed):
    print("batch_table_regions", k, canonical, packed, flush=True)
    monkeypatch.setenv("TK_BATCH_CT_PACKED", packed)
    rng = np.random.default_rng(5)
    # one region, two, the most in LDS, one more: of 8192 one-word or 4096 two-word slots
    one = 4096 if packed == "1" and k <= 25 else 2048
    comps = []
    for windows, piece in [(one, 300), (1, 300), (one + 1, 5000), (2 * one, 1), (16 * one, 900), (40, 7), (3 * one, 1 << 20),
                           (256 * one, 60000), (256 * one + 1, 90000)]:
        cs = _contigs(rng, k, windows, piece)
        whole = [c for c in cs if len(c) >= k]
        reads = []
        for _ in range(150):
            c = whole[int(rng.integers(len(whole)))]
            b = int(rng.integers(len(c) - k + 1))
            reads.append(c[b:b + 150])
        comps.append((reads + ["".join(rng.choice(list("ACGT"), size=100))], cs))
    comps.insert(2, (["A" * 80] * 3, []))
    comps.append((["A" * 80] * 3, ["", "ACG"]))
    # regions sent more keys than they hold: a few k-mers over and over
    comps.append((comps[0][0][:20] + ["A" * 90, "ACG" * 30], comps[0][1] + ["A" * 9000, "ACG" * 9000, "A" * 90]))
    reads = [r for rs, _ in comps for r in rs]
    contigs = [c for _, cs in comps for c in cs]
    ro = np.cumsum([0] + [len(rs) for rs, _ in comps]).astype(np.uint64)
    co = np.cumsum([0] + [len(cs) for _, cs in comps]).astype(np.uint64)
    b = api.Batch(ctx, api.Reads.from_list(ctx, reads), ro, api.Reads.from_list(ctx, contigs), co, k=k,
                  canonical=canonical, use_graph=True)
    n = len(reads)
    d_st, d_vo = api.DeviceBuffer(ctx, n * 32), api.DeviceBuffer(ctx, n * 12)
    vo = np.zeros(n, api.R2T_VOTE_DTYPE)
    for rep in range(3):
        b.run_d(d_st.ptr, d_vo.ptr)
        d_vo.download(vo)
        for c, (rs, cs) in enumerate(comps):
            seq, off = concat(rs)
            bseq, boff = concat(cs)
            if cs:
                keys, cv = O.r2t_build(bseq, boff, np.arange(len(cs)), k, canonical)
                want = O.r2t_vote(seq, off, keys, cv, k, canonical)
            else:
                want = np.zeros(len(rs), O.R2T_VOTE_DTYPE)
                want["comp"] = 0xFFFFFFFF
                want["nwin"] = [max(0, len(r) - k + 1) for r in rs]
            a, z = int(ro[c]), int(ro[c + 1])
            assert np.array_equal(vo[a:z], want.astype(vo.dtype)), (rep, c)
    b.free()


def _with_runs_of_empties(rng, k, runs):
    """Contigs of 40 to 400 bases with runs of empty ones between them, and
    reads from them."""
    contigs = []
    for n in runs:
        contigs += ["".join(rng.choice(list("ACGT"), size=int(rng.integers(40, 400)))) for _ in range(20)] + [""] * n
    contigs.append(contigs[0])
    whole = [c for c in contigs if c]
    return contigs, [whole[int(rng.integers(len(whole)))][:150] for _ in range(300)]


@pytest.mark.parametrize("k", [25, 31])
def test_runs_of_empty_contigs(api, ctx, k):
    """The passes that go over packed contig words find each word's contig past
    runs of empty ones, shorter and longer than they step over one by one: one
    table, and a batch whose table has several regions."""
    print("runs_of_empty_contigs", k, flush=True)
    contigs, reads = _with_runs_of_empties(np.random.default_rng(6), k, [0, 1, 2, 3, 4, 5, 6, 7, 100, 1000] * 3)
    seq, off = concat(reads)
    bseq, boff = concat(contigs)
    keys, cv = O.r2t_build(bseq, boff, np.arange(len(contigs)), k, True)
    want = O.r2t_vote(seq, off, keys, cv, k, True)
    r, b = api.Reads(ctx, seq, off), api.Reads(ctx, bseq, boff)
    t = api.CTable(ctx, b, np.arange(len(contigs), dtype=np.uint32), k, True)
    assert np.array_equal(t.vote(r), want.astype(api.R2T_VOTE_DTYPE))
    n = len(reads)
    batch = api.Batch(ctx, r, np.array([0, n], np.uint64), b, np.array([0, len(contigs)], np.uint64), k=k)
    d_st, d_vo = api.DeviceBuffer(ctx, n * 32), api.DeviceBuffer(ctx, n * 12)
    batch.run_d(d_st.ptr, d_vo.ptr)
    vo = np.zeros(n, api.R2T_VOTE_DTYPE)
    d_vo.download(vo)
    assert np.array_equal(vo, want.astype(vo.dtype))
    batch.free()


def test_long_run_of_empty_contigs_is_stepped_over(api, ctx):
    """A million empty sequences between two others cost the table build a
    bisection, not a million steps of one lane."""
    print("long_run_of_empty_contigs", flush=True)
    contigs, reads = _with_runs_of_empties(np.random.default_rng(7), 25, [1_000_000, 0])
    bseq, boff = concat(contigs)
    b = api.Reads(ctx, bseq, boff)
    comps = np.arange(len(contigs), dtype=np.uint32)
    ctx.timing(True)
    ctx.timing_reset()
    t = api.CTable(ctx, b, comps, 25, True)
    ctx.sync()
    ms = ctx.kernel_time("ctable_build")[0]
    ctx.timing(False)
    seq, off = concat(reads)
    keys, cv = O.r2t_build(bseq, boff, comps, 25, True)
    assert np.array_equal(t.vote(api.Reads(ctx, seq, off)), O.r2t_vote(seq, off, keys, cv, 25, True).astype(api.R2T_VOTE_DTYPE))
    print("ctable_build", ms, "ms", flush=True)
    assert ms < 5  # 0.02; 84 step by step
