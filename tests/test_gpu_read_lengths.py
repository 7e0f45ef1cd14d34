"""Per-read passes at the read lengths where their runs end (64, 128 and 256
windows), with counts on both sides of the 32-bit sums, against the oracle (GPU)."""
from __future__ import annotations

import numpy as np
import pytest

from data import concat
from oracle import oracle as O

pytestmark = pytest.mark.gpu

WINDOWS = [0, 1, 2, 31, 32, 33, 63, 64, 65, 96, 126, 127, 128, 129, 160, 191, 192, 193, 254, 255, 256, 257, 400]
LARGE = [5792, 5793, 4095, 4096, 8190, 8191, 8192, 2**20, 2**31, 2**32 - 1]


@pytest.fixture(scope="module")
def api():
    from trinityrnaseq_amd import api as A
    return A


def _reads(k, longest, n_rate, seed):
    """Three reads of every window count up to `longest` (and some shorter than k), the longest last."""
    rng = np.random.default_rng(seed)
    out = ["", "ACGT"]
    for w in sorted(WINDOWS):
        if w > longest:
            continue
        for _ in range(3):
            s = rng.choice(list("ACGT"), size=w + k - 1 if w else k - 1)
            s[rng.random(len(s)) < n_rate] = "N"
            out.append("".join(s))
    return out


@pytest.mark.parametrize("pipe", ["1", "0"])
@pytest.mark.parametrize("k,canonical", [(25, True), (25, False), (31, True), (13, True), (16, True)])
@pytest.mark.parametrize("longest", [64, 128, 256, 400])
def test_stats_run_ends(api, ctx, monkeypatch, longest, k, canonical, pipe):
    print("stats_run_ends", longest, k, canonical, pipe, flush=True)
    monkeypatch.setenv("TK_STATS_PIPE", pipe)
    seqs = _reads(k, longest, 0.004, 11 + longest)
    seq, off = concat(seqs)
    keys, counts = O.count(seq, off, k, canonical)
    rng = np.random.default_rng(3)
    reads = api.Reads(ctx, seq, off)
    for large in (False, True):
        c = rng.choice([1, 2, 3, 7, 50, 5792, 4095] if not large else [1, 2, 9] + LARGE, size=len(keys)).astype(np.uint32)
        here = rng.random(len(keys)) < 0.8
        t = api.Table(ctx, k, canonical, len(keys), 0.7)
        t.load(keys[here], c[here])
        for nwin, med in [(0, 0), (1, 1), (0, 2)]:
            got = api.read_cov_stats(ctx, t, reads, min_count=2, nwin_policy=nwin, median_policy=med)
            want = O.read_stats(seq, off, keys[here], c[here], k, canonical, 2, 1, nwin, med)
            assert np.array_equal(got, want.astype(got.dtype)), (large, nwin, med)
        t.free()
    reads.free()


@pytest.mark.parametrize("pipe", ["1", "0"])
@pytest.mark.parametrize("k,canonical", [(25, True), (25, False), (31, True), (13, True)])
@pytest.mark.parametrize("longest", [64, 128, 400])
def test_vote_run_ends(api, ctx, monkeypatch, longest, k, canonical, pipe):
    """Each read's windows spread over several components, ties among them."""
    print("vote_run_ends", longest, k, canonical, pipe, flush=True)
    monkeypatch.setenv("TK_VOTE_PIPE", pipe)
    seqs = _reads(k, longest, 0.004, 5 + longest)
    rng = np.random.default_rng(4)
    pieces, comps = [], []
    for s in seqs:
        for a in range(0, len(s) - k + 1, 9):
            if rng.random() < 0.7:
                pieces.append(s[a:a + k + 5])
                comps.append(int(rng.choice([0, 1, 2, 7, 2**32 - 2])))
    comps = np.array(comps, np.uint32)
    seq, off = concat(seqs)
    cseq, coff = concat(pieces)
    reads, bundles = api.Reads(ctx, seq, off), api.Reads(ctx, cseq, coff)
    ct = api.CTable(ctx, bundles, comps, k, canonical)
    bk, bc = O.r2t_build(cseq, coff, comps, k, canonical)
    got = ct.vote(reads)
    want = O.r2t_vote(seq, off, bk, bc, k, canonical)
    assert np.array_equal(got, want.astype(got.dtype))
    for o in (ct, bundles, reads):
        o.free()


@pytest.mark.parametrize("resident", ["0", "1"])
@pytest.mark.parametrize("k,canonical", [(25, True), (25, False), (21, True), (17, True), (16, True), (13, False)])
def test_count_merge_quarters(api, ctx, monkeypatch, k, canonical, resident):
    """The block merge on reads whose quarters end anywhere in their words,
    repeated enough to pass its run limit, and on one-window and empty reads."""
    print("count_merge_quarters", k, canonical, resident, flush=True)
    monkeypatch.setenv("TK_ORDER_MIN_READS", "0")
    monkeypatch.setenv("TK_RESIDENT", resident)
    monkeypatch.setenv("TK_REGION_KB", "4")
    seqs = _reads(k, 400, 0.004, 21) + ["A" * 150] * 200 + _reads(k, 128, 0.0, 22) * 3
    seq, off = concat(seqs)
    reads = api.Reads(ctx, seq, off)
    t = api.Table(ctx, k, canonical, 4096, 0.5)
    t.count(reads)
    keys, counts = t.dump()
    ok, oc = O.count(seq, off, k, canonical)
    assert np.array_equal(keys, ok) and np.array_equal(counts, oc)
    t.free()
    reads.free()


@pytest.mark.parametrize("n", [1, 3, 500])
@pytest.mark.parametrize("k", [13, 25, 31])
def test_small_sets_spread(api, ctx, k, n):
    """Few sequences of very different lengths (windows spread over the whole
    device in the unordered count, the component table and the sketch)."""
    print("small_sets_spread", k, n, flush=True)
    rng = np.random.default_rng(k + n)
    seqs = ["".join(rng.choice(list("ACGTN"), size=int(L), p=[0.2495] * 4 + [0.002]))
            for L in rng.choice([0, 5, 24, 25, 31, 33, 64, 300, 4097, 9000], size=n)] + ["ACGT" * 500]
    seq, off = concat(seqs)
    comps = rng.integers(0, 4, size=len(seqs)).astype(np.uint32)
    reads = api.Reads(ctx, seq, off)
    t = api.Table(ctx, k, True, 64, 0.5)
    t.count(reads)
    keys, counts = t.dump()
    ok, oc = O.count(seq, off, k, True)
    assert np.array_equal(keys, ok) and np.array_equal(counts, oc)
    est = api.estimate_distinct(ctx, reads, k, True)
    assert abs(est - len(ok)) <= 0.1 * len(ok) + 2
    ct = api.CTable(ctx, reads, comps, k, True)
    bk, bc = O.r2t_build(seq, off, comps, k, True)
    assert ct.info()[0] == len(bk)
    want = O.r2t_vote(seq, off, bk, bc, k, True)
    assert np.array_equal(ct.vote(reads), want.astype(api.R2T_VOTE_DTYPE))
    for o in (ct, t, reads):
        o.free()


@pytest.mark.parametrize("n", [0, 1, 2, 16384, 16385])
def test_uploaded_and_device_reads_agree(api, ctx, n):
    """Sizes and windows of a read set, taken on the host up to 16,384 reads of
    an upload and on the device otherwise, with empty reads and reads below k."""
    print("uploaded_and_device_reads", n, flush=True)
    rng = np.random.default_rng(n)
    lens = rng.choice([0, 1, 24, 25, 26, 31, 32, 33, 64, 90], size=n)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    seq = rng.choice(np.frombuffer(b"ACGTN", np.uint8), p=[.24, .24, .24, .24, .04], size=int(off[-1])).tobytes()
    up = api.Reads(ctx, seq, off)
    d_seq, d_off = api.DeviceBuffer(ctx, max(1, len(seq))), api.DeviceBuffer(ctx, off.nbytes)
    if seq:
        d_seq.upload(np.frombuffer(seq, np.uint8))
    d_off.upload(off)
    dev = api.Reads.from_device(ctx, d_seq.ptr, d_off.ptr, n)
    keys, counts = O.count(seq, off, 25, True)
    for r in (up, dev):
        assert tuple(r.info()) == (n, int(off[-1]), int(lens.max()) if n else 0)
        for k in (1, 25, 31):
            assert r.windows(k) == int(np.maximum(lens - k + 1, 0).sum())
        t = api.Table(ctx, 25, True, 1 << 12)
        t.count(r)
        gk, gc = t.dump()
        assert np.array_equal(gk, keys) and np.array_equal(gc, counts)
        t.free()
        r.free()
