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
