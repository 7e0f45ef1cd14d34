"""Streaming passes over a finished table (histogram, dump, prune, Inchworm's
seeds) at the sizes where their tiles and bins end, against numpy (GPU)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from trinityrnaseq_amd import api as A
    return A


def _pairs(n, k, seed=5):
    """n distinct sorted keys of k bases; mostly small counts, some past the slot's count field and every LDS bin."""
    rng = np.random.default_rng(seed)
    keys = np.unique(rng.integers(0, 1 << (2 * k), size=2 * n + 16, dtype=np.uint64))
    keys = np.sort(rng.permutation(keys)[:n])
    counts = rng.choice([1, 1, 1, 1, 2, 3, 40, 8190, 8191, 8192, 10000, 10001, 15359, 15360, 15361, 19999, 20000,
                         2**20, 2**32 - 1], size=n).astype(np.uint32)
    return keys, counts


def _table(api, ctx, keys, counts, k=25, canonical=True):
    t = api.Table(ctx, k, canonical, max(len(keys), 1), 0.5)
    if len(keys):
        t.load(keys, counts)
    return t


@pytest.mark.parametrize("n", [0, 1, 31, 2000, 70_001])
def test_histo_bins(api, ctx, n):
    print("histo_bins", n, flush=True)
    keys, counts = _pairs(n, 25)
    t = _table(api, ctx, keys, counts)
    for low, high, inc in [(1, 10000, 1), (1, 1, 1), (2, 20, 3), (1, 15358, 1), (1, 15359, 1), (1, 15360, 1),
                           (5, 40000, 2), (1, 25000, 1), (1, 10000, 10000)]:
        assert np.array_equal(t.histo(low, high, inc), O.histo(counts, low, high, inc)), (low, high, inc)
    t.free()


# one bucket; the last tile of 4,096 slots full, one slot pair over, ragged; many tiles per block
@pytest.mark.parametrize("n", [0, 1, 7, 2047, 2048, 2049, 60_000, 3_000_001])
def test_dump_and_prune_tiles(api, ctx, n):
    print("dump_and_prune_tiles", n, flush=True)
    keys, counts = _pairs(n, 25)
    t = _table(api, ctx, keys, counts)
    for lo, hi in [(1, 2**32 - 1), (2, 2**32 - 1), (8192, 10001), (2**32 - 1, 2**32 - 1)]:
        m = (counts >= lo) & (counts <= hi)
        k, c = t.dump(lo, hi)
        assert np.array_equal(k, keys[m]) and np.array_equal(c, counts[m]), (lo, hi)
    pk, pc = O.prune(keys, counts, 25, 2, 1.5)
    assert t.prune(2, api.entropy_keep_table(25, 1.5)) == len(pk)
    k, c = t.dump()
    assert np.array_equal(k, pk) and np.array_equal(c, pc)
    assert t.prune(3) == int((pc >= 3).sum())
    t.free()


@pytest.mark.parametrize("k", [1, 5, 16, 31])
def test_prune_composition_all_k(api, ctx, k):
    print("prune_composition", k, flush=True)
    keys, counts = _pairs({1: 2, 5: 300}.get(k, 900), k)
    t = _table(api, ctx, keys, counts, k)
    pk, pc = O.prune(keys, counts, k, 2, 1.2)
    assert t.prune(2, api.entropy_keep_table(k, 1.2)) == len(pk)
    gk, gc = t.dump()
    assert np.array_equal(gk, pk) and np.array_equal(gc, pc)
    t.free()


@pytest.mark.parametrize("n", [1, 300, 5000])
def test_inchworm_seeds(api, ctx, n):
    """Random keys hardly overlap, so nearly every seed gives a contig of its own."""
    print("inchworm_seeds", n, flush=True)
    keys, counts = _pairs(n, 25, seed=9)
    t = _table(api, ctx, keys, counts, canonical=False)
    keep = api.entropy_keep_table(25, 1.5)
    contigs, sums, seeds, _ = api.inchworm(ctx, t, 2, keep)
    want, wsum, wseed = O.inchworm(keys, counts, 25, False, 2, keep)
    assert contigs == want and np.array_equal(sums, wsum) and np.array_equal(seeds, wseed)
    t.free()
