"""Sizes at which the layout of buffers changes: tries whose runs end at, straddle and repeat over
the 2,048-pair tiles of the compaction, columns on both sides of the 512 KB staging limit, and
window-written results whose length is no whole number of cache lines, staging blocks or
windows."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["distinct", "one-run", "pairs-repeat", "all-equal", "runs-of-tile"])
@pytest.mark.parametrize("n", [1, 2, 255, 2047, 2048, 2049, 4096, 8192, 8193, 20_481, 300_007])
def test_trie_levels_are_the_sorted_distinct_pairs(ctx, n, kind):
    rng = np.random.default_rng(n)
    i = np.arange(n)
    x, y = {"distinct": (i, rng.integers(-2**31, 2**31, n)),
            "one-run": (np.full(n, -3), i),
            "pairs-repeat": (i // 7 // 2 - 5, i // 7),          # every pair seven times
            "all-equal": (np.full(n, 9), np.full(n, -9)),
            "runs-of-tile": (i // 2048, rng.integers(0, 1500, n))}[kind]
    p = rng.permutation(n)
    x, y = x.astype(np.int32)[p], y.astype(np.int32)[p]
    want = np.unique(np.stack([x, y], 1), axis=0)
    d0, first, runs = np.unique(want[:, 0], return_index=True, return_counts=True)
    t = ctx.trie([x, y])
    g0, off, g1 = t.levels()
    assert np.array_equal(g0, d0)
    assert np.array_equal(np.asarray(off, np.int64), np.append(first, len(want)))
    assert np.array_equal(g1, want[:, 1])
    t.close()


@pytest.mark.parametrize("n", [1, 1023, 65_535, 65_536, 65_537, 131_071, 131_072, 131_073, 300_001])
def test_uploads_do_not_alias_the_callers_arrays(ctx, n):
    """Columns are the call's: writing over the arrays right after relation() returns, and
    reusing the freed blocks of an earlier relation, leaves what was uploaded. Rows come back
    through a one-table join, on both sides of the staging limit."""
    for seed in (1, 2):
        rng = np.random.default_rng(seed)
        a = np.arange(n, dtype=np.int32) * 3 + seed
        k = rng.integers(0, n, n).astype(np.int32)
        v = rng.integers(-2**31, 2**31, n).astype(np.int32)
        kept = [a.copy(), k.copy()]
        probe = ctx.relation([a, k], [0, 1])
        a[:] = -1
        k[:] = 0
        bk = np.arange(n, dtype=np.int32)
        vv = v.copy()
        build = ctx.relation([bk, vv], [1, 2])
        bk[:] = 0
        vv[:] = 0
        table = ctx.hash_table(build)
        r = ctx.execute(probe, [table], fetch=True)
        assert r.count == n
        assert np.array_equal(r.cols[0], kept[0]) and np.array_equal(r.cols[1], kept[1])
        assert np.array_equal(r.cols[2], v[kept[1]])
        table.close()
        probe.close()
        build.close()


@pytest.mark.parametrize("suffix", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 4095, 4097, 70_003])
def test_window_written_results_at_ragged_lengths(ctx, n, suffix):
    """n results of a 4-way chain: the rows of the window writer, hashed or not, are those of the
    count/write engine."""
    rng = np.random.default_rng(n)
    keys = max(1, n // 3)
    rels = [([np.arange(n, dtype=np.int32), rng.integers(0, keys, n).astype(np.int32)], [0, 1])]
    for t in range(3):  # two rows per key in the second table, one in the others
        k = np.repeat(np.arange(keys), 2 if t == 1 else 1)
        rels.append(([k.astype(np.int32), rng.integers(0, keys, len(k)).astype(np.int32)],
                     [t + 1, t + 2]))
    want = ctx.chain_join(rels, fetch=True)
    for checksum in (True, False):
        got = ctx.chain_join(rels, fetch=True, fib=1, fib_suffix=suffix, checksum=checksum)
        assert got.path != want.path and got.count == want.count == 2 * n
        if checksum:
            assert got.checksum == want.checksum
        a, b = (np.stack(r.cols, 1) for r in (got, want))
        assert np.array_equal(a[np.lexsort(a.T)], b[np.lexsort(b.T)])


def test_a_relation_is_there_for_another_context_when_the_call_returns(ctx):
    """Small relations made through one context and read at once by another one's stream."""
    from accmultiwayjoins_amd import Context
    with Context(0) as other:
        for i in range(200):
            n = 60_001 + i  # two columns below the staging limit
            rng = np.random.default_rng(i)
            key = rng.permutation(n).astype(np.int32)
            val = rng.integers(-2**31, 2**31, n).astype(np.int32)
            build = ctx.relation([key, val], [1, 2])
            table = other.hash_table(build)
            probe = ctx.relation([val, key], [0, 1])
            r = other.execute(probe, [table], fetch=True)
            assert r.count == n
            assert np.array_equal(r.cols[0], val) and np.array_equal(r.cols[2], val)
            table.close()
            probe.close()
            build.close()


def test_more_columns_in_one_call_than_the_staging_buffer_holds(ctx):
    """Six relations of just under 512 KB each: the buffer of 2 MB is started over while copies out
    of it may still be running."""
    n = 65_000
    rng = np.random.default_rng(6)
    rels = [([np.arange(n, dtype=np.int32), rng.permutation(n).astype(np.int32)], [0, 1])]
    rels += [([np.arange(n, dtype=np.int32), rng.permutation(n).astype(np.int32)], [t, t + 1])
             for t in range(1, 6)]
    want = [rels[0][0][0], rels[0][0][1]]
    for cols, _ids in rels[1:]:
        want.append(cols[1][want[-1]])
    for _ in range(3):
        r = ctx.chain_join(rels, fetch=True)
        assert r.count == n
        order = np.argsort(r.cols[0], kind="stable")
        for got, w in zip(r.cols, want):
            assert np.array_equal(got[order], w)
