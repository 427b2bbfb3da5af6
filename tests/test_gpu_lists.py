"""Intersections of the compiled triangle and 4-clique shapes at the list lengths and values where
their variants meet: LDS tables (up to 7/16 of 64 .. 2,048 slots), lists that do not fit or do not
settle in a table, lists past the stage, streamed and flattened children, duplicates in CSR tries."""
import math

import numpy as np
import pytest

import oracle_ffi as O

pytestmark = pytest.mark.gpu

TRI = [(0, 1), (1, 2), (0, 2)]


def _csr(lists):
    """(d0, off, d1) of {value: children} with the children sorted, duplicates kept."""
    d0 = np.array(sorted(lists), np.int32)
    runs = [np.sort(np.asarray(lists[int(v)], np.int32)) for v in d0]
    off = np.concatenate([[0], np.cumsum([len(r) for r in runs])]).astype(np.uint64)
    return d0, off, (np.concatenate(runs) if runs else np.empty(0)).astype(np.int32)


def _slots(v, words):
    """The two table slots of a value."""
    x = (v ^ (v >> 11)) & 0xFFFFFFFF
    return x & (words - 1), ((((x & 0xFFFFFF) * 0x9AD2D5) & 0xFFFFFFFF) >> 12) & (words - 1)


def _values(kind, n, rng):
    if kind == "random":
        return rng.choice(2**31 - 1, 2 * n, replace=False)[:n].astype(np.int64)
    if kind == "consecutive":
        return 1000 + np.arange(n, dtype=np.int64)
    # colliding: many values share both slots of a 2,048-slot table, so no table settles
    v = rng.integers(0, 2**31 - 1, 4_000_000).astype(np.int64)
    a, b = _slots(v, 2048)
    pair = a * 2048 + b
    u, c = np.unique(pair, return_counts=True)
    same = np.unique(v[np.isin(pair, u[c >= 3][:max(1, n // 8)])])
    rest = rng.choice(2**31 - 1, n, replace=False).astype(np.int64)
    return np.unique(np.concatenate([same, rest]))[:n] if len(same) < n else same[:n]


@pytest.mark.parametrize("kind", ["random", "consecutive", "colliding"])
@pytest.mark.parametrize("n", [31, 32, 64, 65, 111, 112, 113, 447, 449, 895, 896, 897, 1024, 1025])
def test_triangle_lists_match_set_intersections(ctx, n, kind):
    rng = np.random.default_rng(n)
    kept = _values(kind, n, rng)
    a1s = [7, 8, 9, 10, 11, 12]
    streamed = {}
    for i, a1 in enumerate(a1s):  # shorter, longer and equal lists, partly in the kept one
        m = [n, max(1, n // 2), 33, 64, min(2 * n, 1024), 300][i]
        own = rng.choice(kept, min(m, n), replace=False)
        streamed[a1] = np.unique(np.concatenate([own[: max(1, 2 * len(own) // 3)],
                                                 rng.integers(0, 2**31 - 1, m)]))
    roots = {5: a1s, 6: a1s[:2]}
    tries = [ctx.trie_from_csr(*_csr(roots), attr_ids=(0, 1)),
             ctx.trie_from_csr(*_csr({5: kept, 6: kept[::2]}), attr_ids=(0, 2)),
             ctx.trie_from_csr(*_csr(streamed), attr_ids=(1, 2))]
    want = sorted((a0, a1, int(v)) for a0 in roots for a1 in roots[a0]
                  for v in np.intersect1d(kept if a0 == 5 else kept[::2], streamed[a1]))
    try:
        for kw in (dict(), dict(dro=1), dict(ws=1)):
            r = ctx.lftj(tries, [0, 1, 2], "DFS", fetch=True, **kw)
            assert sorted(map(tuple, r.tuples().tolist())) == want, kw
            assert r.checksum == O.checksum(want), kw
        for algo in ("DFS", "BFS"):
            c = ctx.lftj(tries, [0, 1, 2], algo, materialize=False)
            assert (c.count, c.checksum) == (len(want), O.checksum(want)), algo
    finally:
        for t in tries:
            t.close()


def test_duplicate_children_count_as_the_shorter_list_has_them(ctx):
    """Candidates come from the shorter list, each as often as it holds it; the other list is asked
    only whether it holds the value. Lists long enough for the wave-wide path."""
    base = np.arange(0, 400, 2)
    short = np.concatenate([base[:60], base[:60], base[100:110]])  # 130 values, 60 of them twice
    long = np.concatenate([base, base[:50]])                        # 250 values
    for kept, streamed in ((short, long), (long, short)):
        tries = [ctx.trie_from_csr(*_csr({1: [2]}), attr_ids=(0, 1)),
                 ctx.trie_from_csr(*_csr({1: kept}), attr_ids=(0, 2)),
                 ctx.trie_from_csr(*_csr({2: streamed}), attr_ids=(1, 2))]
        want = sorted((1, 2, int(v)) for v in short if v in set(long.tolist()))
        r = ctx.lftj(tries, [0, 1, 2], "DFS", fetch=True)
        assert sorted(map(tuple, r.tuples().tolist())) == want
        for t in tries:
            t.close()


@pytest.mark.parametrize("ws", [0, 1])
@pytest.mark.parametrize("n", [5, 34, 66, 97, 130, 225, 300, 450, 470, 780])
def test_cliques_of_complete_graphs(ctx, n, ws):
    """C(n, 4) 4-cliques and C(n, 3) triangles of K_n, its vertices spread over the ids."""
    ids = np.sort(np.random.default_rng(n).choice(1 << 20, n, replace=False)).astype(np.int32)
    i, j = np.triu_indices(n, 1)
    s, d = ids[i], ids[j]
    t3 = ctx.lftj_pattern(s, d, "TRI", "DFS", materialize=False, ws=ws)
    t4 = ctx.lftj_pattern(s, d, "FOUR", "DFS", materialize=False, ws=ws)
    assert t3.count == n * (n - 1) * (n - 2) // 6
    assert t4.count == n * (n - 1) * (n - 2) * (n - 3) // 24
    if n <= 130:
        assert (t3.count, t3.checksum) == O.triangles(s, d)
        assert (t4.count, t4.checksum) == O.four_cliques(s, d)
        w = ctx.lftj_pattern(s, d, "FOUR", "DFS", materialize=True, ws=ws)
        assert (w.count, w.checksum) == (t4.count, t4.checksum)
        ctx.free(w)


@pytest.mark.parametrize("query,n,stall", [("FOUR", 512, 50), ("TRI", 1000, 10)])
def test_ws_long_units_with_progress_are_not_a_stall(ctx, query, n, stall):
    """K_n in a few units of 64 roots and no tasks (a split longer than any run): a few waves work
    for much longer than the stall limit while all others are idle. What the working waves
    report from inside their lists keeps the pass alive."""
    i, j = np.triu_indices(n, 1)
    s, d = i.astype(np.int32), j.astype(np.int32)
    want = ctx.lftj_pattern(s, d, query, "DFS", materialize=False)
    assert want.count == (math.comb(n, 4) if query == "FOUR" else math.comb(n, 3))
    r = ctx.lftj_pattern(s, d, query, "DFS", materialize=False, ws=1,
                         ws_split_threshold=1 << 20, ws_stall_ms=stall)
    assert (r.count, r.checksum) == (want.count, want.checksum)
    assert r.detail == 0  # no tasks
