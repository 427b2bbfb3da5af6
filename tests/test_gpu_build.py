"""Hash-table builds at the sizes and key patterns where their variants meet: the one-workgroup
build (up to 8,192 rows), the tiled sort (4,096-row tiles) and the bucket index (2,048 buckets per
workgroup, heavy buckets searched), tables of keys below and past the bucket count. Every build is read
back through a two-relation join whose rows must come out in exactly the order a stable sort
gives."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 1023, 1024, 1025, 4095, 4097, 8191, 8192, 8193, 12_289, 65_536, 70_001,
         1_000_003]


def _keys(kind, n, rng):
    if kind == "uniform-small":    # every key below the bucket count: an identity table
        return rng.integers(0, max(1, n // 4), n)
    if kind == "uniform-wide":     # keys over all 32 bits, negative ones among them
        return rng.integers(-2**31, 2**31, n)
    if kind == "past-buckets":     # some keys past the bucket count, several per bucket
        return rng.integers(0, 3 * n + 2, n)
    if kind == "heavy":            # one key holds most rows, the rest spread
        return np.where(rng.random(n) < 0.9, 7, rng.integers(0, 2 * n + 1, n))
    if kind == "sorted":
        return np.sort(rng.integers(0, n + 1, n))
    if kind == "equal":
        return np.full(n, -5)
    raise ValueError(kind)


@pytest.mark.parametrize("kind", ["uniform-small", "uniform-wide", "past-buckets", "heavy",
                                  "sorted", "equal"])
@pytest.mark.parametrize("n", SIZES)
def test_build_rows_come_out_in_stable_key_order(ctx, n, kind):
    rng = np.random.default_rng(n)
    key = _keys(kind, n, rng).astype(np.int32)
    val = rng.integers(-2**31, 2**31, n).astype(np.int32)
    # probes: keys present, keys next to them, and keys of nothing; few rows of a heavy key
    uniq, counts = np.unique(key, return_counts=True)
    light = uniq[counts <= 64]
    pk = np.concatenate([light[:3000], uniq[:2], uniq[-2:], (light[:500] + 1).astype(np.int32),
                         np.array([-2**31, 2**31 - 1, 0], np.int32)]).astype(np.int32)
    pa = np.arange(len(pk), dtype=np.int32)
    order = np.argsort(key, kind="stable")
    sk, sv = key[order], val[order]
    lo, hi = np.searchsorted(sk, pk, "left"), np.searchsorted(sk, pk, "right")
    reps = hi - lo
    want_a = np.repeat(pa, reps)
    want_v = np.concatenate([sv[a:b] for a, b in zip(lo, hi)] + [np.empty(0, np.int32)])
    r = ctx.chain_join([([pa, pk], [0, 1]), ([key, val], [1, 2])], fetch=True)
    assert r.count == len(want_a)
    if r.count:
        assert np.array_equal(r.cols[0], want_a)
        assert np.array_equal(r.cols[1], np.repeat(pk, reps))
        assert np.array_equal(r.cols[2], want_v)


@pytest.mark.parametrize("n", [1, 1024, 4097, 8192, 8193, 70_001])
def test_build_with_sorted_values_checks_both_columns(ctx, n):
    """sort_vals: a closing relation C(0, 1) over the pairs of the probe, so that every probe row
    (a, b) yields the rows of C equal to (a, b)."""
    rng = np.random.default_rng(n + 1)
    a = rng.integers(-40, 40, n).astype(np.int32)
    b = rng.integers(0, 2 * n, n).astype(np.int32)
    rel, ht = ctx.relation([a, b], [0, 1]), None
    try:
        ht = ctx.hash_table(rel, 0, sort_vals=True)
        r = ctx.execute(rel, [ht], fetch=True)
        pair = (a.astype(np.int64) << 32) + b
        _, inv, cnt = np.unique(pair, return_inverse=True, return_counts=True)
        reps = cnt[inv]
        assert r.count == int(reps.sum())
        assert np.array_equal(r.cols[0], np.repeat(a, reps))
        assert np.array_equal(r.cols[1], np.repeat(b, reps))
    finally:
        if ht is not None:
            ht.close()
        rel.close()


@pytest.mark.parametrize("n", [1 << 20, (1 << 20) + 4097])
def test_grouped_probe_rows_come_out_in_stable_key_order(ctx, n):
    """fib groups the probe rows by join key (unsigned) when there are at least 2^20."""
    rng = np.random.default_rng(n)
    pa = rng.integers(-2**31, 2**31, n).astype(np.int32)
    pk = rng.integers(-3, 200_000, n).astype(np.int32)
    key = rng.permutation(np.arange(-3, 150_000, dtype=np.int32))
    val = rng.integers(0, 2**31, len(key)).astype(np.int32)
    r = ctx.chain_join([([pa, pk], [0, 1]), ([key, val], [1, 2])], fetch=True, fib=1)
    order = np.argsort(pk.view(np.uint32), kind="stable")
    ga, gk = pa[order], pk[order]
    hit = (gk >= -3) & (gk < 150_000)
    of_key = np.empty(150_003, np.int32)
    of_key[key + 3] = val
    assert r.count == int(hit.sum())
    assert np.array_equal(r.cols[0], ga[hit])
    assert np.array_equal(r.cols[1], gk[hit])
    assert np.array_equal(r.cols[2], of_key[gk[hit] + 3])
