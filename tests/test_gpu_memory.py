"""What a context's memory figures cover: the bytes of tables, blocks and results as they are held
on the device, and the HBM budget of a query against them."""
import numpy as np
import pytest

from accmultiwayjoins_amd import AmjError

pytestmark = pytest.mark.gpu


@pytest.fixture
def own():
    """A context of its own: its figures are those of the test alone."""
    from accmultiwayjoins_amd import Context
    with Context(0) as c:
        yield c


@pytest.mark.parametrize("n", [1000, 8192, 70_001, 1_000_003])
def test_a_table_takes_its_rows_and_bucket_bounds_only(own, n):
    """Keys past the bucket count: keys, values and bucket bounds are 8 n + 4 (B + 1) bytes; the
    three blocks may be rounded up by 64 KiB each."""
    rng = np.random.default_rng(n)
    key = rng.integers(-2**31, 2**31, n).astype(np.int32)
    rel = own.relation([key, np.arange(n, dtype=np.int32)], [0, 1])
    own.hash_table(rel).close()  # the sort's scratch buffers are there from now on
    before = own.allocated_bytes()
    table = own.hash_table(rel)
    assert not table.identity
    held = own.allocated_bytes() - before
    assert 8 * n + 4 * (table.buckets + 1) <= held <= 8 * n + 4 * (table.buckets + 1) + (3 << 16)
    table.close()
    rel.close()


def test_a_budget_counts_the_tables_whole(own):
    """A result that the budget has no room for beside what the context holds is refused, whatever
    of that the tables take."""
    n = 1_000_003
    key = np.arange(n, dtype=np.int32) * 4 + 3  # far past the bucket count
    probe = own.relation([np.arange(n, dtype=np.int32), key], [0, 1])
    build = own.relation([key, np.arange(n, dtype=np.int32)], [1, 2])
    table = own.hash_table(build)
    own.execute(probe, [table], materialize=False)
    result = 3 * 4 * n
    with pytest.raises(AmjError, match="budget"):
        own.execute(probe, [table], hbm_budget_bytes=own.allocated_bytes() + result // 2)
    r = own.execute(probe, [table], hbm_budget_bytes=own.allocated_bytes() + 2 * result)
    assert r.count == n
    for x in (table, probe, build):
        x.close()
