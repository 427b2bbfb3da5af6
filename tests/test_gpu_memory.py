"""What a context's memory figures cover: the bytes of tables, blocks and results as they are held
on the device, and the HBM budget of a query against them."""
import numpy as np
import pytest

from accmultiwayjoins_amd import AmjError

pytestmark = pytest.mark.gpu


def _device_free():
    """Free bytes of the device, from the HIP runtime that the library has loaded."""
    import ctypes as C
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so.7").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


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


def test_memory_info_covers_what_the_device_gave(own):
    """Blocks of awkward sizes: what the device has less is what the context says it holds, up to
    2 MiB a block (the granularity of the device's own bookkeeping), and little more than was
    asked for."""
    from accmultiwayjoins_amd.serving import DeviceColumns
    rows = [33_600_001, 33_700_001, 17_000_777, 8_400_003, 300_007, 1_100_003]
    own.relation([np.zeros(1, np.int32)], [0]).close()
    free0, held0 = _device_free(), own.allocated_bytes()
    cols = [DeviceColumns(own, n) for n in rows]
    taken = free0 - _device_free()
    held = own.allocated_bytes() - held0
    asked = sum(2 * 4 * n for n in rows)
    assert asked <= held <= asked + 2 * len(rows) * (64 << 10)
    assert taken <= held + 2 * len(rows) * (2 << 20)
    for c in cols:
        c.close()
    assert own.allocated_bytes() == held0


def test_a_block_freed_with_another_size_is_not_reused_past_its_end(own):
    """amj_device_free with more bytes than were allocated: the next allocation of that size gets
    a block of its own, which holds it."""
    import ctypes as C
    from accmultiwayjoins_amd import _native as N
    from accmultiwayjoins_amd.serving import DeviceColumns
    held = own.allocated_bytes()
    p = C.c_void_p()
    own._check(N.lib().amj_device_alloc(own.h, 1 << 16, C.byref(p)))
    first = p.value
    N.lib().amj_device_free(own.h, first, 48 << 20)
    assert own.allocated_bytes() == held
    n = (48 << 20) // 4
    c = DeviceColumns(own, n, ncols=1)
    assert c.ptrs[0] != first
    c.close()
