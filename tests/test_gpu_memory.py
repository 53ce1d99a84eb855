"""Device memory: blocks that the library frees are kept and handed back to the
next allocation of the same rounded size (2 MiB steps from 4 MiB on, quarters
of a power of two below); the kept bytes count as free in
gooseberry_device_memory; a reused block serves a new computation correctly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def test_large_block_reused_for_same_rounded_size(gb):
    a = gb.DeviceArray(3 * MIB, np.uint8)          # 3 MiB: below the cache's floor
    b = gb.DeviceArray(9 * MIB + 5, np.uint8)      # rounds to 10 MiB
    pb = b.ptr
    b.free()
    c = gb.DeviceArray(10 * MIB - 7, np.uint8)     # the same rounded size
    assert c.ptr == pb
    d = gb.DeviceArray(12 * MIB, np.uint8)         # another size: a new block
    assert d.ptr != pb
    for x in (a, c, d):
        x.free()


def test_kept_bytes_count_as_free(gb):
    # blocks taken from the pool may not move the driver's free count, but
    # blocks the library keeps after a free must be reported as free
    arrs = [gb.DeviceArray(64 * MIB + 3 * i, np.uint8) for i in range(4)]
    gb.synchronize()
    f1, total = gb.device_memory()
    for x in arrs:
        x.free()
    gb.synchronize()
    f2, _ = gb.device_memory()
    assert f2 >= f1 + 4 * 64 * MIB - 8 * MIB and f2 <= total


def test_reused_blocks_give_the_same_results(gb, oracle):
    rp, ri, rv = gb.laplacian(3, 60)
    n = rp.size - 1
    x = gb.uniform(4, n)
    want = oracle.spmv(rp, ri, rv, x)
    for _ in range(3):
        M = gb.Matrix(rp, ri, rv)           # arrays of 1.5-12 MiB, reused each time
        junk = gb.DeviceArray.from_host(np.full(n, np.nan))
        y = M.spmv(x)
        assert np.max(np.abs(y - want)) <= 1e-14 * np.max(np.abs(want))
        del M
        junk.free()


@pytest.mark.parametrize("n", [1, 32, 33, 160, 161, 4000, 524287, 524289])
def test_small_blocks_reused_and_whole(gb, n):
    # sizes around the steps of the rounding (256 bytes, quarters of a power of
    # two, 4 MiB): every block holds its own contents to its last element
    print("small blocks", n, flush=True)
    first = [gb.DeviceArray.from_host(np.full(n, i + 0.5)) for i in range(6)]
    ptrs = {x.ptr for x in first}
    for x in first:
        x.free()
    again = [gb.DeviceArray.from_host(np.full(n, -i - 0.5)) for i in range(6)]
    assert {x.ptr for x in again} == ptrs
    for i, x in enumerate(again):
        assert np.array_equal(x.numpy(), np.full(n, -i - 0.5))
        x.free()


def test_many_small_blocks_are_given_back(gb):
    # more blocks than the cache keeps: the oldest go back to the pool
    xs = [gb.DeviceArray.from_host(np.full(8, float(i))) for i in range(1500)]
    assert all(np.array_equal(x.numpy(), np.full(8, float(i))) for i, x in enumerate(xs))
    for x in xs:
        x.free()
    ys = [gb.DeviceArray.from_host(np.full(8, -float(i))) for i in range(1500)]
    assert all(np.array_equal(y.numpy(), np.full(8, -float(i))) for i, y in enumerate(ys))
    for y in ys:
        y.free()


def test_kept_blocks_by_kind(gb):
    # many small arrays neither push the large blocks out nor pass their own
    # limits (1024 blocks, 1 GiB); a fuller device takes everything back
    mib = 1 << 20
    big = [gb.DeviceArray((40 + 2 * i) * mib, np.uint8) for i in range(5)]
    for x in big:
        x.free()
    large = gb.device_cache()[1]
    assert large[0] >= 5 and large[1] >= sum((40 + 2 * i) * mib for i in range(5))
    xs = [gb.DeviceArray(100 + i, np.uint8) for i in range(1500)]
    for x in xs:
        x.free()
    (n, size), after = gb.device_cache()
    assert n == 1024 and size <= 1024 * 2048 and after == large
    # blocks of 3.5 MiB: 292 fill 1 GiB
    xs = [gb.DeviceArray(3 * mib + mib // 2, np.uint8) for _ in range(400)]
    kept = gb.device_cache()[1]
    for x in xs:
        x.free()
    (n, size), after = gb.device_cache()
    assert size <= 1 << 30 and n <= 1024 and size > (1 << 30) - 4 * mib and after == kept
