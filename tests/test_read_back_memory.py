"""Host memory of batch read-backs: arrays that are alive never share memory,
memory of arrays that are gone is used again, a bounded amount is kept and none
without a batch."""
import gc
import threading

import numpy as np
import pytest

from pfpa.hostmem import BlockPool


@pytest.mark.parametrize("shape", [(1,), (3, 5), (64, 64), (602, 402), (1000, 1026)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_array(shape, dtype):
    p = BlockPool(1 << 30)
    p.open(1)
    a = p.array(shape, dtype)
    assert a.shape == shape and a.dtype == dtype and a.flags.c_contiguous and a.flags.writeable
    a[...] = 3
    first = a.ctypes.data
    view = a.reshape(-1)[-1:]
    del a
    b = p.array(shape, dtype)
    assert b.ctypes.data != first and view[0] == 3      # a view keeps the memory
    b[...] = 4
    assert view[0] == 3
    del view
    c = p.array(shape, dtype)
    assert c.ctypes.data == first                       # and gives it back
    c[...] = 5
    assert (b == 4).all()


def test_size_class():
    """At most an eighth more than asked for (or the rest of a page)."""
    for n in list(range(1, 20000, 37)) + [2 ** k + d for k in range(12, 40) for d in (-1, 0, 1)]:
        c = BlockPool.size_class(n)
        assert n <= c <= max(n + n // 8, (n + 4095) // 4096 * 4096), n
        assert BlockPool.size_class(c) == c


def test_bounded_and_given_back():
    p = BlockPool(10 << 20)
    for user in (1, 2):
        p.open(user)
    live = [p.array((1 << 20,), np.uint8) for _ in range(20)] + [p.array((3 << 20,), np.uint8)]
    live.clear()
    p.array((1,), np.uint8)
    held = sum(len(b) for v in p.free.values() for b in v)
    assert held == p.free_bytes and 4 << 20 < held <= 10 << 20
    p.close(1)
    assert p.free_bytes
    p.close(2)
    assert not p.free and not p.free_bytes
    late = p.array((1 << 20,), np.uint8)                # no user: nothing is kept
    del late
    assert not p.free and not p.returned


def test_an_array_may_die_inside_the_pool():
    """A finalizer that runs while its own thread holds the pool's lock."""
    p = BlockPool(1 << 30)
    p.open(1)
    a = p.array((5000,), np.uint8)
    with p.lock:
        del a
    assert len(p.returned) == 1
    p.array((1,), np.uint8)
    assert not p.returned


def test_threads():
    p = BlockPool(1 << 20)
    p.open(1)
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        keep = []
        for i in range(400):
            a = p.array((int(rng.integers(1, 60000)),), np.int64)
            a[...] = k * 1000 + i
            keep.append((a, k * 1000 + i))
            if len(keep) > 5:
                b, v = keep.pop(int(rng.integers(0, 5)))
                if not (b == v).all():
                    bad.append(k)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    gc.collect()
    assert not bad
    p.close(1)
    assert not p.free_bytes


@pytest.mark.gpu
def test_reads_of_a_batch_fault_no_pages(gpu):
    """Passes over a batch whose fields are read back, one pass's arrays alive
    while the next are made: after the first two, none maps fresh pages.  What
    is held keeps its values."""
    import resource

    from pfpa import batch as B
    from pfpa import model as M

    n = 500
    s = M.make_setup(n, n, bc=1)
    f = M.init_matrix_with_particles(n, n, s.dx, 1, seed=3)
    b = B.Batch(B.PF_STORAGE_F64, 6 * B.job_bytes(B.PF_STORAGE_F64, n, n), max_jobs=6)
    ids = [b.add(B.make_desc(s, 1 << 40, instance=k), f) for k in range(6)]
    b.commit()
    held, faults = None, []
    for _ in range(6):
        b.run(1)
        b.sync()
        before = resource.getrusage(resource.RUSAGE_SELF).ru_minflt
        now = [b.read(j) for j in ids]
        faults.append(resource.getrusage(resource.RUSAGE_SELF).ru_minflt - before)
        if held is not None:
            assert all((x[0] == y).all() for x, y in zip(held, copies))
        held, copies = now, [x[0].copy() for x in now]
    pages = 6 * 4 * 8 * (n + 2) ** 2 // 4096
    assert max(faults[2:]) < pages // 20, (faults, pages)
    b.close()
