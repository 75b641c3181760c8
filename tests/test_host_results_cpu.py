"""Memory of results in host arrays: kept for reuse only when no array uses it, bounded, safe across threads."""
import gc
import threading
import types

import numpy as np

from conftest import load_pkg


def test_memory_comes_back_with_the_last_array_over_it_only():
    pool = load_pkg("engine")._HostPool(1 << 20)
    a = pool.empty(3, 1000)
    assert a.shape == (3, 1000) and a.dtype == np.float32 and a.flags.writeable and a.flags.c_contiguous
    view, where = a[1, 5:], a.ctypes.data
    a[:] = 7.0
    del a
    gc.collect()
    b = pool.empty(3, 1000)
    assert b.ctypes.data != where      # the view still uses it
    b[:] = 1.0
    assert (view == 7.0).all()
    del view
    gc.collect()
    assert pool.empty(3, 1000).ctypes.data == where


def test_no_more_is_kept_than_the_limit():
    pool = load_pkg("engine")._HostPool(1 << 20)
    arrays = [pool.empty(100, 1000) for _ in range(8)]     # 400 KB each
    del arrays
    gc.collect()
    assert pool._kept <= 1 << 20 and sum(len(v) for v in pool._free.values()) == 2
    big = pool.empty(1000, 1000)                           # beyond the limit: an array of its own
    assert big.flags.owndata
    assert pool.empty(0, 5).shape == (0, 5)


def test_threads_never_share_memory_in_use():
    pool, wrong = load_pkg("engine")._HostPool(1 << 22), []

    def work(k):
        for i in range(300):
            a = pool.empty(20, 1000)
            a[:] = k * 1000 + i
            b = pool.empty(20, 1000)
            b[:] = -1.0
            if not (a == k * 1000 + i).all():
                wrong.append((k, i))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not wrong


def test_arrays_own_their_memory():
    """Resized in place like any array: smaller, within its pages, beyond them, and with the memory back in the pool after."""
    pool = load_pkg("engine")._HostPool(1 << 20)
    a = pool.empty(3, 1000)
    assert a.flags.owndata and a.base is None
    a[:] = np.arange(3000).reshape(3, 1000)
    for rows in (2, 3, 50, 1):
        a.resize((rows, 1000))
        keep = min(rows, 2)
        assert (a[:keep].ravel() == np.arange(1000 * keep)).all()
    assert (a.size, a.flags.owndata) == (1000, True)
    del a
    gc.collect()
    assert pool._kept > 0
    kept = np.empty(1000)
    assert kept.flags.owndata and np.zeros(10).sum() == 0      # arrays made elsewhere are numpy's own


def test_sizes_that_are_no_longer_asked_for_make_room():
    """A batch that shrinks: what the larger results left must not keep the smaller ones from being reused."""
    pool = load_pkg("engine")._HostPool(1 << 20)
    for rows in range(100, 10, -1):
        pool.empty(rows, 1000)
    gc.collect()
    assert pool._kept <= 1 << 20
    where = set()
    for _ in range(5):
        a = pool.empty(8, 1000)
        where.add(a.ctypes.data)
        del a
        gc.collect()
    assert len(where) == 1 and 8 * 4096 in pool._free


def test_arrays_outlive_their_pool():
    engine = load_pkg("engine")
    pool = engine._HostPool(1 << 20)
    a, b = pool.empty(20, 1000), pool.empty(20, 1000)
    a[:], view = 3.0, b[2:]
    view[:] = 4.0
    del pool, b
    gc.collect()
    assert (a == 3.0).all() and (view == 4.0).all()
    a.resize((40, 1000))
    assert (a[:20] == 3.0).all()
    del a, view
    gc.collect()


def test_a_closed_engine_gives_back_what_its_results_left():
    mod = load_pkg("engine")
    e = mod.Engine.__new__(mod.Engine)
    e.L = types.SimpleNamespace(gptoss_engine_info=lambda *a: 0, gptoss_engine_destroy=lambda h: None)
    e._adopt(1)
    pool = e._results
    a, b = pool.empty(20, 1000), pool.empty(20, 1000)
    a[:] = 3.0
    del b
    gc.collect()
    assert pool._kept > 0
    e.close()
    assert pool._kept == 0 and (a == 3.0).all()
    del a                                                  # the pool is released: its memory goes, nothing is kept
    gc.collect()
    assert pool._kept == 0 and pool.empty(20, 1000).flags.owndata
