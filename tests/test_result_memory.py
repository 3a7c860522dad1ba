"""The memory that large results stand in: owned by numpy, recycled, resizable, usable from several threads and after a fork."""
import os
import threading

import numpy as np
import pytest

from grilly_amd import _lib as L
from grilly_amd.backend import core

LARGE = core.RECYCLED_MIN // 4


def test_large_results_are_recycled_and_owned():
    lib = L.load()
    a = core.result_array(lib, (2, LARGE))
    assert a.shape == (2, LARGE) and a.dtype == np.float32 and a.flags.owndata and a.flags.writeable and a.flags.c_contiguous
    a[:] = 1.0
    at = a.ctypes.data
    view = a[1, 5:9]
    del a
    b = core.result_array(lib, (2, LARGE))
    assert b.ctypes.data != at and (view == 1.0).all()      # still in use by the view
    del view
    c = core.result_array(lib, (LARGE - 7, 2))
    assert c.ctypes.data == at
    assert np.empty(LARGE, np.float32).ctypes.data not in (at, b.ctypes.data)      # other arrays: numpy's usual memory


@pytest.mark.parametrize("to", [LARGE // 8, LARGE - 1, LARGE, 3 * LARGE])
def test_resize(to):
    a = core.result_array(L.load(), (LARGE,))
    a[:] = np.arange(LARGE)
    a.resize(to, refcheck=False)
    n = min(to, LARGE)
    np.testing.assert_array_equal(a[:n], np.arange(n, dtype=np.float32))
    assert (a[n:] == 0).all()


def test_small_and_empty_results():
    lib = L.load()
    for shape in [(0, LARGE), (LARGE, 0), (3,), (), (1, 7)]:
        a = core.result_array(lib, shape)
        assert a.shape == shape and a.flags.owndata


def test_threads_and_forked_children():
    """Threads take and give blocks while the process forks; each child takes, writes and gives blocks of its own."""
    lib, stop, wrong = L.load(), threading.Event(), []

    def worker(t):
        while not stop.is_set():
            a = core.result_array(lib, (LARGE + 1024 * t,))
            a[::4096] = t
            if not (a[::4096] == t).all():
                wrong.append(t)

    kept = core.result_array(lib, (LARGE,))
    kept[:] = 9.0
    threads = [threading.Thread(target=worker, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    try:
        for _ in range(6):
            child = os.fork()
            if child == 0:
                ok = bool((kept == 9.0).all())
                kept[:] = 1.0
                a = core.result_array(lib, (LARGE,))
                a[:] = 2.0
                ok = ok and (kept == 1.0).all() and (a == 2.0).all()
                del a
                os._exit(0 if ok else 1)
            assert os.waitpid(child, 0)[1] == 0
    finally:
        stop.set()
        for t in threads:
            t.join()
    assert not wrong and (kept == 9.0).all()
