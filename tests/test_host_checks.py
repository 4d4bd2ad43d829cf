"""Input checks of the host commit, on a host without a GPU too: the first element
that is not canonical is named, wherever it is, also where several threads check
at once; on a GPU a table is refused before its commit, by the workers that copy it.
"""
import re
import threading
import time

import numpy as np
import pytest

from conftest import P


@pytest.fixture(scope="module")
def lib(tvhmod):
    return tvhmod.load()


def refusal(lib, a, cols=1):
    """(status, index named) of a host commit."""
    root, n = np.zeros(5, np.uint64), a.size // cols
    rc = lib.raw("tvh_commit_host", a.ctypes.data, cols, n, None, 0, 1, 7, 4 * n, None, None,
                 root.ctypes.data)
    m = re.match(r"element (\d+) >= p", lib.last_error())
    return rc, int(m.group(1)) if m else None


def test_status_code(lib):
    assert "canonical" in lib.status_string(refusal(lib, np.array([P], np.uint64))[0]).lower()


@pytest.mark.parametrize("log_n", [0, 10, 16, 17, 20])
def test_first_bad_element_is_named(lib, log_n):
    n = 1 << log_n
    rng = np.random.RandomState(log_n)
    status = refusal(lib, np.array([P], np.uint64))[0]
    a = rng.randint(0, P, n, dtype=np.uint64)
    places = {0, n - 1, n // 2, min(n - 1, 1023), min(n - 1, 1024), min(n - 1, 8191),
              min(n - 1, 8192)} | {int(v) for v in rng.randint(0, n, 8)}
    for at in sorted(places):
        b = a.copy()
        b[rng.randint(0, n, 5)] = P - 1  # canonical, with a high word of ones
        for later in rng.randint(at, n, 3):  # more of them behind it
            b[later] = np.uint64(P + 1 + int(rng.randint(0, 1000)))
        b[at] = P
        assert refusal(lib, b) == (status, at)


def test_threads_check_at_once(lib):
    n, status = 1 << 19, refusal(lib, np.array([P], np.uint64))[0]
    rng = np.random.RandomState(1)
    a = rng.randint(0, P, n, dtype=np.uint64)
    wrong = []

    def work(seed):
        r = np.random.RandomState(seed)
        for _ in range(20):
            b, at = a.copy(), int(r.randint(0, n))
            b[at] = 0xFFFFFFFFFFFFFFFF
            if refusal(lib, b) != (status, at):
                wrong.append((seed, at))

    ts = [threading.Thread(target=work, args=(s,)) for s in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong


@pytest.mark.gpu
@pytest.mark.parametrize("log_n,cols", [(7, 3), (12, 30), (13, 100), (14, 300)])
def test_first_bad_element_is_named_on_the_way(tvh, log_n, cols):
    """Copied at once, by the staging workers, and in two pieces of the ring: the ends of
    their shares (4 KiB steps) and stretches (32 KiB), more of them behind it."""
    n = cols << log_n
    status = refusal(tvh, np.array([P], np.uint64))[0]
    rng = np.random.RandomState(cols)
    a = rng.randint(0, P, n, dtype=np.uint64)
    a[rng.randint(0, n, 50)] = P - 1
    piece, share = 4 << 20, -(-min(n, 4 << 20) // 8 // 512) * 512
    places = {0, n - 1, 8192, 4096, share - 1, share, 3 * share + 4095, piece - 1, piece, piece + 5}
    for at in sorted(p for p in places if p < n):
        b = a.copy()
        b[rng.randint(at, n, 3)] = P + 5
        b[at] = P
        assert refusal(tvh, b, cols) == (status, at)
    assert refusal(tvh, a, cols)[0] == 0  # and then a good one


@pytest.mark.gpu
def test_refusal_comes_before_the_work(tvh):
    """An element that is not canonical ends the call before its table is sent and
    committed (it once waited for both: 2.4 ms here, against microseconds)."""
    n, cols = 1 << 14, 379
    a = np.random.RandomState(2).randint(0, P, n * cols, dtype=np.uint64)
    root, t = np.zeros(5, np.uint64), {}
    for name, at in (("good", None), ("first", 0), ("middle", n * cols // 2)):
        b = a.copy()
        if at is not None:
            b[at] = P
        best = 1e9
        for _ in range(4):
            t0 = time.perf_counter()
            rc = tvh.raw("tvh_commit_host", b.ctypes.data, cols, n, None, 0, 1, 7, 4 * n, None, None,
                         root.ctypes.data)
            best = min(best, time.perf_counter() - t0)
            assert (rc == 0) == (at is None)
        t[name] = best
    assert t["first"] < 0.1 * t["good"]
    assert t["middle"] < 0.7 * t["good"]
