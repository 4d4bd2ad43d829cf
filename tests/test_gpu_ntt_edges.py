"""NTTs and low-degree extensions at the borders of the kernels' shapes, on values
that leave the usual path of their folds, against the oracle (bit for bit).

Shapes: transforms of up to 16 points (one matrix product, several to a group), of
up to 2^12 (whole transforms in a tile, with a last tile that is not full), split
ones with long rows whose cosets run one after the other (2^20 rows, four cosets)
or share a tile, and more randomizers than rows of the split.
"""
import numpy as np
import pytest

from conftest import P

pytestmark = pytest.mark.gpu


def edge_elements(seed, count):
    """Powers of two, 0, 1, p - 1, elements with a word of zeros or ones, and random
    ones between; some stretches hold a single value (sums at their extremes)."""
    pool = [1 << k for k in range(64)] + [0, 0, 1, P - 1, P - 1, P - 2, (1 << 32) - 1, P - (1 << 32),
                                          0xFFFFFFFE << 32, 0x80808080, 0x7F7F7F7F7F7F7F7F]
    pool = np.array([v % P for v in pool], np.uint64)
    g = np.random.RandomState(seed)
    x = np.where(g.randint(0, 4, count) == 0, g.randint(0, P, count, dtype=np.uint64),
                 pool[g.randint(0, pool.size, count)])
    for lo in range(0, count, 1 << 10):
        if g.randint(0, 4) == 0:
            x[lo:lo + 512] = pool[g.randint(0, pool.size)]
    return x


@pytest.mark.parametrize("log_n,cols", [(0, 3), (1, 5), (3, 300), (4, 257), (5, 129), (8, 17), (9, 65),
                                        (11, 9), (12, 5), (13, 3), (16, 3), (18, 2)])
def test_ntt_edges(T, oracle, log_n, cols):
    n = 1 << log_n
    x = edge_elements(log_n, n * cols)
    for run, ref in ((T.lib.ntt_forward_batched, oracle.ntt), (T.lib.ntt_inverse_batched, oracle.intt)):
        d = T.dev(x)
        run(d, n, cols)
        want = np.concatenate([ref(c) for c in x.reshape(cols, n)])
        assert np.array_equal(T.host(d).reshape(-1), want)


@pytest.mark.parametrize("log_n,E,cols,k", [
    (0, 1, 3, 0), (2, 4, 70, 3), (4, 16, 33, 5), (8, 16, 3, 300), (9, 16, 3, 40), (10, 4, 5, 98),
    (12, 2, 3, 7), (12, 4, 3, 98), (13, 4, 2, 98), (16, 4, 2, 700), (17, 8, 2, 98), (19, 4, 1, 9),
    (20, 4, 2, 700),
])
def test_lde_edges(T, oracle, log_n, E, cols, k):
    n = 1 << log_n
    m = E * n
    k = min(k, n)
    x = edge_elements(100 + log_n, n * cols)
    r = edge_elements(200 + k, k * cols) if k else None
    out = T.empty(m * cols)
    T.lib.lde_batch(T.dev(x), cols, n, T.dev(r) if k else None, k, 3, 7, m, out)
    want = oracle.lde_table(x, n, cols, m, 3, 7, None if r is None else r.reshape(cols, k))
    assert np.array_equal(T.host(out).reshape(-1), np.asarray(want).reshape(-1))
