"""Few short columns: the tile holds more transforms than there are, and only those
that exist (rounded up to a power of two) are transformed.  Against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_n", [0, 2, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("cols", [1, 2, 3, 5, 63])
def test_ntt_part_tiles(T, oracle, log_n, cols):
    n = 1 << log_n
    x = oracle.splitmix(log_n + 100 * cols, n * cols)
    for run, ref in ((T.lib.ntt_forward_batched, oracle.ntt), (T.lib.ntt_inverse_batched, oracle.intt)):
        d = T.dev(x)
        run(d, n, cols)
        want = np.concatenate([ref(c) for c in x.reshape(cols, n)])
        assert np.array_equal(T.host(d, n * cols), want)


@pytest.mark.parametrize("log_n,E", [(5, 1), (5, 16), (6, 4), (7, 2), (8, 1), (8, 8), (9, 1)])
@pytest.mark.parametrize("cols", [1, 3, 5, 17])
def test_lde_part_tiles(T, oracle, log_n, E, cols):
    n, m = 1 << log_n, E << log_n
    x = oracle.splitmix(log_n + 100 * cols, n * cols)
    out = T.empty(m * cols)
    T.lib.lde_batch(T.dev(x), cols, n, None, 0, 3, 7, m, out)
    want = oracle.lde_table(x, n, cols, m, 3, 7, None)
    assert np.array_equal(T.host(out, m * cols), np.asarray(want).reshape(-1))
