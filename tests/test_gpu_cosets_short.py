"""Coset evaluations of columns of up to 2^12 rows: whole columns in a tile, several
to a group of the matrix product below 16 rows, the last tile not full, more
columns than a block each could serve (2^24 blocks of 256 threads are a grid's
limit), against the oracle's NTT of the scaled coefficients (bit for bit)."""
import numpy as np
import pytest

from conftest import P

pytestmark = pytest.mark.gpu


def scaled(oracle, coeff, rand, delta, base):
    """(c_i + [i < k] r_i delta) base^i, then the forward NTT."""
    out, s = np.empty(coeff.size, np.uint64), 1
    for i, c in enumerate(coeff):
        v = int(c) + (oracle.mul(int(rand[i]), delta) if i < len(rand) else 0)
        out[i] = oracle.mul(v % P, s)
        s = oracle.mul(s, base)
    return oracle.ntt(out)


def check(T, oracle, n, cols, k, in_place, picked):
    toff, base = 3, oracle.mul(7, oracle.root_of_unity(9))
    delta = (oracle.pow(base, n) - oracle.pow(toff, n)) % P
    d, r = T.empty(n * cols), T.empty(max(1, k * cols))
    T.lib.fill_uniform(d, n * cols, 10 + n)
    if k:
        T.lib.fill_uniform(r, k * cols, 20 + k)
    coeff = {c: d.download(n, c * n) for c in picked}
    out = d if in_place else T.empty(n * cols)
    T.lib.evaluate_coset(d, cols, n, r if k else None, k, toff, base, out)
    for c in picked:
        rand = r.download(k, c * k) if k else []
        assert np.array_equal(out.download(n, c * n), scaled(oracle, coeff[c], rand, delta, base)), c


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("n,cols,k", [(1, 300, 1), (2, 131, 2), (8, 513, 3), (16, 257, 5), (32, 129, 32),
                                      (64, 65, 7), (256, 17, 98), (2048, 3, 98), (4096, 2, 4096)])
def test_evaluate_short_columns(T, oracle, n, cols, k, in_place):
    picked = range(cols) if n * cols < 5000 else (0, cols // 2, cols - 1)
    check(T, oracle, n, cols, k, in_place, picked)


def test_evaluate_more_columns_than_blocks(T, oracle):
    cols = (1 << 24) + 3
    check(T, oracle, 4, cols, 1, False, (0, 1, 2, 4, 255, 256, 1 << 20, (1 << 24) - 1, 1 << 24, cols - 1))
