"""Tip5 on the values that leave the kernels' usual path, at the edges of their
16-sponge waves and 64-sponge blocks, against the oracle (bit for bit).

The kernels fold products with one branch for the borrow that a random product
takes once in 2^32.  State words that are powers of two in Montgomery form take
it in the first round (the product's low half is zero), table elements with a
zero low word take it on the way into Montgomery form.
"""
import numpy as np
import pytest

from conftest import P

pytestmark = pytest.mark.gpu

R_INV = pow(1 << 64, P - 2, P)


def edge_words(seed, count):
    """Words whose Montgomery form is 2^k, 0, 1, p - 1 or near a word border,
    elements that are such numbers themselves, and random ones between."""
    mont = [1 << k for k in range(64)] + [0, 1, P - 1, P - 2, (1 << 32) - 1, (1 << 32) + 1,
                                          P - (1 << 32), P - (1 << 32) - 1]
    plain = [v % P for v in mont] + [c << 32 for c in (3, 0xFFFFFFFE, 0x80000000)]
    pool = np.array([m * R_INV % P for m in mont] + plain, np.uint64)
    g = np.random.RandomState(seed)
    words = pool[g.randint(0, pool.size, count)]
    rnd = g.randint(0, P, count, dtype=np.uint64)
    return np.where(g.randint(0, 4, count) == 0, rnd, words)


@pytest.mark.parametrize("count", [1, 15, 16, 17, 63, 64, 65, 400])
def test_permutation_edge_words(T, oracle, count):
    st = edge_words(count, 16 * count).reshape(count, 16)
    d = T.dev(st.reshape(-1))
    T.lib.permutation_batch(d, count)
    want = np.array([oracle.permutation(s) for s in st], np.uint64)
    assert np.array_equal(T.host(d).reshape(count, 16), want)


@pytest.mark.parametrize("rows,cols", [(1, 9), (17, 10), (64, 11), (65, 29), (130, 38)])
def test_hash_rows_edge_words(T, oracle, rows, cols):
    t = edge_words(rows + cols, rows * cols)
    dg = T.empty(rows * 5)
    T.lib.hash_bfield_rows(T.dev(t), rows, cols, dg)
    assert np.array_equal(T.host(dg, rows * 5).reshape(rows, 5), oracle.hash_rows(t, rows, cols))


@pytest.mark.parametrize("logn", [6, 7, 11, 16, 18])
def test_merkle_edge_leaves(T, oracle, logn):
    """One block, several blocks, several launches (2^16 nodes is the last level
    whose parents share launches), whole levels before them."""
    n = 1 << logn
    leaves = edge_words(logn, 5 * n)
    tree = T.empty(5 * (2 * n - 1))
    T.lib.merkle_tree(T.dev(leaves), tree, n, 0)
    want = oracle.merkle_level_order(leaves.reshape(n, 5))
    assert np.array_equal(T.host(tree).reshape(-1), np.asarray(want).reshape(-1))


@pytest.mark.parametrize("rows", [3, 4, 5, 16383, 16384, 16385])
def test_hash_rows_few_and_many(T, oracle, rows):
    """Four sponges to a wave up to 2^14 rows, 16 above: partial waves of both."""
    cols = 21
    t = edge_words(rows, rows * cols)
    dg = T.empty(rows * 5)
    T.lib.hash_bfield_rows(T.dev(t), rows, cols, dg)
    assert np.array_equal(T.host(dg, rows * 5).reshape(rows, 5), oracle.hash_rows(t, rows, cols))


@pytest.mark.parametrize("logn", [1, 3, 14, 15])
def test_merkle_few_parents(T, oracle, logn):
    """Levels of up to 2^14 parents, four to a wave; 2^15 leaves are the largest
    tree of only such levels."""
    n = 1 << logn
    leaves = edge_words(40 + logn, 5 * n)
    tree = T.empty(5 * (2 * n - 1))
    T.lib.merkle_tree(T.dev(leaves), tree, n, 0)
    want = oracle.merkle_level_order(leaves.reshape(n, 5))
    assert np.array_equal(T.host(tree).reshape(-1), np.asarray(want).reshape(-1))
