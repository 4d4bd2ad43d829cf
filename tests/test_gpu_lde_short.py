"""LDEs of short columns and of many cosets, against the oracle (bit for bit).

Columns of up to 16 elements: 256 outputs, several whole columns, to a matrix
product, the last one not full, one product and several to a wave.  Splits whose
rows would fall below 2^5 elements: 2^11 rows in 16 cosets, 2^12 in 8 and 16, and
2^9 in 16 under the smallest row tile.  The same tables in a batch plan.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("log_n,cols,k", [(0, 1, 1), (0, 257, 0), (1, 65, 2), (2, 33, 1), (3, 130, 8),
                                          (4, 1, 16), (4, 17, 5), (4, 1000, 0)])
def test_lde_short_columns(T, oracle, log_n, E, cols, k):
    n = 1 << log_n
    m = E * n
    x = oracle.splitmix(log_n + cols, n * cols)
    r = oracle.splitmix(7 + k, k * cols) if k else None
    out = T.empty(m * cols)
    T.lib.lde_batch(T.dev(x), cols, n, T.dev(r) if k else None, k, 3, 7, m, out)
    want = oracle.lde_table(x, n, cols, m, 3, 7, None if r is None else r.reshape(cols, k))
    assert np.array_equal(T.host(out, m * cols), np.asarray(want).reshape(-1))


def test_lde_short_several_products_a_wave(T, oracle):
    """2^16 columns of 16 rows in 4 cosets: 2^14 products and one in part."""
    n, E, cols, k = 16, 4, (1 << 16) + 1, 2
    x, r = T.empty(n * cols), T.empty(k * cols)
    T.lib.fill_uniform(x, n * cols, 1)
    T.lib.fill_uniform(r, k * cols, 2)
    out = T.empty(E * n * cols)
    T.lib.lde_batch(x, cols, n, r, k, 1, 7, E * n, out)
    for c in (0, 1, 255, 256, 511, 512, 40000, cols - 2, cols - 1):
        want = oracle.lde_table(x.download(n, c * n), n, 1, E * n, 1, 7, r.download(k, c * k).reshape(1, k))
        assert np.array_equal(out.download(E * n, c * E * n), np.asarray(want).reshape(-1)), c


@pytest.mark.parametrize("xfe_rand", [False, True])
def test_lde_short_xfe(T, oracle, xfe_rand):
    """Limb-major XFE columns (three limbs of a column share its randomizers' rules)
    give what the three B-field columns give one by one."""
    n, E, xcols, k = 8, 4, 21, 3
    x = oracle.splitmix(5, 3 * xcols * n).reshape(xcols, 3, n)
    r = oracle.splitmix(6, xcols * k * (3 if xfe_rand else 1)).reshape(xcols, k, -1)
    out = T.empty(3 * xcols * n * E)
    T.lib.lde_xfe_limbs(T.dev(x), xcols, n, T.dev(r), k, 1, 7, n * E, out, xfe_rand)
    got = T.host(out, 3 * xcols * n * E).reshape(xcols, 3, n * E)
    for c in range(xcols):
        for limb in range(3):
            rl = r[c, :, limb] if xfe_rand else (r[c, :, 0] if limb == 0 else np.zeros(k, np.uint64))
            want = oracle.lde_table(x[c, limb], n, 1, n * E, 1, 7, np.ascontiguousarray(rl).reshape(1, k))
            assert np.array_equal(got[c, limb], np.asarray(want).reshape(-1)), (c, limb)


@pytest.mark.parametrize("log_n,E,cols,k,variant", [(11, 16, 3, 98, 0), (12, 8, 3, 98, 0), (12, 16, 2, 300, 0),
                                                    (9, 16, 3, 98, 66), (9, 16, 3, 0, 74), (10, 16, 3, 40, 70)])
def test_lde_many_cosets(T, oracle, log_n, E, cols, k, variant):
    n = 1 << log_n
    m = E * n
    x = oracle.splitmix(log_n, n * cols)
    r = oracle.splitmix(k, k * cols) if k else None
    out = T.empty(m * cols)
    T.lib.lde_set_variant(log_n, E.bit_length() - 1, variant)
    try:
        T.lib.lde_batch(T.dev(x), cols, n, T.dev(r) if k else None, k, 1, 7, m, out)
    finally:
        T.lib.lde_set_variant(log_n, E.bit_length() - 1, 0)
    want = oracle.lde_table(x, n, cols, m, 1, 7, None if r is None else r.reshape(cols, k))
    assert np.array_equal(T.host(out), np.asarray(want).reshape(-1))


def test_batch_of_short_and_many_cosets(T, oracle):
    shapes = [(2, 2, 40, 1), (4, 16, 17, 5), (0, 8, 3, 0), (11, 16, 2, 98), (12, 8, 2, 98), (12, 16, 1, 98),
              (6, 4, 5, 3), (13, 4, 1, 0)]
    descs, tables = [], []
    for i, (log_n, E, cols, k) in enumerate(shapes):
        n, m = 1 << log_n, E << log_n
        x, r = oracle.splitmix(i, n * cols), oracle.splitmix(50 + i, max(1, k * cols))
        bufs = T.dev(x), T.dev(r), T.empty(m * cols), T.empty(5 * (2 * m - 1))
        descs.append(T.lib.table_desc(bufs[0], cols, n, m, bufs[2], bufs[3], rand=bufs[1] if k else None, k=k))
        tables.append((x, r, bufs))
    T.lib.commit_batch(descs)
    T.sync()
    for (log_n, E, cols, k), (x, r, bufs) in zip(shapes, tables):
        n, m = 1 << log_n, E << log_n
        want = oracle.lde_table(x, n, cols, m, 1, 7, r.reshape(cols, k) if k else None)
        assert np.array_equal(T.host(bufs[2], m * cols), np.asarray(want).reshape(-1)), (log_n, E)
        digests = oracle.hash_rows(np.asarray(want).reshape(-1), m, cols)
        tree = oracle.merkle_level_order(np.asarray(digests).reshape(m, 5))
        assert np.array_equal(T.host(bufs[3], 5 * (2 * m - 1)), np.asarray(tree).reshape(-1)), (log_n, E)


@pytest.mark.parametrize("log_n,E,E_few", [(4, 16, 1), (12, 16, 4)])
def test_cosets_are_not_in_turn(T, log_n, E, E_few):
    """Sixteen cosets of one short column (or of rows of a short split) run side by
    side: one after the other in each lane they took 7 times as long as the few."""
    n = 1 << log_n
    x, out = T.empty(n), T.empty(E * n)
    T.lib.fill_uniform(x, n, 1)
    rt = T.mod.hip_rt

    def best(e):
        T.lib.lde_prepare(n, e * n)
        t = []
        for _ in range(5):
            a, b = rt.Event(), rt.Event()
            a.record()
            for _ in range(20):
                T.lib.lde_batch(x, 1, n, None, 0, 1, 7, e * n, out)
            b.record()
            b.synchronize()
            t.append(a.elapsed_ms(b))
        return min(t)

    assert best(E) < 4 * best(E_few)


@pytest.mark.parametrize("log_n,E,cols,k", [(5, 2, 3, 32), (7, 1, 1, 98), (7, 4, 33, 98), (8, 8, 3, 200)])
def test_randomizers_of_a_part_filled_tile(T, oracle, log_n, E, cols, k):
    """The randomizer terms are spread over the rows that the tile holds, not over
    those it could hold (one column of 2^7 rows: 47 us, 14 with its terms alone)."""
    test_lde_short_columns(T, oracle, log_n, E, cols, k)


@pytest.mark.parametrize("log_n,E", [(22, 16), (23, 8)])
def test_lde_of_2p26(T, log_n, E):
    """Refused by default, taken by a variant with the 2^14 row tile; each coset is
    the coset evaluation of the column's coefficients."""
    n, m, log_e = 1 << log_n, E << log_n, E.bit_length() - 1
    x, coeff, one, out = T.empty(n), T.empty(n), T.empty(n), T.empty(m)
    T.lib.fill_uniform(x, n, 4)
    P = 0xFFFFFFFF00000001
    with pytest.raises(T.mod.TVHError, match="unsupported"):
        T.lib.lde_batch(x, 1, n, None, 0, 1, 7, m, out)
    T.lib.lde_set_variant(log_n, log_e, T.mod.LDE_SPLIT)
    try:
        T.lib.lde_batch(x, 1, n, None, 0, 1, 7, m, out)
    finally:
        T.lib.lde_set_variant(log_n, log_e, 0)
    T.lib.trace_coefficients(x, 1, n, 1, coeff)
    got = T.host(out, m)
    w = pow(7, (P - 1) // m, P)
    for s in (0, 1, E - 1):
        T.lib.evaluate_coset(coeff, 1, n, None, 0, 1, 7 * pow(w, s, P) % P, one)
        assert np.array_equal(T.host(one, n), got[s::E]), s
