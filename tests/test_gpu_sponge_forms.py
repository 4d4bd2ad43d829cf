"""Tip5 entry points on both sides of the count where the kernels change from four
sponges a wave to sixteen, and where blocks take several sets of states: partial
waves, blocks and sets, against the oracle (bit for bit)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SETS = 2048 * 64  # states that one set to each block takes


@pytest.mark.parametrize("num,first,count,traced", [
    (1, 0, 5, True), (17, 2, 2, True), (65, 4, 1, False), (3, 5, 0, True),
    (SETS, 1, 1, False), (SETS + 1, 3, 2, False), (3 * SETS + 64 + 5, 0, 5, False), (SETS + 65, 2, 1, True)])
def test_rounds(T, oracle, num, first, count, traced):
    st = T.empty(16 * num)
    T.lib.fill_uniform(st, 16 * num, num)
    before = T.host(st, 16 * num).reshape(num, 16)
    trace = T.empty(16 * num * (count + 1)) if traced else None
    T.lib.tip5_rounds(st, num, first, count, trace)
    after = T.host(st, 16 * num).reshape(num, 16)
    tr = T.host(trace, 16 * num * (count + 1)).reshape(num, count + 1, 16) if traced else None
    step = max(1, num // 2000)
    for i in sorted(set(range(0, num, step)) | set(range(max(0, num - 70), num))):
        want = before[i]
        for r in range(count + 1):
            if traced:
                assert np.array_equal(tr[i, r], want), (i, r)
            if r < count:
                want = oracle.tip5_round(want, first + r)
        assert np.array_equal(after[i], want), i


@pytest.mark.parametrize("num", [16384, 16385, 16400, 20011])
def test_permutation_few_and_many(T, oracle, num):
    st = oracle.splitmix(num, 16 * num).reshape(num, 16)
    d = T.dev(st.reshape(-1))
    T.lib.permutation_batch(d, num)
    got = T.host(d, 16 * num).reshape(num, 16)
    for i in list(range(0, num, 37)) + list(range(num - 70, num)):
        assert np.array_equal(got[i], oracle.permutation(st[i])), i


@pytest.mark.parametrize("num", [1, 16384, 16385, 16430, 20011])
def test_pairs_few_and_many(T, oracle, num):
    l, r = oracle.splitmix(num, 5 * num).reshape(num, 5), oracle.splitmix(num + 1, 5 * num).reshape(num, 5)
    out = T.empty(5 * num)
    T.lib.hash_pairs(T.dev(l.reshape(-1)), T.dev(r.reshape(-1)), out, num)
    got = T.host(out, 5 * num).reshape(num, 5)
    for i in sorted(set(range(0, num, 37)) | set(range(max(0, num - 70), num))):
        assert np.array_equal(got[i], oracle.hash_pair(l[i], r[i])), i


@pytest.mark.parametrize("log_n,E", [(12, 4), (13, 2), (13, 4)])
@pytest.mark.parametrize("cols,chunk,k", [(23, 1, 0), (40, 7, 98), (75, 64, 98), (9, 20, 5), (41, 10, 0), (33, 32, 98)])
def test_streamed_commit_few_and_many_rows(T, oracle, log_n, E, cols, chunk, k):
    """Rows absorbed in chunks of columns: 2^14 rows are the last in four-sponge waves,
    2^15 go in sixteens.  The tree equals the plain commit's and its first, middle
    and last leaves the oracle's row hashes."""
    n, m = 1 << log_n, E << log_n
    x, r = T.empty(n * cols), T.empty(max(1, k * cols))
    T.lib.fill_uniform(x, n * cols, 5)
    T.lib.fill_uniform(r, max(1, k * cols), 6)
    rand = r if k else None
    cw, want = T.empty(m * cols), T.empty(5 * (2 * m - 1))
    T.lib.commit(x, cols, n, rand, k, 1, 7, m, cw, want)
    work, tree = T.empty(T.lib.frugal_workspace_elems(cols, n, m, chunk)), T.empty(5 * (2 * m - 1))
    T.lib.commit_frugal(x, cols, n, rand, k, 1, 7, m, chunk, work, tree)
    assert np.array_equal(T.host(tree, 5 * (2 * m - 1)), T.host(want, 5 * (2 * m - 1)))
    for row in (0, 15, 16, m // 2, m - 1):
        digest = oracle.hash_varlen(cw.gather_strided(row, m, cols))
        assert np.array_equal(tree.download(5, 5 * row), digest), row
