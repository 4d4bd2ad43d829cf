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
