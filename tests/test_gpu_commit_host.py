"""The host form of the commit checks its inputs beside the GPU's work: an element
that is not canonical is refused, wherever it is, with the outputs as they were."""
import numpy as np
import pytest

from conftest import P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("where", ["first", "last", "rand"])
def test_commit_host_refuses_late_elements(T, oracle, where):
    n, cols, k = 64, 3, 5
    m = 4 * n
    trace, rand = oracle.splitmix(1, n * cols), oracle.splitmix(2, k * cols)
    bad_trace, bad_rand = trace.copy(), rand.copy()
    if where == "rand":
        bad_rand[-1] = P + 1
    else:
        bad_trace[0 if where == "first" else -1] = P
    cw, dg, root = (np.full(c, 7, np.uint64) for c in (m * cols, 5 * m, 5))
    with pytest.raises(RuntimeError, match=">= p"):
        T.lib.commit_host(bad_trace, cols, n, m, 1, 7, rand=bad_rand, k=k, codewords=cw, digests=dg,
                          root=root)
    assert (cw == 7).all() and (dg == 7).all() and (root == 7).all()
    T.lib.commit_host(trace, cols, n, m, 1, 7, rand=rand, k=k, codewords=cw, digests=dg, root=root)
    want = oracle.lde_table(trace, n, cols, m, 1, 7, rand.reshape(cols, k))
    assert np.array_equal(cw, np.asarray(want).reshape(-1))
