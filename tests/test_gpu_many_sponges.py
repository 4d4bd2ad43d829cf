"""Hashing calls of more than 2^30 sponges: a sponge takes four threads and more,
so their launches pass the 2^32 threads that one grid axis can have."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COUNT = (1 << 30) + 17


def spots(rng):
    """Places at both ends, round 2^30 and between."""
    around = [0, 1, 63, 64, (1 << 23) * 64 - 1, (1 << 29) + 5, (1 << 30) - 1, 1 << 30, COUNT - 1]
    return around + [int(v) for v in rng.randint(0, COUNT, 20)]


@pytest.mark.parametrize("form", ["rows", "pairs"])
def test_hash_more_than_2p30(T, oracle, form):
    if T.mod.hip_rt.mem_info()[0] < 110 << 30:
        pytest.skip("needs 110 GiB of free device memory")
    rng = np.random.RandomState(3)
    width = 1 if form == "rows" else 5
    x, dg = T.empty(COUNT * width), T.empty(COUNT * 5)
    places = spots(rng)  # (the elements between hold what the memory held)
    for i in places:
        T.lib.fill_uniform(x.view(i * width, width), width, 1000 + i)
    if form == "rows":
        T.lib.hash_bfield_rows(x, COUNT, 1, dg)
    else:
        T.lib.hash_pairs(x, x, dg, COUNT)
    T.sync()
    for i in places:
        v = x.download(width, i * width)
        want = oracle.hash_rows(v, 1, 1)[0] if form == "rows" else oracle.hash_pair(v, v)
        assert np.array_equal(dg.download(5, 5 * i), np.asarray(want).reshape(-1)), i
