"""The k-means assignment's variants at their edges, bit for bit against the
CPU restatement: centers split over four waves (few objects, k from 16 on),
one and two objects per lane, group sizes around the tiles of 64, 128, 256 and
512 objects, duplicates (ties go to the lower cluster), values beyond the
fixed-point clamp, and a pass limit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def features(rng, n):
    f = rng.normal(0, 3, (max(n // 8, 1), 9))[rng.integers(0, max(n // 8, 1), n)]
    return (f + rng.normal(0, 0.3, (n, 9))).astype(np.float32)


def compare(oracle, f, off, k, seed, max_pass=501):
    import geaxdock_gpu_amd as gd
    with gd.Engine() as eng:
        med, sz, ps = eng.kmeans_medoids(f, off, k, seed=seed, max_pass=max_pass)
    for g in range(len(off) - 1):
        _, om, osz, op = oracle.kmeans(f[off[g]:off[g + 1]], k, group=g, level=0, seed=seed,
                                       max_pass=max_pass)
        assert np.array_equal(med[g], om) and np.array_equal(sz[g], osz), g
        if off[g + 1] - off[g] >= k:
            assert ps[g] == op, g


@pytest.mark.parametrize("k", [1, 15, 16, 17, 63, 130, 512])
def test_few_objects(oracle, k):
    rng = np.random.default_rng(k)
    sizes = [k, 63, 64, 65, 129, 255, 257, 600, 1025]
    parts = [features(rng, n) for n in sizes]
    parts[5][100:200] = parts[5][:100]
    parts[6][::7] *= 1e8
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    compare(oracle, np.concatenate(parts), off, k, seed=k)


@pytest.mark.parametrize("n_groups,k", [(700, 5), (2200, 3)])
def test_many_objects(oracle, n_groups, k):
    """Over two waves of objects per CU (unsplit centers), then over 32 (two
    objects per lane)."""
    rng = np.random.default_rng(n_groups)
    sizes = rng.integers(200, 290, n_groups)
    sizes[:4] = [511, 512, 513, 1]
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    compare(oracle, features(rng, int(off[-1])), off, k, seed=5, max_pass=4)
