"""k-means whose workgroups gather their changes in LDS, bit for bit against the
CPU restatement: up to 128 centers with the objects alone filling the chip, and
up to 15 centers with several tiles a workgroup (groups of thousands of
objects), one and two objects per lane, group sizes around the tiles."""
import numpy as np
import pytest

from test_gpu_kmeans_tiles import compare, features

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [2, 15, 16, 128, 129])
@pytest.mark.parametrize("sizes", [[16383, 16384, 16385, 33000, 32768, 17000, 1025],
                                   [65537, 131072, 40000, 300000, 1]])
def test_gathered_sums(oracle, k, sizes):
    rng = np.random.default_rng(k)
    parts = [features(rng, n) for n in sizes]
    parts[0][::11] *= 1e8  # beyond the fixed-point clamp
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    compare(oracle, np.concatenate(parts), off, k, seed=k, max_pass=4)
