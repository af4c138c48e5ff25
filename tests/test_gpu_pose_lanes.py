"""Large pose sets of contexts with few ladders use fewer lanes per pose.

Under spread packing a complex's lane shape is widened; enough poses to fill
the chip without that are evaluated with the shape of fewest lane slots, adding
in the wide shape's order. Energies must have the bits of the wide shape, which
small calls use: for every pair of shapes (2 or 3 atoms per narrow lane in 2, 4
and 8 times as many wide lanes), atom counts at the edges of the shapes, and
receptors of a few points to a few thousand, in LDS and in tiles.
"""
import numpy as np
import pytest

from geaxdock_gpu_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gd():
    import geaxdock_gpu_amd as g
    return g


# ladders x temperatures set the wide shape; the narrow one follows from lna
@pytest.mark.parametrize("pnp,pnk,pos,tile", [(3, 0, 0, 0), (402, 60, 3, 0), (2501, 700, 21, 0),
                                              (1501, 60, 3, 200), (6003, 60, 3, 0)])
@pytest.mark.parametrize("lna,n_lig,n_tmp", [(9, 1, 8), (16, 1, 4), (17, 2, 8), (24, 3, 1),
                                             (25, 1, 8), (31, 2, 8), (32, 1, 8), (33, 1, 2),
                                             (40, 20, 8), (44, 17, 8), (48, 2, 8), (49, 1, 8),
                                             (50, 40, 8), (64, 1, 8), (64, 30, 8)])
def test_many_poses_equal_small_calls(gd, lna, n_lig, n_tmp, pnp, pnk, pos, tile):
    cx = synth.make_complex(70 + lna, lna=lna, pnp=pnp, pnk=pnk, pos=pos, mcs_atoms=min(5, lna),
                            n_lig=n_lig, n_prt=2, n_tmp=n_tmp, void_radius=3.0)
    n, small = 8 * 256 + 37, 100
    rng = np.random.default_rng(lna + pnp)
    mm = np.zeros((n, 6), np.float32)
    mm[:, :3] = rng.normal(0.0, 2.0, (n, 3))
    mm[:, 3:] = rng.uniform(-np.pi, np.pi, (n, 3))
    il, ip = (rng.integers(0, k, n).astype(np.int32) for k in (n_lig, 2))
    with gd.Engine(seed=3, receptor_tile=tile) as e:
        e.add_complex(cx)
        got = e.calc_energy(0, il, ip, mm)
        want = [e.calc_energy(0, il[b:b + small], ip[b:b + small], mm[b:b + small])
                for b in range(0, n, small)]
    assert got.tobytes() == np.concatenate(want).tobytes()
