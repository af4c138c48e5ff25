"""The chunk loop with and without distance tests.

Launches of at most 256 lanes a workgroup go without the tests, wider ones of
receptors with many far points take them. Both skip nothing but exact zeros, so
poses evaluated one at a time and together, and runs of one and of two ladders
a workgroup, agree bit for bit at the same split.
"""
import numpy as np
import pytest

from geaxdock_gpu_amd import surrogate as sg
from geaxdock_gpu_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gd():
    import geaxdock_gpu_amd as g
    return g


# lanes, atoms per lane, ligand atoms, temperatures: a ladder of two waves
SHAPES = [(32, 1, 30, 4), (16, 2, 29, 8), (32, 2, 61, 4), (16, 3, 44, 8), (16, 4, 62, 8)]


@pytest.mark.parametrize("pnp,tile,pos,da", [(1, 0, 3, False), (700, 0, 3, False),
                                             (3501, 0, 3, False), (3501, 256, 3, False),
                                             (3501, 0, 3, True), (3501, 0, 40, True)])
@pytest.mark.parametrize("lpr,apl,lna,n_tmp", SHAPES)
def test_one_and_two_ladders_a_workgroup(gd, lpr, apl, lna, n_tmp, pnp, tile, pos, da):
    cx = synth.make_complex(pnp, lna=lna, pnp=pnp, pnk=40, pos=pos, mcs_atoms=5, n_lig=4, n_prt=2,
                            n_tmp=n_tmp, void_radius=4.0)
    out = []
    for ladders in (1, 2):
        with gd.Engine(seed=4, receptor_split=2, ladders_per_pack=ladders, receptor_tile=tile,
                       lanes_per_replica=lpr, atoms_per_lane=apl) as e:
            e.add_complex(cx)
            recs = []
            if da:  # 40 templates: the split's groups share the surrogate's sums
                e.sur_build_grids(1.0, 8.0)
                e.sur_set_params(sg.pack_params(sg.init_params(2)))
                e.sur_tabulate()
                e.run_da(40, 20, 4, 2.0, sink=lambda c, r: recs.append(r))
            else:
                e.run(40, 20, sink=lambda c, r: recs.append(r))
            st = e.state(0)
            out.append([np.concatenate(recs).tobytes()] + [st[k].tobytes() for k in sorted(st)])
    assert out[0] == out[1]


@pytest.mark.parametrize("split", [1, 4])
@pytest.mark.parametrize("lpr,apl,lna,n_tmp", SHAPES)
def test_poses_alone_and_together(gd, lpr, apl, lna, n_tmp, split):
    cx = synth.make_complex(9, lna=lna, pnp=3300, pnk=40, pos=3, mcs_atoms=5, n_lig=2, n_prt=2,
                            n_tmp=2, void_radius=4.0)
    rng = np.random.default_rng(lna)
    n = 33
    mm = np.zeros((n, 6), np.float32)
    mm[:, :3] = rng.normal(0.0, 1.0, (n, 3)) * np.linspace(0.0, 25.0, n)[:, None]
    mm[:, 3:] = rng.uniform(-np.pi, np.pi, (n, 3))
    il, ip = np.arange(n, dtype=np.int32) % 2, np.arange(n, dtype=np.int32) // 2 % 2
    with gd.Engine(seed=4, receptor_split=split, lanes_per_replica=lpr, atoms_per_lane=apl) as e:
        e.add_complex(cx)
        many = e.calc_energy(0, np.repeat(il, 9), np.repeat(ip, 9), np.repeat(mm, 9, axis=0))
        one = np.concatenate([e.calc_energy(0, il[i:i + 1], ip[i:i + 1], mm[i:i + 1])
                              for i in range(n)])
    assert np.repeat(one, 9).tobytes() == many.tobytes()
