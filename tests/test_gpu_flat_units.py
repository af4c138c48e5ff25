"""The flat pair loop of spread packing against the chunk loop.

A context with a fixed receptor split of 8 sums every chunk with the chunk
loop; spread packing (also a split of 8, same forced lane shape) walks unit
lists. Both add the same terms in the same order, so energies and whole runs
must agree bit for bit. Sizes go through the lists' edges: groups with no
points, one point, single units, units across chunks, groups of two and four
points; receptors reach into the ligand, so the near electrostatic corrections
and the contacts run.
"""
import numpy as np
import pytest

from geaxdock_gpu_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gd():
    import geaxdock_gpu_amd as g
    return g


def engines(gd, cx, lpr, apl):
    kw = dict(seed=3, lanes_per_replica=lpr, atoms_per_lane=apl)
    a = gd.Engine(receptor_split=8, **kw)
    b = gd.Engine(launch=abi.LAUNCH_SPREAD, **kw)
    for e in (a, b):
        e.add_complex(cx)
    return a, b


@pytest.mark.parametrize("pnp", [1, 7, 67, 300, 1200, 2501])
@pytest.mark.parametrize("lpr,apl,lna", [(8, 1, 8), (32, 1, 27), (64, 1, 64), (16, 2, 29),
                                         (32, 2, 61), (16, 3, 44), (8, 4, 31)])
def test_energies_equal_the_chunk_loop(gd, lpr, apl, lna, pnp):
    cx = synth.make_complex(100 + pnp, lna=lna, pnp=pnp, pnk=40, pos=3, mcs_atoms=5, n_lig=2,
                            n_prt=2, n_tmp=1, void_radius=1.5, identity_norm=True)
    rng = np.random.default_rng(pnp + lpr)
    n = 60
    mm = np.zeros((n, 6), np.float32)
    mm[:, :3] = rng.normal(0.0, 2.0, (n, 3))
    mm[:, 3:] = rng.uniform(-np.pi, np.pi, (n, 3))
    il, ip = rng.integers(0, 2, n).astype(np.int32), rng.integers(0, 2, n).astype(np.int32)
    a, b = engines(gd, cx, lpr, apl)
    with a, b:
        ea, eb = a.calc_energy(0, il, ip, mm), b.calc_energy(0, il, ip, mm)
    assert ea.tobytes() == eb.tobytes()


@pytest.mark.parametrize("lpr,apl,lna,n_tmp", [(16, 1, 15, 4), (32, 1, 30, 2), (16, 2, 32, 4),
                                               (8, 3, 23, 8), (8, 4, 30, 8)])
def test_runs_equal_the_chunk_loop(gd, lpr, apl, lna, n_tmp):
    cx = synth.make_complex(7, lna=lna, pnp=611, pnk=90, pos=5, mcs_atoms=9, n_lig=3, n_prt=2,
                            n_tmp=n_tmp, void_radius=6.0)
    a, b = engines(gd, cx, lpr, apl)
    with a, b:
        out = []
        for e in (a, b):
            recs = []
            e.run(60, 20, sink=lambda c, r: recs.append(r))
            st = e.state(0)
            out.append([np.concatenate(recs).tobytes()] + [st[k].tobytes() for k in sorted(st)])
    assert out[0] == out[1]
