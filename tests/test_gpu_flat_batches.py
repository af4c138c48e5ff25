"""The flat pair loop of batches against the chunk loop.

Outside spread packing the automatic split takes unit lists where the lane
groups' shares of a chunk are short; a fixed split keeps the chunk loop. Both
add the same terms in the same order, so energies and whole runs agree bit for
bit at the same split (ladders of 1, 2 and 4 waves: splits of 8, 4 and 2).
Receptors go from one point to a few thousand, in contexts of several complexes
of different sizes.
"""
import numpy as np
import pytest

from geaxdock_gpu_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gd():
    import geaxdock_gpu_amd as g
    return g


SHAPES = [(8, 1, 8, 8, 8), (16, 1, 15, 8, 4), (32, 1, 30, 4, 4), (16, 2, 29, 16, 2),
          (32, 2, 61, 8, 2), (16, 3, 44, 4, 8), (16, 4, 62, 8, 4)]


@pytest.mark.parametrize("lpr,apl,lna,n_tmp,ns", SHAPES)
def test_batches_equal_the_chunk_loop(gd, lpr, apl, lna, n_tmp, ns):
    cxs = [synth.make_complex(20 + i, lna=lna, pnp=pnp, pnk=40 + i, pos=3, mcs_atoms=5, n_lig=2,
                              n_prt=1 + i % 2, n_tmp=n_tmp, void_radius=3.0)
           for i, pnp in enumerate((1, 13, 402, 1501, 2502))]
    rng = np.random.default_rng(lpr + ns)
    n = 40
    mm = np.zeros((n, 6), np.float32)
    mm[:, :3] = rng.normal(0.0, 2.0, (n, 3))
    mm[:, 3:] = rng.uniform(-np.pi, np.pi, (n, 3))
    kw = dict(seed=5, lanes_per_replica=lpr, atoms_per_lane=apl, ladders_per_pack=0)
    out = []
    for extra in (dict(receptor_split=ns, ladders_per_pack=1), dict(launch=abi.LAUNCH_NO_SPREAD)):
        with gd.Engine(**{**kw, **extra}) as e:
            for cx in cxs:
                e.add_complex(cx)
            got = [e.calc_energy(c, np.arange(n, dtype=np.int32) % 2, np.zeros(n, np.int32),
                                 mm).tobytes() for c in range(len(cxs))]
            e.run(40, 20)
            for c in range(len(cxs)):
                st = e.state(c)
                got += [st[k].tobytes() for k in sorted(st)]
            out.append(got)
    assert out[0] == out[1]
