"""Delayed acceptance through the flat pair loop against the chunk loop.

With tables, delayed acceptance takes unit lists where plain MC does: under
spread packing, and in batches whose shares of a chunk are short. A fixed split
keeps the chunk loop. Both add the same terms in the same order, so surrogate
totals and whole runs agree bit for bit at the same split, with the surrogate's
KDE and MCS sums shared by the split's groups (large lists) or not.
"""
import numpy as np
import pytest

from geaxdock_gpu_amd import abi, synth
from geaxdock_gpu_amd import surrogate as sg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gd():
    import geaxdock_gpu_amd as g
    return g


def _result(gd, cxs, **kw):
    n = 40
    rng = np.random.default_rng(4)
    mm = np.zeros((n, 6), np.float32)
    mm[:, :3] = rng.normal(0.0, 2.0, (n, 3))
    mm[:, 3:] = rng.uniform(-np.pi, np.pi, (n, 3))
    out, recs = [], []
    with gd.Engine(seed=6, **kw) as e:
        for cx in cxs:
            e.add_complex(cx)
        e.sur_build_grids(1.0, 8.0)
        e.sur_set_params(sg.pack_params(sg.init_params(3)))
        e.sur_tabulate()
        for c in range(len(cxs)):
            out.append(e.sur_surrogate(c, np.arange(n, dtype=np.int32) % 2, np.zeros(n, np.int32),
                                       mm, 2.0).tobytes())
        e.run_da(60, 20, 4, 2.0, sink=lambda c, r: recs.append((c, r.tobytes())))
        for c in range(len(cxs)):
            st = e.state(c)
            out += [st[k].tobytes() for k in sorted(st)] + [b.tobytes() for b in e.best(c)]
    return out + sorted(recs)


# lanes, atoms per lane, ligand atoms, temperatures, split
@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("lpr,apl,lna,n_tmp,ns", [(8, 1, 8, 8, 8), (16, 1, 15, 8, 4),
                                                  (32, 2, 61, 8, 2), (16, 3, 44, 4, 8),
                                                  (16, 4, 62, 8, 4)])
def test_batches_equal_the_chunk_loop(gd, lpr, apl, lna, n_tmp, ns, large):
    lists = dict(pnk=300, pos=36) if large else dict(pnk=40, pos=3)
    cxs = [synth.make_complex(70 + i, lna=lna, pnp=pnp, mcs_atoms=5, n_lig=2, n_prt=1 + i % 2,
                              n_tmp=n_tmp, void_radius=3.0, **lists)
           for i, pnp in enumerate((1, 402, 1501))]
    kw = dict(lanes_per_replica=lpr, atoms_per_lane=apl)
    assert (_result(gd, cxs, receptor_split=ns, ladders_per_pack=1, **kw)
            == _result(gd, cxs, launch=abi.LAUNCH_NO_SPREAD, **kw))


@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("lpr,apl,lna,n_tmp", [(32, 1, 30, 2), (16, 2, 32, 4), (8, 3, 23, 8),
                                               (8, 4, 30, 8)])
def test_spread_equals_the_chunk_loop(gd, lpr, apl, lna, n_tmp, large):
    lists = dict(pnk=300, pos=36) if large else dict(pnk=40, pos=3)
    cx = synth.make_complex(80, lna=lna, pnp=611, mcs_atoms=5, n_lig=2, n_prt=2, n_tmp=n_tmp,
                            void_radius=3.0, **lists)
    kw = dict(lanes_per_replica=lpr, atoms_per_lane=apl)
    assert _result(gd, [cx], receptor_split=8, **kw) == _result(gd, [cx], launch=abi.LAUNCH_SPREAD, **kw)
