"""Small contexts take several MC steps a launch through a tree of energies.

Persistent launches step one at a time, so both must leave the same bits:
states, best poses, records and counts. The packs of a context set the depth
(6 steps for 4 packs or fewer, 2 for 85, none beyond), exchange intervals and
run lengths that it does not divide leave shorter trees, and trees span
exchanges.
"""
import numpy as np
import pytest

from geaxdock_gpu_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gd():
    import geaxdock_gpu_amd as g
    return g


def _result(gd, cxs, persistent, runs, record, **kw):
    launch = abi.LAUNCH_SPREAD | (abi.LAUNCH_PERSISTENT if persistent else 0)
    out = []
    with gd.Engine(seed=9, launch=launch, record=record, **kw) as e:
        for cx in cxs:
            e.add_complex(cx)
        for steps, nc in runs:
            recs = []
            st = e.run(steps, nc, sink=(lambda c, r: recs.append((c, r.tobytes())))
                       if record else None)
            out.append((st["accepted"], st["exchanges_accepted"], recs))
        for c in range(len(cxs)):
            s = e.state(c)
            out += [s[k].tobytes() for k in sorted(s)] + [b.tobytes() for b in e.best(c)]
    return out


# (lna, receptor points, ligand and receptor conformers, temperatures, lanes,
# atoms per lane): packs 1, 4, 8, 9, 17, 36, 37, 85, 86, then ladders of more
# replicas than a workgroup has waves
SHAPES = [(8, 40, 1, 1, 1, 8, 1), (30, 300, 1, 1, 8, 32, 1), (60, 700, 1, 1, 8, 64, 1),
          (29, 500, 3, 3, 4, 16, 2), (48, 2501, 17, 1, 3, 16, 3), (61, 900, 6, 3, 8, 16, 4),
          (20, 130, 37, 1, 2, 32, 1), (16, 60, 17, 5, 2, 16, 1), (16, 60, 43, 2, 2, 16, 1),
          (30, 300, 1, 1, 13, 32, 1), (15, 60, 2, 1, 40, 8, 2)]


@pytest.mark.parametrize("record", [True, False])
@pytest.mark.parametrize("lna,pnp,n_lig,n_prt,n_tmp,lpr,apl", SHAPES)
def test_tree_equals_single_steps(gd, lna, pnp, n_lig, n_prt, n_tmp, lpr, apl, record):
    cx = synth.make_complex(lna, lna=lna, pnp=pnp, pnk=30, pos=2, mcs_atoms=5, n_lig=n_lig,
                            n_prt=n_prt, n_tmp=n_tmp, void_radius=3.0)
    kw = dict(lanes_per_replica=lpr, atoms_per_lane=apl, steps_per_dump=31)
    runs = [(47, 20), (1, 7), (13, 0), (9, 1), (17, 3)]
    assert (_result(gd, [cx], False, runs, record, **kw)
            == _result(gd, [cx], True, runs, record, **kw))


@pytest.mark.parametrize("kw", [dict(), dict(receptor_tile=64)])
def test_tree_of_several_complexes(gd, kw):
    # launch classes of different lane shapes, uniform and Gaussian moves
    cxs = [synth.make_complex(i, lna=lna, pnp=pnp, pnk=30, pos=3, mcs_atoms=5, n_lig=2, n_prt=1,
                              n_tmp=4, void_radius=3.0, move_kind=kind)
           for i, (lna, pnp, kind) in enumerate([(10, 200, abi.MOVE_UNIFORM),
                                                 (33, 801, abi.MOVE_GAUSSIAN),
                                                 (90, 333, abi.MOVE_UNIFORM)])]
    runs = [(45, 20), (6, 4)]
    assert _result(gd, cxs, False, runs, True, **kw) == _result(gd, cxs, True, runs, True, **kw)
