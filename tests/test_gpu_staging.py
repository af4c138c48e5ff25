"""Calls through the context's kept staging: results do not depend on the size
at which a call goes from direct host access to copies, on the order of small
and large calls, or on record rings that grew between runs; a sink may call
back into the engine while a window runs."""
import numpy as np
import pytest

from geaxdock_gpu_amd import abi, synth

pytestmark = pytest.mark.gpu


def poses(n, seed=0):
    rng = np.random.default_rng(seed)
    mm = np.zeros((n, 6), np.float32)
    mm[:, :3] = rng.normal(0.0, 1.0, (n, 3))
    mm[:, 3:] = rng.uniform(-np.pi, np.pi, (n, 3))
    return (rng.integers(0, 2, n).astype(np.int32), rng.integers(0, 2, n).astype(np.int32), mm)


@pytest.mark.parametrize("launch", [0, abi.LAUNCH_NO_SPREAD])
def test_scores_do_not_depend_on_the_call(launch):
    import geaxdock_gpu_amd as gd
    cx = synth.make_complex(11, lna=21, pnp=400, pnk=30, pos=3, mcs_atoms=5, n_lig=2, n_prt=2,
                            n_tmp=3, void_radius=6.0)
    il, ip, mm = poses(3000)
    with gd.Engine(seed=1, launch=launch) as eng:
        cid = eng.add_complex(cx)
        whole = eng.calc_energy(cid, il, ip, mm)
        for n in (1, 2, 640, 700, 760, 800, 801, 1200, 5):
            got = eng.calc_energy(cid, il[:n], ip[:n], mm[:n])
            assert got.tobytes() == whole[:n].tobytes(), n
            na = eng.calc_energy_noalloc(cid, il[:n], ip[:n], mm[:n])
            assert na.tobytes() == got.tobytes(), n


@pytest.mark.parametrize("launch", [0, abi.LAUNCH_NO_SPREAD])
def test_record_rings_grow_between_runs(launch):
    import geaxdock_gpu_amd as gd
    cx = synth.make_complex(12, lna=18, pnp=300, pnk=30, pos=2, mcs_atoms=5, n_lig=3, n_prt=2,
                            n_tmp=4)
    out = []
    for steps in ([20, 7, 13, 0, 260], [300]):
        by_rep = {}

        def sink(cid, recs):
            for r in recs:
                by_rep.setdefault(int(r["replica"][0]), []).append(r.tobytes())

        with gd.Engine(seed=5, steps_per_dump=90, launch=launch) as eng:
            eng.add_complex(cx)
            for k in steps:
                eng.run(k, 20, sink=sink)
            st = eng.state(0)
        out.append((by_rep, {k: v.tobytes() for k, v in st.items()}))
    assert out[0] == out[1]


def test_run_splits_records_by_replica():
    import geaxdock_gpu_amd as gd
    cx = synth.make_complex(13, lna=18, pnp=300, pnk=30, pos=2, mcs_atoms=5, n_lig=5, n_prt=2,
                            n_tmp=2)
    recs, log = gd.run(cx, 120, 20, seed=9, steps_per_dump=50)
    assert sorted(recs) == list(range(cx.n_rep))
    for r, v in recs.items():
        assert np.all(v["replica"][:, 0] == r)
        assert np.all(np.diff(v["step"][1:]) > 0)
    assert sum(len(v) for v in recs.values()) == round(log["ar"] * cx.n_rep * 120)


def test_sink_may_call_back():
    import geaxdock_gpu_amd as gd
    cx = synth.make_complex(14, lna=18, pnp=300, pnk=30, pos=2, mcs_atoms=5, n_lig=4, n_prt=2,
                            n_tmp=4)
    il, ip, mm = poses(900, seed=3)
    res = []
    for call_back in (False, True):
        with gd.Engine(seed=5, steps_per_dump=40, launch=abi.LAUNCH_NO_SPREAD) as eng:
            eng.add_complex(cx)
            seen = []

            def sink(cid, recs):
                seen.append(recs.tobytes())
                if call_back:
                    eng.state(0)
                    eng.calc_energy(0, il, ip, mm)

            st = eng.run(200, 20, sink=sink)
            res.append((seen, st["accepted"], st["exchanges_accepted"],
                        eng.state(0)["movematrix"].tobytes()))
    assert res[0] == res[1]
