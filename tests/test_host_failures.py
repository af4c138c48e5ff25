"""Host code of the engine when a device call fails: allocations and launches
fail where a case says so, on a HIP runtime of host memory that runs no kernel
(tests/cpp/host_hip.cpp). A failed call is an error; what the context does
afterwards must not use memory that is not there.

Each case runs in a process of its own, since the library binds its runtime once.
"""
import ctypes as C
import os
import struct
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


class HostHip:
    """The controls and records of host_hip.cpp."""

    def __init__(self, path):
        # global: the engine's library, loaded later, binds to these symbols
        self.lib = C.CDLL(path, mode=C.RTLD_GLOBAL)
        self.lib.host_hip_alloc_size.restype = C.c_size_t
        self.lib.host_hip_kernel.restype = C.c_char_p
        self.lib.host_hip_grid.restype = C.c_uint
        for f in ("num_allocs", "num_live", "num_made", "num_launches"):
            getattr(self.lib, "host_hip_" + f).restype = C.c_long

    def fail_alloc(self, n=0):
        self.lib.host_hip_fail_alloc(C.c_long(n))

    def fail_launch(self, n=0):
        self.lib.host_hip_fail_launch(C.c_long(n))

    def fail_above(self, size):
        self.lib.host_hip_fail_above(C.c_size_t(size))

    def count(self, what):
        return getattr(self.lib, "host_hip_num_" + what)()

    def allocs(self, begin=0):
        return [self.lib.host_hip_alloc_size(C.c_long(i))
                for i in range(begin, self.count("allocs"))]

    def launches(self, name="", begin=0):
        out = []
        for i in range(begin, self.count("launches")):
            k = self.lib.host_hip_kernel(C.c_long(i)).decode()
            if name in k:
                out.append((k, [self.lib.host_hip_grid(C.c_long(i), a) for a in range(3)],
                            bool(self.lib.host_hip_table(C.c_long(i)))))
        return out


def complex_(seed=1, **kw):
    from geaxdock_gpu_amd import synth
    return synth.make_complex(seed, **{**dict(lna=20, pnp=300, pnk=30, pos=3, mcs_atoms=5,
                                              n_lig=2, n_prt=1, n_tmp=4, void_radius=3.0), **kw})


def poses(n, n_lig=2):
    return (np.arange(n, dtype=np.int32) % n_lig, np.zeros(n, np.int32),
            np.zeros((n, 6), np.float32))


def fails(call, *status):
    """The call ends with one of these statuses."""
    import geaxdock_gpu_amd as gd
    from geaxdock_gpu_amd import abi
    with pytest.raises(gd.GeauxDockError) as e:
        call()
    assert abi.STATUS[e.value.status] in status, str(e.value)


def unit_lists(hip):
    """A unit list that found no memory is built by the next call; before, the
    launches of that call read the list through a null pointer."""
    import geaxdock_gpu_amd as gd
    with gd.Engine(seed=1) as eng:
        eng.add_complex(complex_())
        # the first allocation of the call is the list's
        begin = hip.count("allocs")
        hip.fail_alloc(0)
        fails(lambda: eng.calc_energy(0, *poses(3)), "GD_ERR_HIP")
        size = hip.allocs(begin)[0]
        assert size >= 16 * 8  # at least a unit for each of eight groups
        begin, first = hip.count("allocs"), hip.count("launches")
        eng.calc_energy(0, *poses(3))
        assert hip.allocs(begin)[0] == size
        # the units' instance: <1, 0, false, true>
        assert any("Lb0ELb1E" in k for k, _, _ in hip.launches("gd_mc_kernel", first))


def complex_table(hip):
    """The complex table on the device is replaced only when the new one is
    there: runs after a failed upload read the table they had."""
    import geaxdock_gpu_amd as gd
    with gd.Engine(seed=1, launch=gd.abi.LAUNCH_NO_GRAPH | gd.abi.LAUNCH_NO_SPREAD) as eng:
        eng.add_complex(complex_())
        eng.run(4, 2)
        begin = hip.count("allocs")
        eng.sur_build_grids(1.0, 4.0)
        n = hip.count("allocs") - begin  # the table's is the last
        hip.fail_alloc(n - 2)  # the grid keeps its memory this time
        fails(lambda: eng.sur_build_grids(1.0, 4.0), "GD_ERR_HIP")
        first = hip.count("launches")
        eng.run(4, 2)
        runs = hip.launches("gd_mc_kernel", first)
        assert runs and all(table for _, _, table in runs)


def feature_grids(hip):
    """Grids that found no memory, or never reached the complex table, are no
    grids: the calls that read them refuse until they are built again."""
    import geaxdock_gpu_amd as gd
    target = np.zeros(3, np.float32)
    for failing in range(4):  # grid 0, grid 1, the table; then none
        with gd.Engine(seed=1) as eng:
            for seed in (1, 2):
                eng.add_complex(complex_(seed))
            eng.sur_set_params(np.zeros(eng.sur_num_params, np.float32))
            eng.sur_build_grids(1.0, 4.0)
            eng.sur_tabulate()
            first = hip.count("launches")
            if failing < 3:
                hip.fail_alloc(failing)
                fails(lambda: eng.sur_build_grids(1.0, 5.0), "GD_ERR_HIP")
                uses = [lambda c=c: eng.sur_features(c, *poses(3)) for c in (0, 1)]
                uses += [lambda c=c: eng.sur_dataset_add(c, *poses(3), target) for c in (0, 1)]
                uses += [lambda: eng.sur_dataset_add_multi(np.zeros(3, np.int32), *poses(3), target),
                         lambda: eng.sur_surrogate(0, *poses(3), 1.0), eng.sur_tabulate,
                         lambda: eng.run_da(4, 0, 2, 1.0)]
                for use in uses:
                    fails(use, "GD_ERR_STATE")
                assert not hip.launches("gd_sur_feat", first) and not hip.launches("gd_mc", first)
                eng.calc_energy(0, *poses(3))  # needs no grids
                eng.sur_build_grids(1.0, 5.0)
            for c in (0, 1):
                eng.sur_features(c, *poses(3))
            eng.sur_tabulate()
            eng.run_da(4, 0, 2, 1.0)


def refused_complex(hip):
    """A complex that could not be added is not in the context: the next one
    takes its id, and kernels get no record without arrays."""
    import geaxdock_gpu_amd as gd
    # no memory for the device block, for the staging; tiles beyond LDS
    for kw, failing, status in [({}, 0, "GD_ERR_HIP"), ({}, 1, "GD_ERR_HIP"),
                                (dict(receptor_tile=4000), -1, "GD_ERR_CAPACITY")]:
        with gd.Engine(seed=1, **kw) as eng:
            live = hip.count("live")
            hip.fail_alloc(failing)
            fails(lambda: eng.add_complex(complex_()), status)
            assert eng.num_replicas(0) == -1
            assert hip.count("live") <= live + 1  # at most the staging stays
            if kw:
                continue
            assert eng.add_complex(complex_()) == 0
            first = hip.count("launches")
            eng.calc_energy(0, *poses(3))
            assert hip.launches("gd_ref_kernel", first)[0][1] == [20, 1, 1]  # one complex


def training_buffers(hip):
    """Work buffers that could not grow are gone, not in use after their end:
    every buffer is given back once (host_hip.cpp aborts on a second time)."""
    import geaxdock_gpu_amd as gd
    for failing in range(5):  # rows' gradients, then the four gradient partials
        with gd.Engine(seed=1) as eng:
            eng.add_complex(complex_())
            eng.sur_set_params(np.zeros(eng.sur_num_params, np.float32))
            eng.sur_build_grids(1.0, 4.0)
            eng.sur_dataset_add(0, *poses(40), np.zeros(40, np.float32))
            eng.sur_loss_grad(0, 2)
            hip.fail_alloc(failing)
            fails(lambda: eng.sur_loss_grad(0, 40), "GD_ERR_HIP")
            begin = hip.count("allocs")
            eng.sur_loss_grad(0, 2)
            assert hip.count("allocs") - begin == 5
            eng.sur_loss_grad(0, 40)


def parameter_buffers(hip):
    """Parameters whose buffers were not all allocated get the missing ones in
    the next call; before, it wrote the weights' layouts to null pointers."""
    import geaxdock_gpu_amd as gd
    for failing in range(7):
        with gd.Engine(seed=1) as eng:
            p = np.zeros(eng.sur_num_params, np.float32)
            live = hip.count("live")
            hip.fail_alloc(failing)
            fails(lambda: eng.sur_set_params(p), "GD_ERR_HIP")
            eng.sur_set_params(p)
            assert hip.count("live") == live + 7


def record_rings(hip):
    """After a window whose record rings do not fit, runs of windows that do fit
    go on, with one ring (no sink) or two."""
    import geaxdock_gpu_amd as gd
    record, n_rep = 92, 8
    fit = record * n_rep * 101  # a window of 100 steps
    for sink in (None, lambda c, r: None):
        for launch in (0, gd.abi.LAUNCH_NO_SPREAD):
            with gd.Engine(seed=1, launch=launch, steps_per_dump=1 << 20) as eng:
                eng.add_complex(complex_())
                assert eng.num_replicas(0) == n_rep
                eng.run(10, 0, sink)
                hip.fail_above(fit)
                fails(lambda: eng.run(1 << 20, 0, sink), "GD_ERR_HIP")
                eng.run(100, 0, sink)
                eng.run(10, 0, sink)
                hip.fail_above(0)
                eng.run(200, 0, sink)


def window_steps(hip):
    """A window of several launches that ends in an error has taken the steps
    of the launches before it: its random numbers are not used again."""
    import geaxdock_gpu_amd as gd
    with gd.Engine(seed=1, launch=gd.abi.LAUNCH_SPREAD) as eng:
        eng.add_complex(complex_())  # eight packs: trees of five steps
        eng.run(0, 10)
        step = 0
        # launches of a run: the counts, two trees, an exchange, two trees, an exchange
        for failing, taken in ((1, 0), (2, 5), (3, 10), (4, 10), (5, 15), (6, 20)):
            hip.fail_launch(failing)
            fails(lambda: eng.run(20, 10), "GD_ERR_HIP")
            step += taken
            assert struct.unpack_from("<8I", eng.checkpoint())[4] == step, failing
            rest = -step % 10
            if rest:
                eng.run(rest, 10)
                step += rest


def pose_calls_without_allocations(hip):
    """gd_calc_energy_noalloc allocates and creates nothing, whatever its
    launches, after a gd_calc_energy of one pose or a gd_run."""
    import geaxdock_gpu_amd as gd
    for prepare in (lambda e: e.calc_energy(0, *poses(1)), lambda e: e.run(0)):
        with gd.Engine(seed=1, ladders_per_pack=2) as eng:
            eng.add_complex(complex_(n_lig=3, n_tmp=8))  # conformers of splits of 4 and 8
            prepare(eng)
            for n in (1, 5, 340):  # the last pack of a split may be small
                made, allocs = hip.count("made"), hip.count("allocs")
                first = hip.count("launches")
                eng.calc_energy_noalloc(0, *poses(n, 3))
                assert n == 1 or len(hip.launches("gd_mc_kernel", first)) > 1
                assert (hip.count("made"), hip.count("allocs")) == (made, allocs), n


def many_conformers(hip):
    """Feature grids of more receptor conformers than a launch has rows for."""
    import geaxdock_gpu_amd as gd
    n_prt = 70000
    with gd.Engine(seed=1) as eng:
        eng.add_complex(complex_(pnp=2, n_lig=1, n_prt=n_prt, n_tmp=1))
        first = hip.count("launches")
        eng.sur_build_grids(1.0, 1.01)
        assert sum(g[1] for _, g, _ in hip.launches("gd_sur_grid", first)) == n_prt


def window_drains(hip):
    """Records of a window go to the sink beside the next window by copy engines
    alone: they are compacted before it starts, since a kernel beside it would
    wait for registers until its end."""
    import geaxdock_gpu_amd as gd
    launch = gd.abi.LAUNCH_NO_GRAPH | gd.abi.LAUNCH_NO_SPREAD
    with gd.Engine(seed=1, launch=launch, steps_per_dump=10) as eng:
        eng.add_complex(complex_())
        eng.run(0)
        hip.lib.host_hip_fill(C.c_int(1))  # a cleared count is 1: a record for each replica
        first, got = hip.count("launches"), []
        eng.run(30, 0, sink=lambda c, r: got.append((hip.count("launches"), len(r))))
        hip.lib.host_hip_fill(C.c_int(0))
        kernels = [("C" if "compact" in k else "M") for k, _, _ in hip.launches("", first)
                   if "compact" in k or "gd_mc_kernel" in k]
        assert kernels == list("MCMCMC")
        # the first two windows' records arrive with the next window's launch made
        assert [n for _, n in got] == [eng.num_replicas(0)] * 3
        made = [i for i in range(first, hip.count("launches"))
                if "gd_mc_kernel" in hip.lib.host_hip_kernel(C.c_long(i)).decode()]
        assert got[0][0] > made[1] and got[1][0] > made[2]


CASES = [unit_lists, complex_table, feature_grids, refused_complex, training_buffers,
         parameter_buffers, record_rings, window_steps,
         pose_calls_without_allocations, many_conformers, window_drains]


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host_hip") / "libhost_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(HERE, "cpp", "host_hip.cpp"), "-o", so],
                   check=True)
    return so


@pytest.mark.parametrize("case", [c.__name__ for c in CASES])
def test_host_failures(runtime, case):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), runtime, case], cwd=ROOT,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    {c.__name__: c for c in CASES}[sys.argv[2]](HostHip(sys.argv[1]))
