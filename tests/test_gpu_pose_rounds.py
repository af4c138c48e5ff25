"""Pose evaluation in rounds (several rounds of poses on one staged receptor,
spread packing) gives each pose the bits it has alone, whatever the number of
poses: below, at and above the sizes where a workgroup takes a second round,
with a last round that is partly empty."""
import numpy as np
import pytest

from geaxdock_gpu_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lna,n", [(20, 2047), (20, 4099), (20, 9001), (40, 1025), (40, 5003)])
def test_rounds_keep_bits(lna, n):
    import geaxdock_gpu_amd as gd
    cx = synth.make_complex(3, lna=lna, pnp=150, pnk=30, pos=3, mcs_atoms=5, n_lig=3, n_prt=2,
                            n_tmp=2, void_radius=5.0)
    rng = np.random.default_rng(n)
    mm = np.zeros((n, 6), np.float32)
    mm[:, :3] = rng.normal(0.0, 1.5, (n, 3))
    mm[:, 3:] = rng.uniform(-np.pi, np.pi, (n, 3))
    il, ip = rng.integers(0, 3, n).astype(np.int32), rng.integers(0, 2, n).astype(np.int32)
    with gd.Engine(seed=1) as eng:
        cid = eng.add_complex(cx)
        e = eng.calc_energy(cid, il, ip, mm)
        some = rng.choice(n, 300, replace=False)
        parts = np.concatenate([eng.calc_energy(cid, il[s], ip[s], mm[s])
                                for s in np.array_split(some, 7)])
    assert parts.tobytes() == e[some].tobytes()
