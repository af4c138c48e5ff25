"""Terms skipped by distance in the chunk pair loop leave every bit as it is.

Where all lanes of a wave are far from a receptor point, the loop goes without
the PMF's exponential, HPC, contacts and H-bond terms. A complex with a value
that is not finite takes no such skip: here the hydrophobicity of a point that
is not flagged hydrophobic, which no energy uses. Both must give the same bits,
for 1 to 4 atoms per lane, receptors in LDS and in tiles, and poses from inside
the receptor to beyond the range where a distance's ninth power overflows.
"""
import numpy as np
import pytest

from geaxdock_gpu_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gd():
    import geaxdock_gpu_amd as g
    return g


def _poses(n):
    rng = np.random.default_rng(n)
    mm = np.zeros((n, 6), np.float32)
    mm[:, :3] = rng.normal(0.0, 1.0, (n, 3))
    mm[:, 3:] = rng.uniform(-np.pi, np.pi, (n, 3))
    # from near to far: 8 to 30 A out of the pocket, then 100 A to 1e7 A
    out = rng.normal(0.0, 1.0, (n, 3))
    out /= np.linalg.norm(out, axis=1, keepdims=True)
    far = np.concatenate([np.zeros(n // 4), np.linspace(8.0, 30.0, n // 2),
                          np.logspace(2.0, 7.0, n - n // 4 - n // 2)])
    mm[:, :3] += (far[:, None] * out).astype(np.float32)
    return mm


@pytest.mark.parametrize("pnp,void,tile", [(1, 3.0, 0), (130, 2.0, 0), (2501, 10.0, 0),
                                           (2501, 4.0, 100), (6001, 10.0, 0)])
@pytest.mark.parametrize("lpr,apl,lna", [(64, 1, 61), (32, 1, 30), (16, 2, 29), (16, 3, 48),
                                         (16, 4, 62)])
def test_skips_keep_the_bits(gd, lpr, apl, lna, pnp, void, tile):
    n = 64
    mm = _poses(n)
    out = []
    for plain in (True, False):
        cx = synth.make_complex(40 + lna, lna=lna, pnp=pnp, pnk=30, pos=2, n_lig=2, n_prt=1,
                                n_tmp=4, void_radius=void)
        if plain:
            unused = np.flatnonzero(cx.prt_c0_and_d12_or_c2 == 0)
            if len(unused) == 0:
                pytest.skip("every point is hydrophobic")
            cx.prt_hpp[unused[0]] = np.nan
        with gd.Engine(seed=3, lanes_per_replica=lpr, atoms_per_lane=apl, receptor_split=1,
                       launch=abi.LAUNCH_NO_SPREAD, receptor_tile=tile) as e:
            e.add_complex(cx)
            got = [e.calc_energy(0, np.arange(n, dtype=np.int32) % 2, np.zeros(n, np.int32),
                                 mm).tobytes()]
            e.run(20, 10)
            st = e.state(0)
            out.append(got + [st[k].tobytes() for k in sorted(st)])
    assert out[0] == out[1]
