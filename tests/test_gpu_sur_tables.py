"""Feature grids and network tables at the edges of their kernels' tiles,
against the FP64 oracle: grids whose side is not a multiple of the 4-node
bricks, node counts that are not a multiple of the 16-point tiles, receptors
around the 64 points a wave tests at a time, several conformers, and a second
build with another spacing on the same context. Bounds as in
test_gpu_surrogate.py (features) and test_gpu_da.py (totals).
"""
import numpy as np
import pytest

from geaxdock_gpu_amd import surrogate as sg
from geaxdock_gpu_amd import synth
from oracle import gdo
from oracle import surrogate as so

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pnp", [1, 63, 65, 200])
@pytest.mark.parametrize("grids", [((1.0, 2.0), (1.0, 3.5)), ((0.9, 7.0), (1.5, 7.0)),
                                   ((1.0, 3.5), (1.0, 3.5))])
def test_grids_and_tables_match_fp64(grids, pnp):
    import geaxdock_gpu_amd as gd
    cx = synth.make_complex(30 + pnp, lna=11, pnp=pnp, pnk=20, pos=2, mcs_atoms=4, n_lig=2,
                            n_prt=3, n_tmp=1, void_radius=2.0, box=14.0)
    p = so.init_params(5)
    rng = np.random.default_rng(pnp)
    n_pose, scale = 7, 3.0
    mm = np.zeros((n_pose, 6), np.float32)
    mm[:, :3] = rng.normal(0, 1.0, (n_pose, 3))
    mm[:, 3:] = rng.uniform(-np.pi, np.pi, (n_pose, 3))
    il, ip = rng.integers(0, 2, n_pose), np.arange(n_pose) % 3
    with gd.Engine(seed=1) as eng:
        cid = eng.add_complex(cx)
        eng.sur_set_params(sg.pack_params(p))
        for spacing, half in grids:
            eng.sur_build_grids(spacing, half)
            eng.sur_tabulate()
        feat = eng.sur_features(cid, il, ip, mm)
        got = eng.sur_surrogate(cid, il, ip, mm, scale)
    n = int(np.ceil(2 * half / spacing)) + 1
    origin = np.float64(cx.pocket_center) - half
    prt = np.stack([cx.prt_x, cx.prt_y, cx.prt_z], 1).reshape(3, cx.pnp, 3)
    grid = [so.grid_features(origin, spacing, n, prt[c], cx.prt_t) for c in range(3)]
    tabs = [so.tabulate(p, g, np.unique(cx.lig_t)) for g in grid]
    d = cx.desc()
    ref = gdo.refmap_f64(d, cx)
    w = np.asarray(cx.enepara_struct.w, np.float64)
    for i in range(n_pose):
        xyz = gdo.place_f64(d, cx, int(il[i]), mm[i]).T
        want = so.features(cx.lig_t, so.interp(grid[ip[i]], origin, spacing, xyz))
        assert np.all(np.abs(feat[i] - want) <= 1e-3 + 1e-3 * np.abs(want))
        y = np.array([so.interp(tabs[ip[i]][int(t)][..., None], origin, spacing,
                                xyz[k:k + 1])[0, 0] for k, t in enumerate(cx.lig_t)])
        o = gdo.energy_f64(d, ref, int(ip[i]), int(il[i]), mm[i])
        cheap = sum(w[j] * o.e[j] for j in (6, 7, 8))
        total = scale * y.sum() / cx.lna + cheap
        tol = 2e-2 * scale * np.abs(y).sum() / cx.lna + 1e-4 * (1 + abs(cheap))
        assert abs(got[i] - total) <= tol, (i, got[i], total, tol)
