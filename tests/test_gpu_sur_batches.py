"""Training batches at the edges of their kernels' tiles, against FP64: the pose
kernel takes 64 poses and 4,096 rows at a time, the batch kernels 64 rows, and
batches may start anywhere in the dataset. Ligands of 100 and 9 atoms give
batches whose 64 poses pass 4,096 rows and whose rows end inside a step.

Predictions are compared in FP64 from the engine's own features: BF16 operands
bound a row's error by 2e-2 of the row outputs' magnitude. Gradients as in
test_gpu_surrogate.py. A training step with the learning rate lr must move
the parameters by Adam's first step of the same gradient.
"""
import numpy as np
import pytest

from geaxdock_gpu_amd import surrogate as sg
from geaxdock_gpu_amd import synth
from oracle import surrogate as so

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup():
    import geaxdock_gpu_amd as gd
    cxs = [synth.make_complex(60 + k, lna=lna, pnp=300, pnk=20, pos=2, mcs_atoms=4, n_lig=1,
                              n_prt=1, n_tmp=1, void_radius=3.0) for k, lna in enumerate((100, 9))]
    rng = np.random.default_rng(2)
    n = 400
    cid = (rng.random(n) < 0.2).astype(np.int32)  # mostly the large ligand
    mm = np.zeros((n, 6), np.float32)
    mm[:, :3] = rng.normal(0, 1.0, (n, 3))
    mm[:, 3:] = rng.uniform(-np.pi, np.pi, (n, 3))
    t = rng.normal(0, 2, n).astype(np.float32)
    zero = np.zeros(n, np.int32)
    p = so.init_params(9)
    eng = gd.Engine(seed=1)
    for cx in cxs:
        eng.add_complex(cx)
    eng.sur_build_grids(0.8, 9.6)
    eng.sur_dataset_add_multi(cid, zero, zero, mm, t)
    F, pose = [], []
    for i in range(n):
        f = eng.sur_features(int(cid[i]), zero[:1], zero[:1], mm[i:i + 1])[0]
        F.append(f.astype(np.float64))
        pose += [i] * len(f)
    yield eng, p, np.concatenate(F), np.array(pose), t.astype(np.float64)
    eng.close()


@pytest.mark.parametrize("b,e", [(0, 1), (0, 63), (3, 67), (5, 70), (0, 130), (17, 400)])
def test_batches_match_fp64(setup, b, e):
    eng, p, F, pose, t = setup
    eng.sur_set_params(sg.pack_params(p))
    rows = (pose >= b) & (pose < e)
    y = so.rows(p, F[rows])
    S, mag = np.zeros(e - b), np.zeros(e - b)
    np.add.at(S, pose[rows] - b, y)
    np.add.at(mag, pose[rows] - b, np.abs(y))
    pred = eng.sur_predict(b, e)
    assert np.all(np.abs(pred - S) <= 2e-2 * mag + 1e-5)
    loss, g = eng.sur_loss_grad(b, e)
    lo, go = so.loss_and_grads(p, F[rows], pose[rows] - b, t[b:e])
    assert abs(loss - lo) <= 2e-2 * lo
    gg = sg.unpack_params(g)
    for k in go:
        a, w = np.asarray(gg[k], np.float64).reshape(-1), np.asarray(go[k]).reshape(-1)
        assert np.linalg.norm(a - w) <= 3e-2 * np.linalg.norm(w), k
    # one batch, one epoch: Adam's first step is lr * sign(g) up to its epsilon
    lr = 1e-3
    hist, _ = eng.sur_train(b, e, 1, e - b, lr)
    step = (sg.pack_params(p) - eng.sur_get_params()).astype(np.float64)
    want = lr * g / (np.abs(g) + 1e-8)
    assert np.all(np.abs(step - want) <= 1e-4 * lr + 1e-6)
    assert hist[0] == pytest.approx(np.mean((eng.sur_predict(b, e).astype(np.float64) - t[b:e]) ** 2),
                                    rel=1e-5)
