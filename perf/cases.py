"""The work that users of the docking engine have it do, as timed cases.

Each case is one pass through the public entry points (`geaxdock_gpu_amd.Engine`
and `geaxdock_gpu_amd.run`) on seeded synthetic complexes of the sizes that the
benchmark, the tests and the sample inputs of this repository have. `exact`
gives what a pass computes in 64 bits with plain torch, without the engine.
"""
import math

import numpy as np
import torch

import geaxdock_gpu_amd as gd
from geaxdock_gpu_amd import abi, surrogate, synth

SPACING, HALF_WIDTH = 0.5, 16.0  # surrogate grids: the engine's defaults
EXACT_PAIRS = 2.5e10             # ligand-receptor pairs that `exact` gets through in about 20 s

_SHAPE = dict(lna=32, lna_max=0, pnp=1200, pnp_max=0, pnk=100, pos=4, n_lig=1, n_prt=1, n_tmp=8)


def _case(kind, **kw):
    return {"kind": kind, **_SHAPE, **kw}


def listed():
    uneven = dict(lna=12, lna_max=64, pnp=800, pnp_max=4000, n_lig=5, n_prt=3)
    coarse = dict(lna=44, pnp=672, pnk=4408, pos=196, move="uniform")
    return [
        # A few poses of one complex, as a rescoring loop or a viewer asks for
        # them: the smallest call.
        _case("score", name="score_8", poses=8),
        # Rescoring of a whole set of poses over all conformers, as the
        # surrogate's training labels and the analysis of a trajectory do.
        _case("score", name="score_16k", poses=16384, lna=38, pnp=2400, n_lig=5, n_prt=3),
        # A receptor that does not fit in LDS, with large KDE and MCS sets.
        _case("score", name="score_large_receptor", poses=2000, lna=61, pnp=8000, pnk=4000,
              pos=40, n_lig=7, n_prt=2),
        # One complex with one temperature ladder: the smallest Monte Carlo
        # run; its accepted states go to a sink.
        _case("mc", name="run_single", complexes=1, steps=200, record=True),
        # The reference's Run() as one call: context, upload, run, records.
        _case("call", name="run_call", lna=31, pnp=350, pnk=454, pos=11, n_lig=21, n_prt=3,
              steps=200, move="uniform"),
        # A crystal ligand with its coarse receptor, 51 ladders, thousands of
        # KDE points and hundreds of MCS templates.
        _case("mc", name="run_coarse", complexes=1, steps=100, record=True, n_lig=17, n_prt=3,
              **coarse),
        # An ensemble: one ligand and receptor in many conformers, 3,520
        # replicas.
        _case("mc", name="run_ensemble", complexes=1, steps=40, record=True, lna=48, pnp=3000,
              pnk=200, pos=8, n_lig=20, n_prt=11, n_tmp=16),
        # A batch of uneven complexes in one context, best poses only: virtual
        # screening, the engine's headline workload.
        _case("mc", name="run_batch", complexes=64, steps=40, record=False, **uneven),
        # The same under delayed acceptance with the tabulated network.
        _case("da", name="da_batch", complexes=16, steps=80, k_sub=4, **uneven),
        # What a delayed-acceptance run needs first: feature grids, the
        # network's tables, and a check of both on poses.
        _case("tables", name="surrogate_tables", complexes=2, poses=1000, lna=38, pnp=2400,
              n_lig=5, n_prt=3),
        # Training of the surrogate and its held-out predictions.
        _case("train", name="surrogate_train", lna=38, pnp=2400, n_prt=2, poses=32768,
              held_out=2000, batch=4096, epochs=2),
        # Clustering of a run's accepted states into medoids, per replica and
        # then over all of them.
        _case("post", name="post_200k", replicas=440, records=455, k_replica=50, k_final=500),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["score", "score", "mc", "mc", "mc", "call", "da", "tables", "train",
                       "post"])
    move = rng.choice(["gaussian", "uniform"])
    shape = dict(lna=_log(rng, 8, 120), pnp=_log(rng, 300, 6000), pnk=_log(rng, 30, 4500),
                 pos=_log(rng, 1, 200), n_lig=_log(rng, 1, 20), n_prt=_log(rng, 1, 6),
                 n_tmp=rng.choice([1, 3, 5, 8, 8, 12, 16]))
    # temperature ladders are at most one workgroup of 512 lanes
    if shape["lna"] > 64:
        shape["n_tmp"] = min(shape["n_tmp"], 8)
    if kind == "score":
        cap = 2e9 / (shape["lna"] * shape["pnp"])
        return _case(kind, poses=_log(rng, 1, max(2, min(20000, cap))), **shape)
    if kind == "mc":
        if rng.random() < 0.4:  # an uneven batch
            lo, hi = sorted((_log(rng, 8, 70), _log(rng, 8, 70)))
            p0, p1 = sorted((_log(rng, 400, 4000), _log(rng, 400, 4000)))
            return _case(kind, complexes=_log(rng, 2, 48), steps=rng.choice([20, 40, 50]),
                         record=rng.random() < 0.5, move=move, lna=lo, lna_max=hi, pnp=p0,
                         pnp_max=p1, n_lig=rng.randint(1, 5), n_prt=rng.randint(1, 3))
        rep = shape["n_lig"] * shape["n_prt"] * shape["n_tmp"]
        cap = 2e10 / (rep * shape["lna"] * (shape["pnp"] + shape["pnk"] / 10))
        return _case(kind, complexes=1, steps=max(10, min(_log(rng, 20, 200), int(cap))),
                     record=rng.random() < 0.7, move=move, **shape)
    if kind == "call":
        shape.update(lna=_log(rng, 8, 60), pnp=_log(rng, 300, 2000))
        return _case(kind, steps=_log(rng, 20, 200), move=move, **shape)
    if kind == "da":
        k = rng.choice([2, 4, 8])
        n = _log(rng, 1, 16)
        lo, hi = sorted((_log(rng, 10, 64), _log(rng, 10, 64)))
        p0, p1 = sorted((_log(rng, 600, 4000), _log(rng, 600, 4000)))
        return _case(kind, complexes=n, steps=80, k_sub=k, move=move, lna=lo, lna_max=hi, pnp=p0,
                     pnp_max=p1, pnk=rng.choice([60, 100, 700]), n_lig=rng.randint(1, 5),
                     n_prt=rng.randint(1, 3))
    if kind == "tables":
        return _case(kind, complexes=rng.randint(1, 2), poses=_log(rng, 10, 1000),
                     lna=_log(rng, 8, 64), pnp=_log(rng, 400, 4000), n_prt=rng.randint(1, 3),
                     n_lig=rng.randint(1, 5))
    if kind == "train":
        return _case(kind, lna=_log(rng, 10, 48), pnp=_log(rng, 600, 3000), n_prt=1,
                     poses=_log(rng, 500, 30000), held_out=_log(rng, 50, 3000),
                     batch=rng.choice([256, 1000, 4096]), epochs=1)
    return _case(kind, replicas=_log(rng, 4, 440), records=_log(rng, 60, 455),
                 k_replica=rng.choice([20, 50]), k_final=rng.choice([100, 500]))


# ---- what a user's program holds before the call ---------------------------

def _complexes(c, seed):
    rng = np.random.default_rng([seed, 0xCA5E])
    out = []
    for i in range(c.get("complexes", 1)):
        lna = int(rng.integers(c["lna"], c["lna_max"] + 1)) if c["lna_max"] else c["lna"]
        pnp = int(rng.integers(c["pnp"], c["pnp_max"] + 1)) if c["pnp_max"] else c["pnp"]
        uniform = c.get("move") == "uniform"
        out.append(synth.make_complex(
            seed * 1009 + i, lna=lna, pnp=pnp, pnk=c["pnk"], pos=c["pos"],
            mcs_atoms=max(1, (5 * lna) // 8), n_lig=c["n_lig"], n_prt=c["n_prt"],
            n_tmp=c["n_tmp"], enepara_seed=seed,
            move_kind=abi.MOVE_UNIFORM if uniform else abi.MOVE_GAUSSIAN,
            trans_sigma=0.1 if uniform else 0.2))
    return out


def _poses(c, n, seed):
    """Poses around the start pose, as a Monte Carlo run visits them."""
    rng = np.random.default_rng([seed, 0x905E])
    mm = np.empty((n, 6), np.float32)
    mm[:, :3] = rng.normal(0.0, 0.8, (n, 3))
    mm[:, 3:] = rng.normal(0.0, 0.4, (n, 3))
    return (rng.integers(0, c["n_lig"], n).astype(np.int32),
            rng.integers(0, c["n_prt"], n).astype(np.int32), mm)


def _network(seed):
    rng = np.random.default_rng([seed, 0x4E7])
    p = surrogate.init_params(seed)
    p["b1"] = rng.normal(0.0, 0.1, surrogate.N_HID)
    p["b2"] = rng.normal(0.0, 0.1, surrogate.N_HID)
    return p


def _targets(mm, seed):
    """Standardized energies with a repulsive tail clipped like training sets."""
    rng = np.random.default_rng([seed, 0x7A6])
    t = np.cos(mm.astype(np.float64) @ rng.normal(0.0, 1.0, 6)) + 0.5 * (mm[:, :3] ** 2).sum(1)
    t = t + 0.3 * rng.standard_normal(len(mm))
    t = (t - t.mean()) / t.std()
    return np.minimum(t, np.percentile(t, 99.5)).astype(np.float32)


def _post_records(c, seed):
    """Accepted states of replicas: each replica's energies wander around its
    own level; replicas have different numbers of them."""
    rng = np.random.default_rng([seed, 0x9057])
    n_rec = rng.integers(c["records"] // 4, 2 * c["records"] - c["records"] // 4, c["replicas"])
    rep = np.repeat(np.arange(c["replicas"]), n_rec)
    n = len(rep)
    walk = np.cumsum(rng.normal(0.0, 0.15, (n, 9)), axis=0)
    first = np.concatenate([[0], np.cumsum(n_rec)[:-1]])
    walk -= np.repeat(walk[first], n_rec, axis=0)
    r = np.zeros(n, abi.RECORD_DTYPE)
    r["replica"][:, 0] = rep
    r["energy"]["e"][:, :9] = (np.tanh(walk) * 2.0 + rng.normal(0.0, 1.5, (c["replicas"], 9))[rep]
                               + rng.normal(0.0, 0.05, (n, 9)))
    r["step"] = np.arange(n) - np.repeat(first, n_rec)
    return r


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "post":
        return dict(case=c, seed=seed, eng=gd.Engine(seed=seed), recs=_post_records(c, seed))
    cxs = _complexes(c, seed)
    # a buffer for every state that a run can accept, filled by its sink
    room = sum(cx.n_rep for cx in cxs) * (c.get("steps", 0) + 1)
    if kind == "call":
        return dict(case=c, seed=seed, cx=cxs[0], recs=np.zeros(room, abi.RECORD_DTYPE))
    eng = gd.Engine(seed=seed, record=bool(c.get("record", False)))
    for cx in cxs:
        eng.add_complex(cx)
    s = dict(case=c, seed=seed, eng=eng)
    if c.get("record"):
        s["recs"] = np.zeros(room, abi.RECORD_DTYPE)
    if kind in ("score", "tables"):
        s["poses"] = [_poses(c, c["poses"], seed + 7 * i) for i in range(len(cxs))]
    if kind == "score":
        eng.calc_energy(0, *(a[:1] for a in s["poses"][0]))  # the contact map, once per complex
    if kind in ("da", "tables", "train"):
        eng.sur_set_params(surrogate.pack_params(_network(seed)))
    if kind in ("da", "train"):
        eng.sur_build_grids(SPACING, HALF_WIDTH)
    if kind == "da":
        eng.sur_tabulate()
    if kind == "train":
        il, ip, mm = _poses(c, c["poses"] + c["held_out"], seed)
        eng.sur_dataset_reserve(len(mm) * c["lna"] + 64)
        eng.sur_dataset_add(0, il, ip, mm, _targets(mm, seed))
        s["params"] = surrogate.pack_params(_network(seed))
    return s


# ---- one pass ---------------------------------------------------------------

def _state(eng):
    st = [eng.state(i) for i in range(len(eng.complexes))]
    cat = lambda k: np.concatenate([x[k] for x in st])  # noqa: E731
    e = cat("energy")
    return dict(movematrix=cat("movematrix"), e=e["e"], cms=e["cms"], rmsd=e["rmsd"],
                replica=cat("replica"), acs_mc=cat("acs_mc"), acs_x=cat("acs_x"))


class _Sink:
    """Collects a run's records in the caller's buffer."""

    def __init__(self, buf):
        self.buf, self.n = buf, 0

    def __call__(self, cid, recs):
        self.buf[self.n:self.n + len(recs)] = recs
        self.n += len(recs)

    def fields(self):
        r = self.buf
        r[self.n:] = 0
        return dict(e=r["energy"]["e"], rmsd=r["energy"]["rmsd"], movematrix=r["movematrix"],
                    replica=r["replica"], step=r["step"])


def run(s):
    c, kind = s["case"], s["case"]["kind"]
    if kind == "call":
        recs, _ = gd.run(s["cx"], c["steps"], 20, seed=s["seed"])
        sink = _Sink(s["recs"])
        for k in sorted(recs):
            sink(0, recs[k])
        return dict(records=sink.fields())
    eng = s["eng"]
    if kind == "score":
        e = eng.calc_energy(0, *s["poses"][0])
        return dict(e=e["e"], cms=e["cms"], rmsd=e["rmsd"])
    if kind == "mc":
        sink = _Sink(s["recs"]) if c["record"] else None
        eng.run(c["steps"], 20, sink=sink)
        out = _state(eng)
        if c["record"]:
            out["records"] = sink.fields()
        else:
            best = [eng.best(i) for i in range(len(eng.complexes))]
            out["best_e"] = np.concatenate([b[0] for b in best])
            out["best_movematrix"] = np.concatenate([b[1] for b in best])
        return out
    if kind == "da":
        eng.run_da(c["steps"], 5 * c["k_sub"], c["k_sub"], 0.5)
        return _state(eng)
    if kind == "tables":
        eng.sur_build_grids(SPACING, HALF_WIDTH)
        eng.sur_tabulate()
        return [dict(features=eng.sur_features(i, *p), total=eng.sur_surrogate(i, *p, 0.5))
                for i, p in enumerate(s["poses"])]
    if kind == "train":
        n = c["poses"]
        eng.sur_set_params(s["params"])
        hist, _ = eng.sur_train(0, n, c["epochs"], c["batch"], 1e-3)
        return dict(loss=hist, params=eng.sur_get_params(),
                    held_out=eng.sur_predict(n, n + c["held_out"]))
    idx, sizes = eng.post_mc(s["recs"], c["k_replica"], c["k_final"], seed=s["seed"])
    return dict(medoid=idx, size=sizes)


# ---- what a pass cannot do without -------------------------------------------

def _mean(c, key):
    return (c[key] + c[key + "_max"]) / 2 if c[key + "_max"] else c[key]


def work(case):
    """36 flops per ligand-receptor pair of an exact evaluation, 2 per network
    weight and row; inputs and outputs once."""
    c, kind = case, case["kind"]
    net = 2.0 * (57 * 128 + 129 * 128 + 128)
    if kind == "post":
        n = c["replicas"] * c["records"]
        n1 = min(n, c["replicas"] * c["k_replica"])
        # one assignment per level; each takes several
        return dict(bytes=40.0 * n + 12.0 * c["k_final"],
                    flops=27.0 * (n * c["k_replica"] + n1 * c["k_final"]))
    lna, pnp, n_cx = _mean(c, "lna"), _mean(c, "pnp"), c.get("complexes", 1)
    inputs = n_cx * (12.0 * lna * c["n_lig"] + 12.0 * pnp * c["n_prt"] + 16.0 * c["pnk"] +
                     12.0 * lna * c["pos"] + 35000.0)
    nodes = (2 * HALF_WIDTH / SPACING + 1) ** 3
    near = min(pnp, 113.0)  # receptor points within 8 A of a node
    if kind == "score":
        return dict(bytes=inputs + 80.0 * c["poses"], flops=36.0 * c["poses"] * lna * pnp)
    if kind in ("mc", "call", "da"):
        n_rep = n_cx * c["n_lig"] * c["n_prt"] * c["n_tmp"]
        evals = n_rep * c["steps"] // c.get("k_sub", 1)
        recs = 92.0 * n_rep * c["steps"] if kind == "call" or c.get("record") else 0.0
        return dict(bytes=inputs + 120.0 * n_rep + recs, flops=36.0 * evals * lna * pnp)
    if kind == "tables":
        types = 24 * (1 - (23 / 24) ** lna)
        sets = n_cx * c["n_prt"] * nodes
        return dict(bytes=inputs + sets * 4.0 * (32 + types) + n_cx * c["poses"] * lna * 224.0,
                    flops=sets * (near * 80.0 + types * net))
    rows = lna * (c["poses"] * (3 * c["epochs"] + 1) + c["held_out"])
    return dict(bytes=128.0 * lna * (c["poses"] * c["epochs"] + c["held_out"]) + 8e5,
                flops=rows * net)


# ---- the same in 64 bits ------------------------------------------------------

class _Model:
    """Energy of poses of one complex in float64: soft Lennard-Jones,
    electrostatics, contact PMF, pocket-specific potential, hydrogen bonds,
    hydrophobic restraint, KDE, MCS restraints, pocket distance."""

    def __init__(self, cx):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        f = lambda a, *s: torch.tensor(np.asarray(a, np.float64), device=self.dev).reshape(*s)  # noqa: E731
        self.cx, self.ep = cx, cx.enepara_struct
        lt, pt = np.asarray(cx.lig_t), np.asarray(cx.prt_t)
        self.lig = torch.stack([f(a, cx.n_lig, cx.lna) for a in (cx.lig_x, cx.lig_y, cx.lig_z)], -1)
        self.prt = torch.stack([f(a, cx.n_prt, cx.pnp) for a in (cx.prt_x, cx.prt_y, cx.prt_z)], -1)
        self.center = f(cx.pocket_center, 3)
        tab = lambda name: f(np.ctypeslib.as_array(getattr(self.ep, name))[lt][:, pt], cx.lna, cx.pnp)  # noqa: E731
        self.p1a, self.p2a, self.pmf0, self.pmf1 = (tab(k) for k in ("p1a", "p2a", "pmf0", "pmf1"))
        h0, self.h1 = tab("hdb0"), tab("hdb1")
        self.h0, self.hb = h0, (h0 > 0.1) * self.h1 * (-1.0 / math.sqrt(2.0 * math.pi))
        self.q, self.ele = f(cx.lig_c, cx.lna, 1), f(cx.prt_ele, 1, cx.pnp)
        flag = np.asarray(cx.prt_c0_and_d12_or_c2) == 1
        self.hpp = f(np.where(flag, cx.prt_hpp, 0.0), cx.pnp)
        two = np.asarray(cx.prt_c) == 2
        psp = np.asarray(cx.psp, np.float64).reshape(-1, cx.n_res)
        self.psp = f(np.where(two[None], psp[lt][:, np.asarray(cx.prt_seq3r)], 0.0), cx.lna, cx.pnp)
        self.hpl = [f(np.ctypeslib.as_array(getattr(self.ep, k))[lt], cx.lna) for k in ("hpl0", "hpl1", "hpl2")]
        self.kde = torch.stack([f(a, -1) for a in (cx.kde_x, cx.kde_y, cx.kde_z)], -1)
        same = lt[:, None] == np.asarray(cx.kde_t)[None]
        self.kde_w = f(same / np.maximum(same.sum(1, keepdims=True), 1), cx.lna, cx.pnk)
        mcs = np.stack([np.asarray(a).reshape(cx.pos, cx.n_mcs)[:, np.asarray(cx.lig_n) + 1]
                        for a in (cx.mcs_x, cx.mcs_y, cx.mcs_z)], -1)
        ok = mcs[..., 0] != np.float32(abi.MCS_INVALID_COORD)
        self.mcs, self.mcs_ok = f(np.where(ok[..., None], mcs, 0.0), cx.pos, cx.lna, 3), f(ok, cx.pos, cx.lna)
        self.tcc = f(cx.mcs_tcc, cx.pos)
        self.ref = None
        zero = torch.zeros(1, 6, dtype=torch.float64, device=self.dev)
        d = torch.cdist(self.place(zero[:, :1].long()[:, 0], zero), self.prt[:1])[0]
        self.ref = d <= self.pmf0

    def place(self, il, mm):
        s, c = torch.sin(mm[:, 3:]), torch.cos(mm[:, 3:])
        (s1, s2, s3), (c1, c2, c3) = s.T, c.T
        R = torch.stack([c1 * c2, c1 * s2 * s3 - c3 * s1, s1 * s3 + c1 * c3 * s2,
                         c2 * s1, c1 * c3 + s1 * s2 * s3, c3 * s1 * s2 - c1 * s3,
                         -s2, c2 * s3, c2 * c3], -1).reshape(-1, 3, 3)
        o = self.lig[il]
        x = (o[:, :, None, :] * R[:, None, :, :]).sum(-1)
        return x + (mm[:, :3] + self.center)[:, None, :]

    def cheap(self, x, mm):
        """KDE, MCS and pocket distance before normalization."""
        cx, ep = self.cx, self.ep
        n = len(x)
        kde = torch.zeros(n, dtype=torch.float64, device=self.dev)
        step = max(1, int(2e7 // max(1, cx.lna * cx.pnk)))
        for b in range(0, n, step):
            d2 = ((x[b:b + step, :, None, :] - self.kde) ** 2).sum(-1)
            kde[b:b + step] = (torch.exp(ep.kde2 * d2) * self.kde_w).sum((1, 2))
        lhm = torch.zeros(n, dtype=torch.float64, device=self.dev)
        step = max(1, int(1e7 // max(1, cx.lna * cx.pos)))
        cnt = self.mcs_ok.sum(1)
        for b in range(0, n, step):
            d2 = ((x[b:b + step, None] - self.mcs) ** 2).sum(-1) * self.mcs_ok
            lhm[b:b + step] = (self.tcc * torch.sqrt(d2.sum(-1) / cnt.clamp(min=1))).sum(-1)
        lhm = torch.log(lhm / cx.pos) if cx.pos else lhm
        return kde / ep.kde3 / cx.lna, lhm, mm[:, :3].norm(dim=1)

    def pairs(self, x, prt):
        """Sums over receptor points: six terms and the contact counts."""
        ep = self.ep
        d2 = ((x[:, :, None, :] - prt) ** 2).sum(-1)
        d = torch.sqrt(d2)
        d3 = d2 * d
        vdw = (self.p1a - self.p2a * d3) / (self.p1a * ep.lj0 * (1.0 + ep.lj1 * d2) + d3 * d3 * d3)
        t = ep.el1 * d
        ele = self.q * self.ele * torch.where(t < 1.0, ep.el0 + ep.a1 * t * t + ep.b1 * t ** 3, 1.0 / t)
        pmf = self.pmf1 * torch.sigmoid(-(6.0 - 0.5 * d) * (d - self.pmf0))
        con = d <= self.pmf0
        hdb = self.hb * torch.exp(-0.5 * ((d - self.h0) * self.h1) ** 2)
        u = (1.0 - d2 / 81.0).clamp(min=0.0)
        hpc = (self.hpp * (0.5 * u ** 3 * (1.0 + u))).sum(-1)
        h = (hpc - self.hpl[0]) / self.hpl[1]
        both = lambda v: v.sum((1, 2))  # noqa: E731
        return (both(vdw), both(ele), both(pmf), both(self.psp * con), both(hdb),
                (0.5 * h * h - self.hpl[2]).sum(-1), both(con.double()),
                both((con & self.ref).double()))

    def energy(self, il, ip, mm):
        """(e [n, 10], cms [n], rmsd [n]) of poses given as float64 tensors."""
        cx, ep, n = self.cx, self.ep, len(mm)
        x = self.place(il, mm)
        raw = torch.empty(n, 8, dtype=torch.float64, device=self.dev)
        step = max(1, int(1.6e7 // (cx.lna * cx.pnp)))
        for p in range(cx.n_prt):
            sel = torch.nonzero(ip == p)[:, 0]
            for b in range(0, len(sel), step):
                k = sel[b:b + step]
                raw[k] = torch.stack(self.pairs(x[k], self.prt[p]), -1)
        kde, lhm, dst = self.cheap(x, mm)
        e = torch.cat([raw[:, :6] / cx.lna, torch.stack([kde, lhm, dst], -1)], 1)
        a, b, w = (torch.tensor(list(v)[:9], dtype=torch.float64, device=self.dev)
                   for v in (ep.a_para, ep.b_para, ep.w))
        e = e * a + b
        rmsd = torch.sqrt(((x - (self.lig[il] + self.center)) ** 2).sum((1, 2)) / cx.lna)
        ref = float(self.ref.sum())
        tp, fp = raw[:, 7], raw[:, 6] - raw[:, 7]
        fn = ref - tp
        tn = cx.lna * cx.pnp - ref - fp
        den = torch.sqrt((tp + fp) * (tp + fn) * (tn + fp) * (tn + fn))
        cms = torch.where(den > 0, (tp * tn - fp * fn) / den.clamp(min=1.0), torch.zeros_like(den))
        return torch.cat([e, (e * w).sum(1, keepdim=True)], 1), cms, rmsd


def _philox(c0, c1, c2, c3, seed):
    """Philox4x32-10 of counters (arrays or numbers) under a 64-bit key."""
    x = [np.asarray(v, np.uint64) for v in np.broadcast_arrays(c0, c1, c2, c3)]
    k0, k1, low = seed & 0xFFFFFFFF, seed >> 32, np.uint64(0xFFFFFFFF)
    for r in range(10):
        p0, p1 = np.uint64(0xD2511F53) * x[0], np.uint64(0xCD9E8D57) * x[2]
        a, b = (np.uint64((k + r * w) & 0xFFFFFFFF) for k, w in ((k0, 0x9E3779B9), (k1, 0xBB67AE85)))
        x = [(p1 >> np.uint64(32)) ^ x[1] ^ a, p1 & low, (p0 >> np.uint64(32)) ^ x[3] ^ b, p0 & low]
    return [((v >> np.uint64(8)) + np.uint64(1)).astype(np.float64) * 2.0 ** -24 for v in x]


def _chain64(cx, cid, seed, steps, nc, keep):
    """Replica-exchange Metropolis of one complex from its start poses, with
    the engine's random streams: final poses and energies, accepted states."""
    m = _Model(cx)
    n_lig, n_prt, n_tmp = cx.n_lig, cx.n_prt, cx.n_tmp
    flat = np.arange(cx.n_rep)
    il = torch.tensor(flat % n_lig, device=m.dev)
    ip = torch.tensor(flat // (n_lig * n_tmp), device=m.dev)
    tmp = (flat // n_lig) % n_tmp
    lad = (flat // (n_lig * n_tmp)) * n_lig + flat % n_lig
    slots = np.argsort(lad * n_tmp + tmp).reshape(-1, n_tmp)
    beta = np.asarray(cx.temp_minus_beta, np.float64)
    scale = np.asarray(cx.move_scale, np.float64)
    mm = torch.zeros(cx.n_rep, 6, dtype=torch.float64, device=m.dev)
    e, cms, rmsd = m.energy(il, ip, mm)
    best, best_mm = e[:, 9].clone(), mm.clone()
    log = [(flat, e, rmsd, mm.clone())]
    for s in range(steps):
        u = np.stack(_philox(s, flat, cid, 0, seed) + _philox(s, flat, cid, 1, seed), -1)
        if cx.move_kind == abi.MOVE_GAUSSIAN:
            r, th = np.sqrt(-2.0 * np.log(u[:, 0:6:2])), 2.0 * math.pi * u[:, 1:6:2]
            d = np.stack([r * np.cos(th), r * np.sin(th)], -1).reshape(-1, 6) * scale
        else:
            d = scale * (2.0 * u[:, :6] - 1.0)
        new = mm + torch.tensor(d, device=m.dev)
        en, cn, rn = m.energy(il, ip, new)
        de = (en[:, 9] - e[:, 9]).cpu().numpy()
        ok = u[:, 6] < np.exp(np.minimum(de * beta[tmp], 50.0))
        k = torch.tensor(ok, device=m.dev)
        mm = torch.where(k[:, None], new, mm)
        e, cms, rmsd = torch.where(k[:, None], en, e), torch.where(k, cn, cms), torch.where(k, rn, rmsd)
        low = e[:, 9] < best
        best, best_mm = torch.where(low, e[:, 9], best), torch.where(low[:, None], mm, best_mm)
        if keep:
            log.append((flat[ok], e[k], rmsd[k], mm[k]))
        if (s + 1) % nc == 0 and n_tmp > 1:
            seg = (s + 1) // nc - 1
            mode = 1 if seg % 2 == 0 else 0
            et, ts = e[:, 9].cpu().numpy(), tmp[slots]
            order = np.argsort(ts, 1)
            for pair in range(n_tmp // 2 - (n_tmp % 2 == 0 and mode == 1)):
                i = 2 * pair + mode
                o1 = slots[np.arange(len(slots)), order[:, i]]
                o2 = slots[np.arange(len(slots)), order[:, i + 1]]
                up = _philox(seg, np.arange(len(slots)), cid, 0x100 + pair, seed)[0]
                swap = np.exp(np.minimum((beta[i] - beta[i + 1]) * (et[o2] - et[o1]), 50.0)) > up
                tmp[o1[swap]], tmp[o2[swap]] = i + 1, i
    out = dict(movematrix=mm, e=e, cms=cms, rmsd=rmsd, best_e=best, best_movematrix=best_mm)
    if keep:
        rep = np.concatenate([x[0] for x in log])
        o = torch.tensor(np.argsort(rep, kind="stable"), device=m.dev)
        out["records"] = {}
        for k, i in (("e", 1), ("rmsd", 2), ("movematrix", 3)):
            r = torch.cat([x[i] for x in log])[o]
            room = r.new_zeros(cx.n_rep * (steps + 1), *r.shape[1:])
            room[:len(r)] = r
            out["records"][k] = room
    return out


def _grid64(cx, prt, dev):
    """Radial features on the grid nodes of one receptor conformer."""
    n = int(math.ceil(2 * HALF_WIDTH / SPACING)) + 1
    # the engine places its nodes from an origin rounded to float32
    ax = [float(np.float32(np.float32(v) - np.float32(HALF_WIDTH))) + SPACING * torch.arange(n, dtype=torch.float64, device=dev)
          for v in cx.pocket_center]
    P = torch.tensor(np.stack([np.asarray(a, np.float64).reshape(cx.n_prt, -1)[prt]
                               for a in (cx.prt_x, cx.prt_y, cx.prt_z)], -1), device=dev)
    cls = torch.tensor(np.asarray(cx.prt_t) % 4, device=dev)
    yz = torch.stack(torch.meshgrid(ax[1], ax[2], indexing="ij"), -1).reshape(-1, 2)
    g = torch.zeros(n, n * n, 32, dtype=torch.float64, device=dev)
    for i in range(n):
        pts = torch.cat([ax[0][i].expand(len(yz), 1), yz], 1)
        for c in range(4):
            q = P[(cls == c) & ((P[:, 0] - ax[0][i]).abs() < 8.0)]
            d = torch.sqrt(((pts[:, None] - q) ** 2).sum(-1))
            fc = torch.where(d < 8.0, 0.5 * (1.0 + torch.cos(math.pi * d / 8.0)), torch.zeros_like(d))
            for k in range(8):
                g[i, :, 8 * c + k] = (torch.exp(-0.5 * (d - (k + 1)) ** 2) * fc).sum(-1)
    return g.reshape(n, n, n, 32), [float(a[0]) for a in ax]


def _interp(grid, origin, x):
    n = grid.shape[0]
    u = ((x - torch.tensor(origin, dtype=torch.float64, device=x.device)) / SPACING).clamp(0, n - 1 - 1e-9)
    i = u.long()
    t = u - i
    out = 0.0
    for c in range(8):
        b = [(c >> 2) & 1, (c >> 1) & 1, c & 1]
        w = math.prod(t[..., k] if b[k] else 1.0 - t[..., k] for k in range(3))
        out = out + w[..., None] * grid[i[..., 0] + b[0], i[..., 1] + b[1], i[..., 2] + b[2]]
    return out


def _params64(flat):
    return [v.to(torch.float64) for v in
            torch.split(flat, [64 * 128, 128 * 128, 128, 128, 1])]


def _net64(p, F):
    """Network outputs of feature rows F [N, 57] (the last column is 1)."""
    silu = torch.nn.functional.silu
    h = silu(F @ p[0].view(64, 128)[:57])
    return silu(h @ p[1].view(128, 128) + p[2]) @ p[3] + p[4]


def _rows64(cx, radial):
    lt = torch.nn.functional.one_hot(torch.tensor(np.asarray(cx.lig_t), device=radial.device).long(), 24)
    lt = lt.to(torch.float64).expand(len(radial), -1, -1)
    return torch.cat([lt, radial, torch.ones_like(radial[..., :1])], -1)


def _tables64(c, seed):
    out = []
    for i, cx in enumerate(_complexes(c, seed)):
        m = _Model(cx)
        p = _params64(torch.tensor(surrogate.pack_params(_network(seed)), device=m.dev))
        il, ip, mm = (torch.tensor(a, device=m.dev) for a in _poses(c, c["poses"], seed + 7 * i))
        il, mm = il.long(), mm.double()
        x = m.place(il, mm)
        radial = torch.zeros(len(mm), cx.lna, 32, dtype=torch.float64, device=m.dev)
        y = torch.zeros(len(mm), cx.lna, dtype=torch.float64, device=m.dev)
        for q in range(cx.n_prt):
            sel = ip == q
            g, o = _grid64(cx, q, m.dev)
            radial[sel] = _interp(g, o, x[sel])
            flat = g.reshape(-1, 32)
            for t in np.unique(cx.lig_t):
                hot = torch.zeros(len(flat), 25, dtype=torch.float64, device=m.dev)
                hot[:, int(t)] = hot[:, 24] = 1.0
                tab = torch.cat([_net64(p, torch.cat([hot[b:b + 65536, :24], flat[b:b + 65536], hot[b:b + 65536, 24:]], 1))
                                 for b in range(0, len(flat), 65536)])
                at = torch.tensor(np.nonzero(np.asarray(cx.lig_t) == t)[0], device=m.dev)
                y[sel.nonzero(), at] = _interp(tab.reshape(*g.shape[:3], 1), o, x[sel][:, at])[..., 0]
        ep = m.ep
        s = 0.5 * y.sum(1) / cx.lna
        for k, v in zip((6, 7, 8), m.cheap(x, mm)):
            s = s + (ep.a_para[k] * v + ep.b_para[k]) * ep.w[k]
        out.append(dict(features=_rows64(cx, radial)[..., :56], total=s))
    return out


def _train64(c, seed):
    cx = _complexes(c, seed)[0]
    m = _Model(cx)
    il, ip, mm = _poses(c, c["poses"] + c["held_out"], seed)
    target = torch.tensor(_targets(mm, seed), device=m.dev).double()
    il, ip, mm = torch.tensor(il, device=m.dev).long(), torch.tensor(ip, device=m.dev), torch.tensor(mm, device=m.dev).double()
    grids = [_grid64(cx, q, m.dev) for q in range(cx.n_prt)]

    def rows(b, e):
        x = m.place(il[b:e], mm[b:e])
        r = torch.zeros(e - b, cx.lna, 32, dtype=torch.float64, device=m.dev)
        for q, (g, o) in enumerate(grids):
            sel = ip[b:e] == q
            r[sel] = _interp(g, o, x[sel])
        return _rows64(cx, r)

    flat = torch.tensor(surrogate.pack_params(_network(seed)), device=m.dev).double()
    mom, var, t, n, hist = torch.zeros_like(flat), torch.zeros_like(flat), 0, c["poses"], []
    cuts = [(b, min(n, b + c["batch"])) for b in range(0, n, c["batch"])]
    for ep in range(c["epochs"]):
        sq = 0.0
        for b, e in cuts:
            w = flat.clone().requires_grad_(True)
            res = _net64(_params64(w), rows(b, e)).sum(1) - target[b:e]
            (res * res).mean().backward()
            sq += float((res.detach() ** 2).sum())
            g, t = w.grad, t + 1
            mom, var = 0.9 * mom + 0.1 * g, 0.999 * var + 0.001 * g * g
            flat = flat - 1e-3 * (mom / (1 - 0.9 ** t)) / (torch.sqrt(var / (1 - 0.999 ** t)) + 1e-8)
        hist.append(sq / n)
    with torch.no_grad():
        p = _params64(flat)
        hist[-1] = sum(float(((_net64(p, rows(b, e)).sum(1) - target[b:e]) ** 2).sum()) for b, e in cuts) / n
        held = _net64(p, rows(n, n + c["held_out"])).sum(1)
    return dict(loss=np.array(hist), params=flat, held_out=held)


def exact(case, seed):
    """None for clustering, which returns whole numbers, and for delayed
    acceptance, whose chain follows decisions of a network in bf16."""
    c, kind = case, case["kind"]
    if kind in ("post", "da"):
        return None
    if kind == "tables":
        return _tables64(c, seed)
    if kind == "train":
        return _train64(c, seed)
    if kind == "score":
        il, ip, mm = _poses(c, c["poses"], seed)
        m = _Model(_complexes(c, seed)[0])
        e, cms, rmsd = m.energy(torch.tensor(il, device=m.dev).long(), torch.tensor(ip, device=m.dev),
                                torch.tensor(mm, device=m.dev).double())
        return dict(e=e, cms=cms, rmsd=rmsd)
    cxs = _complexes(c, seed)
    if sum(x.n_rep * x.lna * (x.pnp + x.pnk) for x in cxs) * c["steps"] > EXACT_PAIRS:
        return None
    keep = kind == "call" or (c["record"] and len(cxs) == 1)
    got = [_chain64(x, i, seed, c["steps"], 20, keep) for i, x in enumerate(cxs)]
    if kind == "call":
        return dict(records=got[0]["records"])
    out = {k: torch.cat([g[k] for g in got]) for k in got[0] if k != "records"}
    if c["record"]:
        del out["best_e"], out["best_movematrix"]
    if keep:
        out["records"] = got[0]["records"]
    return out
