"""The calls whose speed this library is about, at the sizes its users run.

Each case is one pass through the public Python mirror of the C ABI
(`pas_cg_amd.pcg`): a plain context stepping one system, a batch advancing
many, a server draining a backlog of jobs, or the drop-in host's per-term
calls. A pass returns what a user reads afterwards: the frame (positions, and
velocities of a plain context) and the energies. Passes on one state continue
its trajectory, as a simulation does.

The proteins are windows of compact self-avoiding walks of the package's own
generator (3.8 A bonds, native contacts below 7.5 A), with residue types, a
small thermal displacement, velocities and noise keys from the seed. The
force fields, lengths, batch sizes and boxes are those of the package's
workloads and tests.
"""
import functools
import math

import numpy as np

import pcg_import

pcg_import.load()
from pas_cg_amd import model as M  # noqa: E402
from pas_cg_amd import params as P  # noqa: E402
from pas_cg_amd import pcg as G  # noqa: E402
from pas_cg_amd import workloads as W  # noqa: E402

A = P.ANGSTROM
WALK = 600          # longest protein of the batched and served workloads
LONG_WALK = 2000    # longest job of the served stream


def listed():
    return [
        # a host that steps one small protein itself and logs the energy of
        # every step: launch latency and synchronisation
        {"name": "chain56_each_step", "kind": "each", "n": 56, "steps": 10},
        # the same protein between two frames of a trajectory
        {"name": "chain56", "kind": "chain", "n": 56, "field": "go", "steps": 200},
        # one mid-sized protein in the full force field, pulled by its end
        {"name": "protein301", "kind": "chain", "n": 301, "field": "full", "steps": 100},
        # the longest single chain the workloads know
        {"name": "chain2000", "kind": "chain", "n": 2000, "field": "full", "steps": 40},
        # reproducing the reference's trajectory: FP64 and its ran2 noise,
        # drawn on the host
        {"name": "parity153_fp64", "kind": "parity", "n": 153, "steps": 20},
        # the drop-in host calling one step's tasks one by one
        {"name": "terms300", "kind": "terms", "n": 300},
        # the crowded solution: 64 chains of 100 in a periodic 1 mM box
        {"name": "box64x100", "kind": "box", "copies": 64, "n": 100, "steps": 40},
        # a protein assembly squeezed by the walls of the simulation box
        {"name": "walls8x60", "kind": "walls", "copies": 8, "n": 60, "steps": 40},
        # an ensemble of replicas of one small chain
        {"name": "replicas1024x56", "kind": "batch", "count": 1024, "lo": 56, "hi": 56,
         "field": "go", "fp64": False, "steps": 500},
        # the headline batch: distinct proteins of 30 to 600 residues
        {"name": "ragged256", "kind": "batch", "count": 256, "lo": 30, "hi": 600,
         "field": "full", "fp64": False, "steps": 250},
        # a smaller batch in FP64, some of it on the heuristic angles and
        # dihedrals of a sequence without a structure
        {"name": "ragged48_fp64", "kind": "batch", "count": 48, "lo": 30, "hi": 400,
         "field": "heur", "fp64": True, "steps": 100},
        # a backlog of short jobs through the server
        {"name": "served64", "kind": "served", "jobs": 64, "steps": 400},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["each", "chain", "chain", "parity", "terms", "box", "walls", "batch",
                       "batch", "served"])
    if kind == "each":
        return {"kind": kind, "n": _log_int(rng, 20, 200), "steps": rng.randint(5, 20)}
    if kind == "chain":
        return {"kind": kind, "n": _log_int(rng, 20, 2000), "field": rng.choice(["go", "full"]),
                "steps": rng.randint(20, 100)}
    if kind == "parity":
        return {"kind": kind, "n": _log_int(rng, 30, 400), "steps": rng.randint(10, 30)}
    if kind == "terms":
        return {"kind": kind, "n": _log_int(rng, 30, 2000)}
    if kind == "box":
        return {"kind": kind, "copies": rng.randint(8, 64), "n": rng.randint(40, 100),
                "steps": rng.randint(20, 40)}
    if kind == "walls":
        return {"kind": kind, "copies": rng.randint(2, 16), "n": rng.randint(30, 80),
                "steps": rng.randint(20, 40)}
    if kind == "batch":
        lo, hi = sorted((_log_int(rng, 20, 600), _log_int(rng, 20, 600)))
        fp64 = rng.random() < 0.25
        return {"kind": kind, "count": _log_int(rng, 8, 160 if hi > 150 else 1024), "lo": lo,
                "hi": hi, "field": rng.choice(["go", "full", "heur"]), "fp64": fp64,
                "steps": rng.randint(50, 100 if fp64 else 250 if hi > 150 else 500)}
    return {"kind": kind, "jobs": rng.randint(8, 64), "steps": rng.randint(100, 400)}


# ------------------------------------------------------------------ inputs ----

@functools.lru_cache(maxsize=None)
def _walk(j, length):
    return M.synthetic_protein(length, M.job_seed(j))


def _protein(n, rng, heur=False):
    """Residues [o, o + n) of one of the walks, its types drawn anew, started
    a few hundredths of an angstrom off the native conformation; with heur a
    third of the angles and dihedrals have no native value."""
    w = _walk(int(rng.integers(0, 6)), WALK) if n <= WALK else _walk(6, LONG_WALK)
    o = int(rng.integers(0, w["n"] - n + 1))
    chain = np.zeros(n, np.int32)
    teth, ang, dih = _lists(n)
    inside = (w["cont"][:, 0] >= o) & (w["cont"][:, 1] < o + n)
    nat = w["pos"][o:o + n] - w["pos"][o:o + n].mean(axis=0)
    m = {"n": n, "pos": nat + rng.normal(scale=0.05 * A, size=(n, 3)), "orig_pos": nat,
         "atype": rng.integers(0, 20, size=n).astype(np.uint8), "chain": chain,
         "seq": np.arange(n, dtype=np.int32), "teth": teth, "ang": ang,
         "ang_has": np.ones(len(ang), np.uint8), "ang_theta": w["ang_theta"][o:o + len(ang)],
         "dih": dih, "dih_has": np.ones(len(dih), np.uint8),
         "dih_phi": w["dih_phi"][o:o + len(dih)], "cont": w["cont"][inside] - np.int32(o),
         "cont_len": w["cont_len"][inside], "cont_type": np.zeros(int(inside.sum()), np.int32),
         "cell": np.zeros(3)}
    if heur:
        m["ang_has"][rng.uniform(size=len(ang)) < 1 / 3] = 0
        m["dih_has"][rng.uniform(size=len(dih)) < 1 / 3] = 0
    return M.empty_tips(m)


@functools.lru_cache(maxsize=None)
def _lists(n):
    return M.chain_lists(np.zeros(n, np.int32))


def _field(name):
    if name == "go":
        return W.base_params()
    p = W.full_params()
    if name == "heur":  # electrostatics and Pauli exclusion instead of QA contacts
        p.update(qa_on=0, pid_on=0)
    return p


def _velocities(n, rng, p):
    """Maxwell velocities of unit masses times dt: the context's y1."""
    return rng.normal(scale=math.sqrt(p["temperature"]) * p["dt"], size=(n, 3))


def _inputs(case, seed):
    """Parameters, model and y1 of a case with one system."""
    rng = np.random.default_rng([seed, 448])
    kind, n = case["kind"], case["n"]
    if kind in ("box", "walls"):
        one, copies = _protein(n, rng), case["copies"]
        if kind == "box":
            p = _field("full")
            p.update(afm_on=0)
            side = W.c1(1, n, one)[1]["cell"][0] * copies ** (1 / 3)
            m = M.replicate(one, copies, side, seed=int(rng.integers(1 << 30)))
        else:
            p = P.default_params()
            p.update(qa_on=0, pid_on=0, afm_on=0)
            P.set_box_walls(p, {"x": "solid", "y": "solid", "z": "solid"}, n * copies)
            m = M.replicate(one, copies, 48.0 * A * (copies * n / 60) ** (1 / 3),
                            seed=int(rng.integers(1 << 30)))
            m["cell"] = np.zeros(3)
    elif kind == "parity":
        p = P.default_params()
        p.update(chir_on=1)
        m = _protein(n, rng)
    else:
        p = _field(case.get("field", "go" if kind == "each" else "full"))
        m = _protein(n, rng)
        if p["afm_on"]:
            m = M.add_pulling(m)
    return p, m, _velocities(m["n"], rng, p)


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng([seed, 448])
    # the lengths belong to the workload, everything else to the seed
    lengths = np.random.default_rng(448)
    if kind == "batch":
        p = _field(case["field"])
        ns = lengths.integers(case["lo"], case["hi"] + 1, size=case["count"])
        same = _protein(int(ns[0]), rng) if case["lo"] == case["hi"] else None
        ms = [same or _protein(int(n), rng, case["field"] == "heur" and k % 3 == 0)
              for k, n in enumerate(ns)]
        if p["afm_on"]:
            ms = [M.add_pulling(m) if k % 10 == 0 else m for k, m in enumerate(ms)]
        b = G.Batch(p, ms, precision=G.FP64 if case["fp64"] else G.MIXED,
                    seeds=[1 + (seed + k) % 1000003 for k in range(len(ms))], philox_seed=seed,
                    steps_per_launch=500)
        b.autotune(100)
        return {"case": case, "b": b}
    if kind == "served":
        p = _field("full")
        jobs = []
        for k in range(case["jobs"]):
            n = int(min(max(round(150.0 * math.exp(0.6 * lengths.normal())), 30), WALK))
            m = _protein(n, rng)
            jobs.append((M.add_pulling(m) if rng.uniform() < 0.2 else m,
                         float(rng.uniform(0.3, 0.45)), 1 + int(rng.integers(1 << 20))))
        srv = G.Server(p, hbm_budget_bytes=32 << 30, chunk_steps=200, philox_seed=seed)
        return {"case": case, "srv": srv, "jobs": jobs}
    p, m, y1 = _inputs(case, seed)
    parity = kind == "parity"
    c = G.Context(p, m, precision=G.FP64 if parity else G.MIXED,
                  noise=G.RAN2 if parity else G.PHILOX, seed=1 + seed % 1000003, philox_seed=seed)
    c.set(1, y1)
    if kind == "box":
        c.use_graph(True)
    if kind == "walls":
        lo, hi = m["pos"].min(axis=0) - 3.5 * A, m["pos"].max(axis=0) + 3.5 * A
        c.box_setup(P.box_params(lo, hi, (0, 0, 0), squeezing=1))
        c.box_start()
    on = [t for t in G.TERMS if W.term_enabled(p).get(t)]
    return {"case": case, "c": c, "terms": on}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        b = state["b"]
        b.run(case["steps"])
        return np.concatenate([b.get(s, 0) for s in range(case["count"])])
    if kind == "served":
        srv = state["srv"]
        ids = [srv.submit(m, case["steps"], temperature=T, seed=s) for m, T, s in state["jobs"]]
        while srv.round():
            pass
        res = [srv.result(j) for j in ids]
        return np.concatenate([r for r, _ in res]), np.array([V for _, V in res])
    c = state["c"]
    if kind == "terms":
        if c.nl_verify():
            c.fix_nl()
        c.prepare_nh()
        got = [c.eval_term(t) for t in state["terms"]]
        c.qa_finish()
        return np.stack([F for F, _ in got]), np.array([V for _, V in got])
    if kind == "each":
        V = []
        for _ in range(case["steps"]):
            c.step(1)
            V.append(c.energy()[0])
        return c.get(0), np.array(V)
    c.step(case["steps"])
    if kind == "walls":
        return c.get(0), c.get(7), c.box_state(raw=True)
    return c.get(0), c.get(7), np.array([c.energy()[0]])


def work(case):
    """State (Gear derivatives, types, static lists) in and out once a pass,
    and the operations of its steps: bonded items, native contacts, pairs
    within the QA radius, the integrator, and the pair tests of a list rebuild
    every thirty steps."""
    kind, steps = case["kind"], case.get("steps", 1)
    if kind == "batch":
        n = case["count"] * (case["lo"] + case["hi"]) / 2
        size = (case["lo"] + case["hi"]) / 2
    elif kind == "served":
        n, size = 170.0 * case["jobs"], 170.0
    else:
        n, size = float(case["n"] * case.get("copies", 1)), float(case["n"])
    qa = kind not in ("each", "walls") and case.get("field") not in ("go", "heur")
    contacts = max(0.0, 4.6 - 12.0 / math.sqrt(size)) * n
    near = (25.0 * contacts / 4.6) if qa else 0.0
    rebuild = n * min(size, 600.0) * 8 / 30 if kind != "terms" else n * size * 4
    flops = 450.0 * n + 50.0 * contacts + 12.0 * near + 150.0 * n + rebuild
    if kind == "terms":
        state = n * (24 + 24 * 10)
    else:
        state = n * (2 * 6 * 24 + 24)
    return {"bytes": state + n * 60 + contacts * 16, "flops": flops * steps}


# --------------------------------------------------------------- 64 bits ----

def exact(case, seed):
    """What a plain context's pass returns, in 64-bit numpy: the force field
    and the Gear-5 Langevin step from their formulas, on the same inputs.
    None for the batches and the server (hundreds of systems take minutes)
    and where the noise or the box protocol is the outcome of a state machine
    on the host or device (ran2, walls)."""
    kind = case["kind"]
    if kind not in ("each", "chain", "terms", "box"):
        return None
    p, m, y1 = _inputs(case, seed)
    e = _Exact(p, m, y1, seed)
    if kind == "terms":
        e.rebuild()
        got = e.terms()
        on = [t for t in G.TERMS if W.term_enabled(p).get(t)]
        zero = (np.zeros((m["n"], 3)), 0.0)
        return (np.stack([got.get(t, zero)[0] for t in on]),
                np.array([got.get(t, zero)[1] for t in on]))
    V = [e.step() for _ in range(case["steps"])]
    if kind == "each":
        return e.y[0], np.array(V)
    return e.y[0], e.y[1] / p["dt"], np.array(V[-1:])


def _philox(key, step, n):
    """Philox4x32-10 (Salmon et al. 2011) of counters (step, residue, 0x5043)."""
    mask = np.uint64(0xFFFFFFFF)
    s32 = np.uint64(32)
    c = [np.full(n, step & 0xFFFFFFFF, np.uint64), np.full(n, step >> 32, np.uint64),
         np.arange(n, dtype=np.uint64), np.full(n, 0x5043, np.uint64)]
    k0, k1 = key & 0xFFFFFFFF, key >> 32
    for _ in range(10):
        a, b = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(b >> s32) ^ c[1] ^ np.uint64(k0), b & mask, (a >> s32) ^ c[3] ^ np.uint64(k1),
             a & mask]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return [x.astype(np.float64) * 2.0 ** -32 for x in c]


def _mix64(x):
    x = (x + 0x9E3779B97F4A7C15) % 2 ** 64
    x = ((x ^ (x >> 30)) * 0xBF58476D1CE4E5B9) % 2 ** 64
    x = ((x ^ (x >> 27)) * 0x94D049BB133111EB) % 2 ** 64
    return x ^ (x >> 31)


def _norm(d):
    return np.sqrt((d * d).sum(axis=1))


class _Exact:
    def __init__(self, p, m, y1, seed):
        self.p, self.m, self.n = p, m, m["n"]
        self.y = [m["pos"].copy(), y1.copy()] + [np.zeros_like(y1) for _ in range(4)]
        self.step_no, self.t = 0, 0.0
        self.key = _mix64(seed ^ _mix64(1))
        self.cell = np.asarray(m["cell"])
        self.orig = None
        d = m["dih"]
        r = m["pos"]
        b12, b23, b34 = r[d[:, 1]] - r[d[:, 0]], r[d[:, 2]] - r[d[:, 1]], r[d[:, 3]] - r[d[:, 2]]
        self.chir1 = 1.0 / _norm(b23) ** 3
        self.chir0 = (b12 * np.cross(b23, b34)).sum(axis=1) * self.chir1
        self.teth_len = _norm(m["orig_pos"][m["teth"][:, 1]] - m["orig_pos"][m["teth"][:, 0]])
        self.sync = np.array(p["base_sync"])[m["atype"]]
        self.hi = np.array(p["qa_lj_r_high"])
        self.max_req = self.hi.max()
        same_next = np.diff(m["chain"]) == 0
        self.inner = np.zeros(self.n, bool)
        self.inner[1:-1] = same_next[1:] & same_next[:-1]
        self.qc = []  # contacts: [i, j, original distance, type, saturation, deltas, vacant]
        self.free = 0

    def _wrap(self, d):
        if not self.cell.any():
            return d
        return d - self.cell * np.round(d / self.cell)

    def _pair(self, ij):
        return self._wrap(self.y[0][ij[:, 1]] - self.y[0][ij[:, 0]])

    def _scatter(self, parts):
        F = np.zeros((self.n, 3))
        for i, f in parts:
            for c in range(3):
                F[:, c] += np.bincount(i, f[:, c], self.n)
        return F

    def rebuild(self):
        p, m, r = self.p, self.m, self.y[0]
        self.orig = r.copy()
        reach = max(p["nl_cutoff"], p["dh_cutoff"]) + p["nl_pad"]
        keep, dist = [], []
        for a in range(0, self.n, 256):
            rows = np.arange(a, min(a + 256, self.n))
            d = self._wrap(r[None, a:] - r[rows][:, None])
            d2 = (d * d).sum(axis=2)
            i, j = np.nonzero(d2 < reach * reach)
            i, j, d2 = i + a, j + a, d2[i, j]
            near = (m["chain"][i] == m["chain"][j]) & (np.abs(m["seq"][i] - m["seq"][j]) < 3)
            ok = (j > i) & ~near
            keep.append(np.stack([i[ok], j[ok]], axis=1))
            dist.append(np.sqrt(d2[ok]))
        ij, d = np.concatenate(keep), np.concatenate(dist)
        code = np.sort(m["cont"].astype(np.int64), axis=1) @ np.array([self.n, 1])
        order = np.argsort(code)
        at = np.searchsorted(code[order], ij[:, 0] * self.n + ij[:, 1])
        at = order[np.minimum(at, len(code) - 1)] if len(code) else np.zeros(len(ij), int)
        nat = (code[at] == ij[:, 0] * self.n + ij[:, 1]) if len(code) else np.zeros(len(ij), bool)
        inner = d < p["nl_cutoff"] + p["nl_pad"]
        nat &= inner
        self.nc, self.nc_len = ij[nat], (m["cont_len"][at][nat] if len(code) else d[:0])
        qa = ~nat & inner if p["qa_on"] else np.zeros(len(ij), bool)
        near = qa & (d <= self.max_req)
        self.free = int(qa.sum())
        self.qh, self.qh_d = ij[near], d[near]
        self.qh_vac = np.zeros(len(self.qh), bool)
        rest = ~nat & ~qa
        q = np.array(p["charge"])[m["atype"]]
        dh = rest & (q[ij[:, 0]] * q[ij[:, 1]] != 0) & (d < p["dh_cutoff"] + p["nl_pad"])
        self.dh = ij[dh] if p["dh_on"] else ij[:0]
        self.dh_q = q[self.dh[:, 0]] * q[self.dh[:, 1]]
        pauli = p["pauli_on"] and not p["qa_on"]
        self.pauli = ij[rest & (d < p["rep_cutoff"] + p["nl_pad"])] if pauli else ij[:0]

    def _repulsion(self, ij, depth):
        d = self._pair(ij)
        r = _norm(d)
        ok = r < self.p["rep_cutoff"]
        ij, d, r = ij[ok], d[ok], r[ok]
        s6 = (self.p["rep_cutoff"] / r) ** 6
        dV = np.clip(12.0 * depth / r * (s6 - s6 * s6), -1e3, 1e3)
        f = (dV / r)[:, None] * d
        return self._scatter([(ij[:, 0], f), (ij[:, 1], -f)]), float(
            (depth * (s6 * s6 - 2.0 * s6 + 1.0)).sum())

    def terms(self):
        p, m, r = self.p, self.m, self.y[0]
        out = {}
        t, a, q = m["teth"], m["ang"], m["dih"]
        d = r[t[:, 1]] - r[t[:, 0]]
        ln = _norm(d)
        dr = ln - self.teth_len
        f = (np.clip(dr * (p["tether_H1"] + 2 * p["tether_H2"] * dr * dr), -1e3, 1e3) / ln)[:, None] * d
        out["tether"] = (self._scatter([(t[:, 0], f), (t[:, 1], -f)]),
                         float((0.5 * dr * dr * (p["tether_H1"] + p["tether_H2"] * dr * dr)).sum()))
        cell, self.cell = self.cell, np.zeros(3)  # bonded items are not wrapped
        out["lrep"] = self._repulsion(a[:, [0, 2]], p["lrep_depth"])
        self.cell = cell
        # bond angles
        r12, r23 = r[a[:, 1]] - r[a[:, 0]], r[a[:, 2]] - r[a[:, 1]]
        x = np.cross(r12, r23)
        l12, l23, lx = _norm(r12)[:, None], _norm(r23)[:, None], _norm(x)[:, None]
        d1 = np.cross(r12, x) / (lx * l12 * l12)
        d3 = np.cross(r23, x) / (lx * l23 * l23)
        th = np.arctan2(lx[:, 0], -(r12 * r23).sum(axis=1))
        dth = th - m["ang_theta"]
        g = (2.0 * p["CBA"] * dth)[:, None]
        out["nat_ang"] = (self._scatter([(a[:, 0], -g * d1), (a[:, 1], g * (d1 + d3)),
                                         (a[:, 2], -g * d3)]), float((p["CBA"] * dth * dth).sum()))
        # dihedrals (the complex native variant) and chirality
        r12, r23, r34 = r[q[:, 1]] - r[q[:, 0]], r[q[:, 2]] - r[q[:, 1]], r[q[:, 3]] - r[q[:, 2]]
        x1, x2 = np.cross(r12, r23), np.cross(r23, r34)
        n1, n2, l23 = _norm(x1), _norm(x2), _norm(r23)
        phi = np.arctan2(l23 * (x1 * r34).sum(axis=1), (x1 * x2).sum(axis=1)) - m["dih_phi"]
        g = (p["CDA"] * np.sin(phi) + 3.0 * p["CDB"] * np.sin(3.0 * phi))[:, None]
        d1, d4 = -x1 * (l23 / n1 ** 2)[:, None], x2 * (l23 / n2 ** 2)[:, None]
        df = (-d1 * (r12 * r23).sum(axis=1)[:, None] +
              d4 * (r23 * r34).sum(axis=1)[:, None]) / (l23 ** 2)[:, None]
        d2, d3 = -d1 + df, -d4 - df
        out["cnd"] = (self._scatter([(q[:, k], -g * dk) for k, dk in enumerate((d1, d2, d3, d4))]),
                      float((p["CDA"] * (1 - np.cos(phi)) + p["CDB"] * (1 - np.cos(3 * phi))).sum()))
        if p["chir_on"]:
            c13 = np.cross(r12, r34)
            cd = (r12 * x2).sum(axis=1) * self.chir0 - self.chir1
            g = (p["e_chi"] * cd * self.chir0)[:, None]
            out["chir"] = (self._scatter([(q[:, 0], g * x1), (q[:, 1], -g * (c13 + x2)),
                                          (q[:, 2], g * (x1 + c13)), (q[:, 3], -g * x1)]),
                           float((0.5 * p["e_chi"] * cd * cd).sum()))
        # native contacts
        d = self._pair(self.nc)
        ln = _norm(d)
        ok = ln < p["nl_cutoff"]
        ij, d, ln, nat = self.nc[ok], d[ok], ln[ok], self.nc_len[ok]
        s6 = (nat / ln) ** 6
        dV = np.clip(12.0 * p["nat_cont_depth"] / ln * (s6 - s6 * s6), -1e3, 1e3)
        f = (dV / ln)[:, None] * d
        out["nat_cont"] = (self._scatter([(ij[:, 0], f), (ij[:, 1], -f)]),
                           float((p["nat_cont_depth"] * (s6 * s6 - 2 * s6)).sum()))
        out["pauli"] = self._repulsion(self.pauli, p["pauli_depth"])
        # Debye-Hueckel, constant permittivity
        d = self._pair(self.dh)
        ln = _norm(d)
        ok = ln <= p["dh_cutoff"]
        ij, d, ln = self.dh[ok], d[ok], ln[ok]
        V = self.dh_q[ok] * np.exp(-ln / p["dh_screen_dist"]) / (4 * math.pi * p["dh_perm"] * ln)
        f = (-V * (1 / p["dh_screen_dist"] + 1 / ln) / ln)[:, None] * d
        out["const_dh"] = (self._scatter([(ij[:, 0], f), (ij[:, 1], -f)]), float(V.sum()))
        if p["afm_on"] and len(m["tip_res"]):
            d = m["tip_orig"] + self.t * m["tip_vel"] - r[m["tip_res"]]
            ln = _norm(d)
            ok = ln > 1e-10
            d, ln, res = d[ok], ln[ok], m["tip_res"][ok]
            dV = np.clip(ln * (p["afm_H1"] + 2 * p["afm_H2"] * ln * ln), -1e3, 1e3)
            out["vel_afm"] = (self._scatter([(res, (dV / ln)[:, None] * d)]),
                              float((0.5 * ln * ln * (p["afm_H1"] + p["afm_H2"] * ln * ln)).sum()))
        if p["qa_on"]:
            out["qa_cand"] = self._candidates()
            out["qa_cont"] = self._contacts()
        return out

    def _candidates(self):
        p, r = self.p, self.y[0]
        live = np.flatnonzero(~self.qh_vac)
        d = self._pair(self.qh[live])
        ln = _norm(d)
        rep = self._repulsion(self.qh[live], p["pauli_depth"])
        ok = ln <= self.max_req
        live, d, ln = live[ok], d[ok], ln[ok]
        i, j = self.qh[live, 0], self.qh[live, 1]
        nv, hv = np.zeros((self.n, 3)), np.zeros((self.n, 3))
        k = np.flatnonzero(self.inner)
        v1, v2 = r[k] - r[k - 1], r[k + 1] - r[k]
        nv[k] = (v2 - v1) / _norm(v2 - v1)[:, None]
        h = np.cross(v2, v1)
        hv[k] = h / _norm(h)[:, None]
        u = d / ln[:, None]
        back1 = np.abs((hv[i] * u).sum(axis=1)) > p["qa_min_cos_hr"]
        back2 = np.abs((hv[j] * u).sum(axis=1)) > p["qa_min_cos_hr"]
        hh = np.abs((hv[i] * hv[j]).sum(axis=1)) > p["qa_min_cos_hh"]
        side1 = (nv[i] * u).sum(axis=1) < p["qa_max_cos_nr"]
        side2 = -(nv[j] * u).sum(axis=1) < p["qa_max_cos_nr"]
        ai, aj = self.m["atype"][i].astype(int), self.m["atype"][j].astype(int)
        ty = np.where(back1 & back2 & hh, 1, np.where(back1 & side2, 2, np.where(
            side1 & back2, 3, np.where(side1 & side2, 4 + ai + 21 * aj, 0))))
        ok = (ty > 0) & (ln <= self.hi[ty] * (1.0 + p["qa_formation_tol"]))
        pt = np.array(p["ptype"])
        s1 = np.stack([back1, side1, side1 & (pt[aj] == 1), side1 & (pt[aj] == 2)], axis=1)
        s2 = np.stack([back2, side2, side2 & (pt[ai] == 1), side2 & (pt[ai] == 2)], axis=1)
        ok &= ((self.sync[i] - s1) >= 0).all(axis=1) & ((self.sync[j] - s2) >= 0).all(axis=1)
        self.cand = sorted((ln[c], live[c], ty[c], s1[c].astype(int), s2[c].astype(int))
                           for c in np.flatnonzero(ok))
        return rep

    def _contacts(self):
        p = self.p
        F, V, self.gone = np.zeros((self.n, 3)), 0.0, []
        for k, c in enumerate(self.qc[:self.free]):
            if c[6]:
                continue
            d = self._wrap(self.y[0][c[1]] - self.y[0][c[0]])
            ln = math.sqrt(d @ d)
            if ln > p["nl_cutoff"]:
                continue
            depth, lo, hi = p["qa_lj_depth"][c[3]], p["qa_lj_r_low"][c[3]], p["qa_lj_r_high"][c[3]]
            s6 = (min(max(ln, lo), hi) / ln) ** 6
            f = c[4] * 12.0 * depth / ln * (s6 - s6 * s6) / ln * d
            F[c[0]] += f
            F[c[1]] -= f
            V += c[4] * depth * (s6 * s6 - 2.0 * s6)
            step = p["dt"] / p["qa_phase_dur"]
            if ln > p["counting_factor"] * P.C216_INV * hi:
                c[4] = min(c[4] - step, 0.0)
                if c[4] == 0.0:
                    self.gone.append(k)
            else:
                c[4] = max(c[4] + step, 0.0)
        return F, V

    def _finish(self):
        for k in self.gone:
            c = self.qc[k]
            self.sync[c[0]] += c[5][:4]
            self.sync[c[1]] += c[5][4:]
            if c[2] <= self.max_req:
                self.qh = np.concatenate([self.qh, [[c[0], c[1]]]])
                self.qh_d = np.append(self.qh_d, c[2])
                self.qh_vac = np.append(self.qh_vac, False)
            self.free += 1
            c[6] = True
        for _, h, ty, s1, s2 in self.cand:
            i, j = self.qh[h]
            if (self.sync[i] - s1 < 0).any() or (self.sync[j] - s2 < 0).any():
                continue
            self.sync[i] -= s1
            self.sync[j] -= s2
            self.qc.append([i, j, self.qh_d[h], ty, 0.0, np.concatenate([s1, s2]), False])
            self.qh_vac[h] = True
        live = [c for c in self.qc if not c[6]]
        if (self.gone or self.cand) and 2 * len(live) < len(self.qc):
            # the items close up, the vacancy flags of the slots stay
            self.qc = [c[:6] + [s[6]] for c, s in zip(live, self.qc)]

    def step(self):
        p = self.p
        if self.orig is None or 2.0 * _norm(self._wrap(self.orig - self.y[0])).max() > p["nl_pad"]:
            self.rebuild()
        got = self.terms()
        if p["qa_on"]:
            self._finish()
        F = sum(f for f, _ in got.values())
        dt = p["dt"]
        half = dt * dt / 2.0
        y = self.y
        if self.t == 0.0:
            y[2] = F * half
        u = _philox(self.key, self.step_no, self.n)
        tiny = 2.0 ** -32
        r1, r2 = np.sqrt(-2.0 * np.log(u[0] + tiny)), np.sqrt(-2.0 * np.log(u[2] + tiny))
        nz = np.stack([r1 * np.cos(2 * math.pi * u[1]), r1 * np.sin(2 * math.pi * u[1]),
                       r2 * np.cos(2 * math.pi * u[3])], axis=1)
        f = F - p["gamma"] / dt * y[1]
        y[1] = y[1] + math.sqrt(2.0 * p["temperature"] * p["gamma"] * dt) * dt * nz
        err = y[2] - half * f
        co = [np.float32(3) / np.float32(16), np.float32(251) / np.float32(360), np.float32(1),
              np.float32(11) / np.float32(18), np.float32(1) / np.float32(6),
              np.float32(1) / np.float32(60)]
        y = [yk - float(ck) * err for yk, ck in zip(y, co)]
        self.y = [sum(math.comb(j, k) * y[j] for j in range(k, 6)) for k in range(6)]
        self.t += dt
        self.step_no += 1
        return sum(v for _, v in got.values())
