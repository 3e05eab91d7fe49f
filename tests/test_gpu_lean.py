"""The persistent kernel's lean form leaves out terms the host has ruled out
for a batch. Each case here turns on one thing that form does not carry (or
that it must still carry), alone, and the batch must follow the oracle
(noise off, FP64, the tolerance of the other batch trajectories)."""
import numpy as np
import pytest

from oracle_ffi import Oracle
from pas_cg_amd import model as M
from pas_cg_amd import params as P
from pas_cg_amd import pcg as G
from pas_cg_amd import workloads as W

pytestmark = pytest.mark.gpu

A = P.ANGSTROM


def protein(n=64, seed=31, heur=0.0, ss=0):
    m = M.synthetic_protein(n, M.job_seed(seed), heuristic_frac=heur)
    rng = np.random.default_rng(seed)
    m["pos"] = m["pos"] + rng.normal(scale=0.2 * A, size=m["pos"].shape)
    return M.add_disulfides(m, ss) if ss else m


CASES = {
    "lean": ({}, {}),
    "lean without QA": ({"qa_on": 0, "pid_on": 0}, {}),
    "heuristic angles and dihedrals": ({}, {"heur": 0.5}),
    "simple dihedral": ({"nat_dih_variant": 1}, {}),
    "relative DH": ({"qa_on": 0, "pid_on": 0, "dh_variant": 1}, {}),
    "PID without QA": ({"qa_on": 0, "pid_on": 1}, {}),
    "PID pairs four apart": ({"qa_include4": 0, "pid_include4": 1, "pid_on": 1}, {}),
    "QA takes every PID pair": ({"qa_include4": 0, "pid_include4": 0, "pid_on": 1}, {}),
    "disulfide contacts": ({"nc_ss_kind": 2}, {"ss": 3}),
    "disulfide kind without such a contact": ({"nc_ss_kind": 2}, {}),
    "no list needed": ({"qa_on": 0, "pid_on": 0, "dh_on": 0, "pauli_on": 0}, {}),
    "no Langevin": ({"lang_on": 0}, {}),
}


@pytest.mark.parametrize("name", list(CASES))
def test_each_feature_follows_oracle(name):
    over, mk = CASES[name]
    p = W.full_params()
    p.update(over)
    # one system alone, and beside others of other sizes (one of 1 residue
    # past a wave, one of a few residues)
    models = [protein(**mk), protein(n=65, seed=32, **mk), protein(n=5, seed=33)]
    b = G.Batch(p, models, seeds=[3, 4, 5], precision=G.FP64, steps_per_launch=23, block=128)
    b.set_noise_scale(0.0)
    b.run(60)
    for s, m in enumerate(models):
        o = Oracle(p, m, seed=3 + s)
        o.set_noise_scale(0.0)
        tr = o.step(60)
        assert np.abs(b.get(s, 0) - o.r()).max() < 1e-8, (name, s)
        assert abs(b.energy(s)[0] - tr[-1]) <= 1e-8 * max(abs(tr[-1]), 1.0), (name, s)
        assert b.sizes(s)["rebuilds"] == o.nl_rebuilds(), (name, s)
    b.close()
