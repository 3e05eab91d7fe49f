"""A step of the stage kernels against the oracle: the lists written by the
rows of the rebuild, and the terms by 64-item chunks, at the sizes where a
chunk's last residues reach into the next one, with every bonded term in its
chain-local and its general form, and several systems beside each other."""
import numpy as np
import pytest

from oracle_ffi import Oracle
from pas_cg_amd import model as M
from pas_cg_amd import params as P
from pas_cg_amd import pcg as G
from pas_cg_amd import workloads as W

pytestmark = pytest.mark.gpu

A = P.ANGSTROM
FULL = W.full_params()


def protein(n, seed=31, heur=0.0):
    m = M.synthetic_protein(n, M.job_seed(seed), heuristic_frac=heur)
    m["pos"] = m["pos"] + np.random.default_rng(seed).normal(scale=0.2 * A, size=(n, 3))
    return m


def crossed(n):
    """One tether that is not between neighbours: no chain-local items."""
    m = protein(n)
    m["teth"] = np.concatenate([m["teth"], [[3, 9]]]).astype(np.int32)
    return m


def crowded(n):
    """Every later residue a native partner of residue 1 (more than 64)."""
    m = protein(n)
    j = np.arange(4, n)
    pair = np.stack([np.ones_like(j), j], axis=1).astype(np.int32)
    d = np.linalg.norm(m["pos"][pair[:, 0]] - m["pos"][pair[:, 1]], axis=1)
    m["cont"], m["cont_len"] = pair, d
    m["cont_type"] = np.zeros(len(pair), np.int32)
    return m


NO_QA = {"qa_on": 0, "pid_on": 1}
CASES = [(f"{k}-{n}", over, protein(n, heur=0.5 if k == "heur" else 0.0))
         for k, over in (("full", {}), ("noqa", NO_QA), ("heur", {}))
         for n in (3, 5, 63, 64, 65, 66, 67, 128, 131)]
CASES += [("simple dihedral", {"nat_dih_variant": 1}, protein(130)),
          ("relative DH", {**NO_QA, "dh_variant": 1}, protein(130)),
          ("four", {"qa_include4": 0, "pid_include4": 1, "pid_on": 1}, protein(130)),
          ("no list", {"qa_on": 0, "pid_on": 0, "dh_on": 0, "pauli_on": 0, "nat_cont_on": 0},
           protein(130)),
          ("bonded off", {"tether_on": 0, "nat_ang_on": 0, "heur_ang_on": 0, "chir_on": 0},
           protein(130)),
          ("no Langevin", {"lang_on": 0}, protein(65)),
          ("crossed", {}, crossed(130)), ("crowded", {}, crowded(130))]


def stages(over, m, prec=G.FP64):
    c = G.Context(dict(FULL, **over), m, precision=prec, noise=G.PHILOX, seed=3)
    c.step_form(G.FORM_STAGES)
    c.set_noise_scale(0.0)
    return c


@pytest.mark.parametrize("over,m", [c[1:] for c in CASES], ids=[c[0] for c in CASES])
def test_lists_and_trajectory_equal_the_oracles(over, m):
    o, c = Oracle(dict(FULL, **over), m, seed=3), stages(over, m)
    o.fix_nl()
    c.fix_nl()
    for kind in (0, 1, 2, 3, 4, 5):
        ours, ref = c.list(kind), o.list(kind)
        np.testing.assert_array_equal(np.stack(ours[:2]), np.stack(ref[:2]), err_msg=str(kind))
    c.close()
    o, c = Oracle(dict(FULL, **over), m, seed=3), stages(over, m)
    o.set_noise_scale(0.0)
    tr = o.step(30)
    c.step(30)
    # the tolerance of the other FP64 trajectories
    assert np.abs(c.get(0) - o.r()).max() < 1e-8
    assert abs(c.energy()[0] - tr[-1]) <= 1e-8 * max(abs(tr[-1]), 1.0)
    assert c.nl_rebuilds() == o.nl_rebuilds()
    c.close()


def test_a_batch_of_stage_systems():
    # one system too large for the persistent kernel takes the batch to the
    # stage kernels; waves of the residue kernels then span several systems
    large = M.replicate(protein(41, 34), 100, 300.0 * A, 34)
    models = [protein(5, 33), protein(65, 32), large, protein(3, 35), protein(130, 36)]
    p = dict(FULL)
    b = G.Batch(p, models, seeds=[3, 4, 5, 6, 7], precision=G.FP64)
    b.set_noise_scale(0.0)
    b.run(6)
    for s, m in enumerate(models):
        o = Oracle(p, m, seed=3 + s)
        o.set_noise_scale(0.0)
        tr = o.step(6)
        assert np.abs(b.get(s, 0) - o.r()).max() < 1e-8, s
        assert abs(b.energy(s)[0] - tr[-1]) <= 1e-8 * max(abs(tr[-1]), 1.0), s
        assert b.sizes(s)["rebuilds"] == o.nl_rebuilds(), s
    b.close()


@pytest.mark.parametrize("prec,tol", [(G.FP64, 1e-9), (G.MIXED, 1e-5)], ids=["fp64", "mixed"])
def test_forces_of_steps_without_langevin(prec, tol):
    """A step that does not integrate leaves its forces where they are read, of
    a plain context, of a batch on the stage kernels, and in a saved state."""
    p = dict(FULL, lang_on=0)
    m = protein(130)
    o = Oracle(p, m, seed=3)
    o.step(1)
    F = o.F()
    c = stages({"lang_on": 0}, m, prec)
    c.step(1)
    err = float(np.abs(c.get(6) - F).max())
    assert err <= tol * float(np.abs(F).max())
    np.testing.assert_array_equal(c.get(6), c.get3(6).T)
    d = stages({"lang_on": 0}, m, prec)
    d.restore(c.checkpoint())
    np.testing.assert_array_equal(d.get(6), c.get(6))
    c.close()
    d.close()
    large = M.replicate(protein(41, 34), 100, 300.0 * A, 34)
    b = G.Batch(p, [large, m], seeds=[3, 3], precision=prec)
    b.run(1)
    err = float(np.abs(b.get(1, 6) - F).max())
    assert err <= tol * float(np.abs(F).max())
    b.close()


@pytest.mark.parametrize("qa_on", [1, 0])
def test_launches_of_a_batch_on_the_stage_kernels(qa_on):
    # cells (two), rows, their scan, rows, terms, QA finish, Langevin
    large = M.replicate(protein(41, 34), 100, 300.0 * A, 34)
    b = G.Batch(dict(FULL, qa_on=qa_on), [large], precision=G.MIXED)
    b.run(3)
    assert b.last_ms()[1] == 3 * (7 + qa_on)
    b.close()


def test_forces_outside_a_step_are_the_arrays_forces():
    # mixed precision accumulates in FP64: what an evaluation leaves, what a
    # reader gets and what an integration takes are the same FP32 forces
    c = stages({}, protein(130), prec=G.MIXED)
    c.fix_nl()
    c.prepare_nh()
    c.eval_forces()
    F = c.get(6)
    np.testing.assert_array_equal(F, F.astype(np.float32))
    f, _ = c.eval_term("tether")
    np.testing.assert_array_equal(c.get(6), f)
    np.testing.assert_array_equal(f, f.astype(np.float32))
    c.close()


@pytest.mark.parametrize("copies,side,steps", [(1, 300.0, 20), (100, 150.0, 6), (150, 170.0, 6)])
def test_qa_contacts_form_break_and_are_compressed(copies, side, steps):
    # contacts that break within a few steps: in the first case the list is
    # compressed on the way, in the others a step forms and breaks hundreds of
    # contacts, in the last more than the finish stages in its LDS
    over = {"qa_phase_dur": 0.02, "nat_cont_on": 0, "temperature": 3.0}
    m = M.replicate(protein(41, 34), copies, side * A, 34)
    o, c = Oracle(dict(FULL, **over), m, seed=3), stages(over, m)
    o.set_noise_scale(0.0)
    for _ in range(steps):
        o.step(1)
        c.step(1)
        sync, num = c.qa_state()
        assert num == o.num_qa_contacts()
        np.testing.assert_array_equal(sync, o.sync())
    ours, ref = c.list(6), o.list(6)
    np.testing.assert_array_equal(np.stack(ours[:2]), np.stack(ref[:2]))
    assert np.abs(c.get(0) - o.r()).max() < 1e-8
    c.close()


@pytest.mark.parametrize("copies,side", [(20, 70.0), (60, 110.0)])
def test_most_qa_contacts_break_in_one_step(copies, side):
    # the positions grow by a factor of two: nearly all contacts break at once,
    # in the first case just as many as the finish keeps in its LDS, in the
    # second more; and form again at half the size
    over = {"qa_phase_dur": 0.02, "nat_cont_on": 0, "temperature": 3.0}
    m = M.replicate(protein(41, 34), copies, side * A, 34)
    o, c = Oracle(dict(FULL, **over), m, seed=3), stages(over, m)
    o.set_noise_scale(0.0)
    o.step(4)
    c.step(4)
    for grow in (2.0, 0.5, 1.0):
        r = o.r() * grow
        o.set_r(r)
        c.set(0, r)
        o.fix_nl()  # (a context's step looks at what its own steps moved)
        c.fix_nl()
        before = o.num_qa_contacts()
        o.step(1)
        c.step(1)
        sync, num = c.qa_state()
        assert num == o.num_qa_contacts()
        np.testing.assert_array_equal(sync, o.sync())
        ours, ref = c.list(6), o.list(6)
        np.testing.assert_array_equal(np.stack(ours[:2]), np.stack(ref[:2]))
        ours, ref = c.list(5), o.list(5)
        np.testing.assert_array_equal(np.stack(ours[:2]), np.stack(ref[:2]))
        np.testing.assert_array_equal(ours[3] != 0, ref[3] != 0)
        if grow > 1.0:
            assert (before > 512) == (copies == 60)
    c.close()
