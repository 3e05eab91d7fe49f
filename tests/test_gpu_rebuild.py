"""The persistent kernel's list rebuild against the oracle's lists, pair for
pair and in order: sizes at the edges of its 64-column chunks, the pairs four
apart that QA or PID leave out, residue numberings other than consecutive,
a periodic cell, and systems whose extent widens the FP32 scan's margins."""
import numpy as np
import pytest

from oracle_ffi import Oracle
from pas_cg_amd import model as M
from pas_cg_amd import params as P
from pas_cg_amd import pcg as G
from pas_cg_amd import workloads as W

pytestmark = pytest.mark.gpu

A = P.ANGSTROM


def protein(n, seed=41):
    m = M.synthetic_protein(n, M.job_seed(seed))
    m["pos"] = m["pos"] + np.random.default_rng(seed).normal(scale=0.2 * A, size=(n, 3))
    return m


def two_chains(n, seq_step=1, swap=False):
    m = protein(n)
    cut = n // 3
    m["chain"] = (np.arange(n) >= cut).astype(np.int32)
    if swap:  # the second chain's index below the first's
        m["chain"] = (1 - m["chain"]).astype(np.int32)
    m["seq"] = np.where(np.arange(n) >= cut, np.arange(n) - cut, np.arange(n)).astype(np.int32) * seq_step
    m["teth"], m["ang"], m["dih"] = M.chain_lists(m["chain"])
    for k in ("ang", "dih"):
        m[k + "_has"] = np.zeros(len(m[k]), np.uint8)
    m["ang_theta"], m["dih_phi"] = np.zeros(len(m["ang"])), np.zeros(len(m["dih"]))
    return m


def stretched(n):
    """A long arc: an extent of hundreds of length units."""
    m = protein(n)
    t = np.arange(n) * (3.8 * A / 900.0)
    m["pos"] = np.stack([900.0 * np.sin(t), 900.0 * np.cos(t), 0.02 * np.arange(n) % 0.6], axis=1) + 5e3
    return m


def in_cell(n):
    m = protein(n)
    side = np.ptp(m["pos"], axis=0).max() + 4.0 * A
    m["cell"] = np.array([side, side, side])
    m["pos"] = m["pos"] + 0.4 * side
    return m


def far_off(n, k, x):
    """Residue k far outside, as a diverged trajectory leaves it."""
    m = protein(n)
    m["pos"] = m["pos"].copy()
    m["pos"][k] = x
    return m


FULL = W.full_params()
NO_QA = dict(FULL, qa_on=0, pid_on=1)
GO = W.base_params()
FOUR = dict(FULL, qa_include4=0, pid_include4=1)
FOUR_DH = dict(FULL, qa_include4=0, pid_include4=0)
WIDE = dict(FULL, nl_cutoff=12.0 * A, dh_cutoff=30.0 * A)
CASES = [(f"{name}-{n}", p, protein(n)) for name, p in (("full", FULL), ("go", GO), ("noqa", NO_QA))
         for n in (2, 4, 5, 63, 64, 65, 127, 128, 129, 193)]
CASES += [("four", FOUR, protein(150)), ("four-dh", FOUR_DH, protein(150)),
          ("wide", WIDE, protein(150)), ("chains", FULL, two_chains(150)),
          ("chains-noqa", NO_QA, two_chains(150)), ("gaps", FULL, two_chains(150, seq_step=2)),
          ("swapped", NO_QA, two_chains(150, swap=True)), ("arc", FULL, stretched(200)),
          ("arc-noqa", NO_QA, stretched(200)), ("cell", FULL, in_cell(150)),
          ("cell-four", FOUR, in_cell(150)), ("long", FULL, protein(900))]
CASES += [(f"off-{k}-{x:g}", FULL, far_off(150, k, x)) for k in (0, 77) for x in (1e5, 1e20, 1e200, np.inf)]
CASES += [("off-noqa", NO_QA, far_off(150, 149, [1e40, 0.0, 0.0])),
          ("reach", dict(FULL, nl_cutoff=1e16, dh_cutoff=1e16), protein(40))]


@pytest.mark.parametrize("prm,m", [c[1:] for c in CASES], ids=[c[0] for c in CASES])
def test_lists_equal_the_oracles(prm, m):
    o = Oracle(prm, m, seed=2)
    o.fix_nl()
    c = G.Context(prm, m, precision=G.MIXED, noise=G.PHILOX, seed=2)
    c.step_form(G.FORM_PERSISTENT)
    c.set_noise_scale(0.0)
    c.step(1)
    for kind in (1, 2, 3, 4):  # native contacts, Pauli, DH, PID
        ours, ref = c.list(kind), o.list(kind)
        np.testing.assert_array_equal(np.stack(ours[:2]), np.stack(ref[:2]), err_msg=str(kind))
        if kind == 4:
            np.testing.assert_array_equal(ours[2], ref[2])
    # QA free pairs: the count of all, and those near enough to become
    # candidates, in the same order with the same distances
    i1, i2, d, _ = o.list(5)
    near = d <= max(prm["qa_lj_r_high"])
    n = c.term_size("qa_cand")
    assert n == int(near.sum()) if prm["qa_on"] else n == 0
    g1, g2, gd, _ = c.list(5)
    assert len(g1) == len(i1)
    np.testing.assert_array_equal(g1[:n], i1[near])
    np.testing.assert_array_equal(g2[:n], i2[near])
    np.testing.assert_array_equal(gd[:n], d[near])
    c.close()
    b = G.Batch(prm, [m], seeds=[2], precision=G.MIXED)
    b.run(1)
    assert b.sizes(0)["nl"] == len(o.list(0)[0])
    b.close()


def test_a_diverged_system_stays_alone():
    """Systems of a batch beside ones with coordinates FP32 cannot hold."""
    ms = [protein(100, 1), far_off(100, 7, np.inf), protein(130, 2), far_off(64, 0, 1e300), protein(90, 3)]
    # the same places (and so the same noise) with ordinary systems between
    calm = [protein(m["n"], 9) if k % 2 else m for k, m in enumerate(ms)]
    b, o = (G.Batch(FULL, x, seeds=[1, 2, 3, 4, 5], precision=G.MIXED) for x in (ms, calm))
    b.run(3)
    o.run(3)
    for k in (0, 2, 4):
        assert b.sizes(k) == o.sizes(k)
        # three steps of mixed forces summed in another order
        np.testing.assert_allclose(b.get(k, 0), o.get(k, 0), rtol=0, atol=1e-9)
    b.close()
    o.close()
