"""The plain context's two step forms (pcg_step_form): the stage kernels and
the persistent single-system kernel take the same FP64 trajectory (noise
off: the forms sum forces in different orders, so they agree to rounding,
not bits); the persistent form equals a one-system batch; switching forms
mid-run rebuilds the lists and stays on the trajectory; ineligible systems
keep the stage form."""
import numpy as np
import pytest

from oracle_ffi import Oracle
from pas_cg_amd import model as M
from pas_cg_amd import params as P
from pas_cg_amd import pcg as G
from pas_cg_amd import workloads as W

pytestmark = pytest.mark.gpu


def _prm(**kw):
    p = P.default_params()
    p.update(chir_on=1, qa_on=0, pid_on=0)
    p.update(kw)
    return p


def _ctx(prm, m, form, seed=11):
    c = G.Context(prm, m, precision=G.FP64, noise=G.PHILOX, seed=seed, philox_seed=5)
    c.set_noise_scale(0.0)
    assert c.step_form(form) == (form if form else G.FORM_PERSISTENT)
    return c


def test_forms_follow_the_same_trajectory():
    m = M.synthetic_protein(150, M.job_seed(21))
    prm = _prm()
    a = _ctx(prm, m, G.FORM_STAGES)
    b = _ctx(prm, m, G.FORM_AUTO)
    for _ in range(4):
        a.step(50)
        b.step(50)
        assert np.abs(a.r() - b.r()).max() < 1e-9
        assert abs(a.energy()[0] - b.energy()[0]) <= 1e-9 * abs(a.energy()[0])
        assert a.time() == b.time()
    assert np.abs(a.F() - b.F()).max() <= 1e-9 * np.abs(a.F()).max()
    # switching forms mid-run: each switch rebuilds the lists (QA and PID
    # off, so a rebuild does not change the forces)
    b.step_form(G.FORM_STAGES)
    b.step(30)
    b.step_form(G.FORM_PERSISTENT)
    b.step(30)
    a.step(60)
    assert np.abs(a.r() - b.r()).max() < 1e-9
    a.close()
    b.close()


def test_persistent_form_equals_a_one_system_batch():
    m = M.synthetic_protein(120, M.job_seed(23))
    prm = _prm(qa_on=1)
    c = G.Context(prm, m, precision=G.FP64, noise=G.PHILOX, seed=4, philox_seed=9)
    assert c.step_form(G.FORM_AUTO) == G.FORM_PERSISTENT
    b = G.Batch(prm, [m], precision=G.FP64, philox_seed=9, seeds=[4])
    c.step(300)
    b.run(300)
    b.sync()
    assert np.abs(c.r() - b.get(0, 0)).max() < 1e-8
    assert c.time()[1] == 300
    c.close()
    b.close()


def test_ineligible_contexts_keep_the_stages():
    m = M.synthetic_protein(60, M.job_seed(25))
    c = G.Context(_prm(), m, precision=G.FP64, noise=G.RAN2, seed=3)
    assert c.step_form(G.FORM_AUTO) == G.FORM_STAGES
    with pytest.raises(G.PcgError):
        c.step_form(G.FORM_PERSISTENT)
    c.close()
    prm = _prm()
    P.set_solid_walls(prm, m["pos"].min(axis=0) - 1.0, m["pos"].max(axis=0) + 1.0)
    c = G.Context(prm, m, precision=G.FP64, noise=G.PHILOX, seed=3)
    assert c.step_form(G.FORM_AUTO) == G.FORM_STAGES
    c.close()


@pytest.mark.parametrize("qa_on,limit", [(1, 700), (0, 900)])
def test_large_contexts_take_the_stages(qa_on, limit):
    m = M.synthetic_protein(limit, M.job_seed(27))
    prm = _prm(qa_on=qa_on)
    auto = G.Context(prm, m, precision=G.FP64, noise=G.PHILOX, seed=11, philox_seed=5)
    auto.set_noise_scale(0.0)
    assert auto.step_form(G.FORM_AUTO) == G.FORM_STAGES
    pers = _ctx(prm, m, G.FORM_PERSISTENT)
    auto.step(40)
    pers.step(40)
    assert np.abs(auto.r() - pers.r()).max() < 1e-9
    assert abs(auto.energy()[0] - pers.energy()[0]) <= 1e-9 * abs(auto.energy()[0])
    auto.close()
    pers.close()
    small = M.synthetic_protein(limit - 1, M.job_seed(28))
    _ctx(prm, small, G.FORM_AUTO).close()


@pytest.mark.parametrize("stage_step", [False, True], ids=["fresh", "after stages"])
@pytest.mark.parametrize("qa_on", [1, 0], ids=["qa", "no qa"])
@pytest.mark.parametrize("prec,eF,eV", [(G.FP64, 1e-9, 1e-9), (G.MIXED, 1e-5, 1e-6)],
                         ids=["fp64", "mixed"])
def test_per_term_calls_on_the_persistent_lists(prec, eF, eV, qa_on, stage_step):
    """The terms one by one and together, on the lists the persistent kernel
    left, in a context that never built any in the stage form and in one whose
    stage lists are of other positions."""
    prm = dict(W.full_params(), qa_on=qa_on)
    m = M.synthetic_protein(150, M.job_seed(29), heuristic_frac=0.3)
    rng = np.random.default_rng(29)
    m["pos"] = m["pos"] + rng.normal(scale=0.2 * P.ANGSTROM, size=(150, 3))
    o = Oracle(prm, m, seed=4)
    c = G.Context(prm, m, precision=prec, noise=G.PHILOX, seed=4)
    o.set_noise_scale(0.0)
    c.set_noise_scale(0.0)
    if stage_step:
        c.step_form(G.FORM_STAGES)
        o.step(1)
        c.step(1)
        r = o.r()
        r = r[::-1] + rng.normal(scale=0.1 * P.ANGSTROM, size=r.shape)  # other pairs are near
        o.set_r(r)
        c.set(0, r)
        o.fix_nl()
    c.step_form(G.FORM_PERSISTENT)
    o.step(1)
    c.step(1)
    # (both on the same positions: mixed steps round)
    c.set(0, o.r())
    o.prepare_nh()
    c.prepare_nh()
    for term, on in W.term_enabled(prm).items():
        if not on:
            continue
        F, V = c.eval_term(term)
        Fo, Vo = o.eval_term(term)
        err = float(np.abs(F - Fo).max())
        assert err <= eF * max(float(np.abs(Fo).max()), 1e-12), term
        assert abs(V - Vo) <= eV * max(abs(Vo), 1e-12), term
    c.eval_forces()
    o.eval_forces()
    err = float(np.abs(c.get(6) - o.F()).max())
    assert err <= eF * float(np.abs(o.F()).max())
    if qa_on:
        c.qa_finish()
        o.qa_finish()
        sync, num = c.qa_state()
        assert num == o.num_qa_contacts()
        np.testing.assert_array_equal(sync, o.sync())
    c.close()
