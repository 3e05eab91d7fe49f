"""Results read back through pinned memory: every accessor on systems whose
size is not a multiple of the fetch's workgroup, on systems of a batch behind
others, in both precisions, against each other and the oracle; and an overflow
raised on the device reported by the next call and by every later one."""
import numpy as np
import pytest

from oracle_ffi import Oracle
from pas_cg_amd import model as M
from pas_cg_amd import pcg as G
from pas_cg_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 21, 22, 341, 342, 700])
@pytest.mark.parametrize("precision", [G.FP64, G.MIXED], ids=["fp64", "mixed"])
def test_accessors_agree(n, precision):
    p = W.base_params()
    m = M.synthetic_protein(n, M.job_seed(n))
    y1 = np.random.default_rng(n).normal(scale=1e-3, size=(n, 3))
    o = Oracle(p, m, seed=1)
    o.set_y(1, y1)
    o.set_noise_scale(0.0)
    c = G.Context(p, m, precision=precision, seed=1)
    c.set(1, y1)
    c.set_noise_scale(0.0)
    c.step(1)
    o.step(1)
    for which, ref in ((0, o.r()), (1, o.y(1)), (6, o.F())):
        got = c.get(which)
        np.testing.assert_array_equal(got, c.get3(which).T)
        if precision == G.FP64:
            assert np.abs(got - ref).max() <= 1e-12 * max(np.abs(ref).max(), 1e-300), which
    np.testing.assert_array_equal(c.get(7), c.get3(7).T)
    F, V = c.eval_term("tether")
    F3, V3 = c.eval_term3("tether")
    np.testing.assert_allclose(F, F3.T, rtol=0, atol=1e-5 * max(np.abs(F).max(), 1e-300))
    assert abs(V - V3) <= 1e-12 * abs(V)
    assert V == pytest.approx(o.eval_term("tether")[1], rel=1e-5, abs=1e-12)
    # what is set comes back, and only where it was set
    b = G.Batch(p, [M.synthetic_protein(5, 3), m, M.synthetic_protein(9, 4)], precision=precision)
    rng = np.random.default_rng(n + 1)
    for which in range(6):
        x = rng.normal(size=(n, 3))
        before = b.get(0, which), b.get(2, which)
        b.set(1, which, x)
        np.testing.assert_array_equal(b.get(1, which), x)
        np.testing.assert_array_equal(b.get(0, which), before[0])
        np.testing.assert_array_equal(b.get(2, which), before[1])
        c.set(which, x)
        np.testing.assert_array_equal(c.get3(which).T, x)
    b.close()
    c.close()


def test_overflow_is_reported_and_stays():
    """Every residue within reach of every other: the NL outgrows 1200 pairs a
    residue."""
    n = 2600
    p = W.base_params()
    m = M.synthetic_protein(60, 5)
    m = M.replicate(m, 1, 100.0, 1)
    idx = np.arange(n) % 60
    big = {"n": n, "pos": m["pos"][idx] * 0.2 + np.random.default_rng(1).normal(scale=0.3, size=(n, 3)),
           "atype": m["atype"][idx], "chain": np.zeros(n, np.int32),
           "seq": np.arange(n, dtype=np.int32), "cell": np.zeros(3)}
    big["orig_pos"] = big["pos"].copy()
    for k, w in (("teth", 2), ("ang", 3), ("dih", 4), ("cont", 2)):
        big[k] = np.zeros((0, w), np.int32)
    for k in ("ang_has", "dih_has"):
        big[k] = np.zeros(0, np.uint8)
    for k in ("ang_theta", "dih_phi", "cont_len"):
        big[k] = np.zeros(0)
    big["cont_type"] = np.zeros(0, np.int32)
    p.update(nl_cutoff=30.0, rep_cutoff=0.01)
    c = G.Context(p, M.empty_tips(big), seed=1)
    c.step_form(G.FORM_STAGES)
    for _ in range(2):
        with pytest.raises(G.PcgError):
            c.step(1)
    with pytest.raises(G.PcgError):
        c.step(0)
    c.close()


@pytest.mark.parametrize("n", [4999, 5000, 32767, 32768])
@pytest.mark.parametrize("precision", [G.FP64, G.MIXED], ids=["fp64", "mixed"])
def test_large_results(n, precision):
    """Sizes on both sides of the lines between the fetch's forms: what is set
    comes back bit for bit, and the forces of one tethered pair in the last
    residues only there."""
    p = W.base_params()
    side = int(np.ceil(n ** (1 / 3)))
    pos = np.stack(np.unravel_index(np.arange(n), (side,) * 3), axis=1) * 8.0
    pos[n - 1] = pos[n - 2] + [0.0, 0.0, 0.9]
    m = {"n": n, "pos": pos, "orig_pos": pos * 0.5, "atype": np.zeros(n, np.uint8),
         "chain": np.zeros(n, np.int32), "seq": np.arange(n, dtype=np.int32), "cell": np.zeros(3),
         "teth": np.array([[n - 2, n - 1]], np.int32), "ang": np.zeros((0, 3), np.int32),
         "dih": np.zeros((0, 4), np.int32), "cont": np.zeros((0, 2), np.int32),
         "ang_has": np.zeros(0, np.uint8), "dih_has": np.zeros(0, np.uint8),
         "ang_theta": np.zeros(0), "dih_phi": np.zeros(0), "cont_len": np.zeros(0),
         "cont_type": np.zeros(0, np.int32)}
    c = G.Context(p, M.empty_tips(m), precision=precision, seed=1)
    rng = np.random.default_rng(n)
    for which in (1, 5):
        x = rng.normal(size=(n, 3))
        c.set(which, x)
        np.testing.assert_array_equal(c.get(which), x)
        np.testing.assert_array_equal(c.get3(which).T, x)
    c.eval_term("tether")
    F = c.get(6)
    np.testing.assert_array_equal(F, c.get3(6).T)
    assert not F[:n - 2].any()
    dr = 0.9 - 0.45
    want = min(dr * (p["tether_H1"] + 2 * p["tether_H2"] * dr * dr), 1e3)  # the harmonic's limit
    np.testing.assert_allclose(F[n - 2:, 2], [want, -want], rtol=1e-6)
    np.testing.assert_array_equal(F, c.eval_term3("tether")[0].T)
    c.close()
