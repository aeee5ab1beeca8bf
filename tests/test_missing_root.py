"""Elements in which every species is missing (each has gaps at more than the
missing share of the sites, but some sites hold bases): their root is a
missing node, so no site carries information and every log-likelihood is the
oracle's 0.  The patterns' terms are log sum_j pi_j with frequencies that add
to 1 within a few units of the last place, so 500 sites stay below 1e-12."""
import numpy as np
import pytest

from oracle import oracle_py as O
from phyloacc_amd import engine as E
from phyloacc_amd import synth
from test_gt_branch import SEED, _gt_workload, _species, _state

pytestmark = pytest.mark.gpu
ATOL = 1e-12


def _blank(align, start, length, rng):
    """All but a tenth of every species' sites of one element become gaps."""
    for s in range(align.shape[0]):
        align[s, start + rng.permutation(length)[: length - length // 10]] = ord("-")


def _species_workload():
    w = synth.small_workload(S=6, C=3, length=112, seed=3, gap=0.02)
    w.conserve = []
    _blank(w.align, w.starts[1], 112, np.random.default_rng(0))
    return w


@pytest.mark.parametrize("prec", [E.PA_FP64, E.PA_FP32])
def test_species_tree_elements(require_gpu, prec):
    w = _species_workload()
    kw = dict(burnin=2, mcmc=6, adapt_freq=3, min_len=1)
    eng = E.Engine.from_workload(w, E.default_options(**kw))
    ids, st = eng.add_elements(w.align, w.starts, w.sizes)
    assert (st == E.PA_ELEM_OK).all()
    m, oo = O.model_from_workload(w), O.default_options(**kw)
    els = [O.Element(m, oo, w.align, w.starts[i], w.sizes[i]) for i in range(3)]
    Z = np.ones((3, eng.N), np.int32)
    Z[:, eng.N - 1] = 0
    rates = np.tile([0.3, 2.0], (3, 1))
    ref = np.array([e.loglik(Z[k], 0.3, 2.0) for k, e in enumerate(els)])
    assert ref[1] == 0.0 and (ref[[0, 2]] < 0).all()
    rtol = 1e-9 if prec == E.PA_FP64 else 1e-6
    np.testing.assert_allclose(eng.loglik(ids, Z, rates, prec), ref, rtol=rtol, atol=ATOL)
    np.testing.assert_allclose(eng.loglik(ids[1:2], Z[1:2], rates[1:2], prec), 0.0, atol=ATOL)
    sel = np.tile([-1.0, 1.0, 0.5], (3, 1))
    assert abs(eng.loglik_gbgc(ids, Z, Z, sel, prec)[1]) <= ATOL
    r = eng.run_chains(ids, precision=prec, traces=True)
    o = els[1].run(oo)
    for ms in range(3):
        np.testing.assert_allclose(r["loglik"][1, ms], o[ms]["loglik"], atol=ATOL)
        np.testing.assert_array_equal(r["Z"][1, ms], o[ms]["Z"])
        np.testing.assert_allclose(r["nrate"][1, ms], o[ms]["nrate"], rtol=1e-9)


@pytest.mark.parametrize("prec", [E.PA_FP64, E.PA_FP32])
def test_own_tree_elements(require_gpu, prec):
    """Whole elements and site prefixes; then the height moves of a session
    (its first pass stores every node, later ones score paths) and the same
    moves scored in full: equal decisions, and 0 for every accepted one."""
    w = _gt_workload(seed=12, n=4, S=7)
    _blank(w.align, w.starts[2], w.sizes[2], np.random.default_rng(1))
    eng = E.Engine.from_workload(w, E.default_options(min_len=1, seed=SEED))
    ids, st = eng.add_elements_with_trees(w.align, w.starts, w.sizes, w.children())
    assert (st == E.PA_ELEM_OK).all()
    m = O.parse_mod(w.mod_text)[0]
    g = w.genes[2]
    assert abs(O.gt_loglik(m, w.tree.S, g.children, g.seg_gene, g.seg_species, g.seg_len * w.scale, w.Z[2], w.r1[2],
                           w.r2[2], w.align, int(w.starts[2]), int(w.sizes[2]))) <= ATOL
    assert abs(eng.loglik_lengths(ids, w.lengths(), prec)[2]) <= ATOL
    lens = np.stack([w.sizes, w.sizes // 3], 1).astype(np.int32)
    ll = np.stack(eng.loglik_lengths_split(ids, w.lengths(), lens[:, 0], lens[:, 1], precision=prec), 1)
    assert (np.abs(ll[2]) <= ATOL).all() and (ll[[0, 1, 3]] < 0).all()
    sp, _ = _species(w)
    N, n = w.tree.N, w.C
    ch, par, H = np.zeros((n, N, 2), np.int32), np.zeros((n, N), np.int32), np.zeros((n, N))
    for c in range(n):
        ch[c], par[c], H[c] = _state(w, c)
    lz = np.full((n, 2), -1e3)           # below any tree's, so that the first moves are accepted
    prior = np.array([E.gt_prior(sp, ch[c], par[c], H[c]) for c in range(n)])
    rates = np.stack([w.r1, w.r2], 1)
    ses = E.GtSession(eng, sp, ids, ch, par, H, w.Z, rates, ll, lz, prior)
    accepted = 0
    for b, v in enumerate(range(w.tree.S, N)):
        ind = np.full(n, b % 2, np.int32)
        a_host = eng.gt_branch_len(sp, ids, ch, par, H, w.Z, rates, v, ind, lens, ll, lz, prior, 0, b, precision=prec)
        np.testing.assert_array_equal(ses.branch_len(v, ind, lens, 0, b, precision=prec), a_host)
        accepted += a_host[2]
    _, ll2, _, _ = ses.read()
    ses.close()
    assert accepted > 0
    np.testing.assert_allclose(ll2, ll, rtol=1e-12, atol=ATOL)
    assert (np.abs(ll2[2]) <= ATOL).all()
