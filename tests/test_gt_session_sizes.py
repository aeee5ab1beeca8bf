"""Height moves on resident partials at the sizes where a move's list of
steps changes shape: one internal node below a word of 64 positions, one
above it, and a third word; short elements beside ones of several blocks of
64 patterns."""
import numpy as np
import pytest

from phyloacc_amd import engine as E
from test_gt_branch import SEED, _gt_workload, _species, _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,prec", [(3, E.PA_FP32), (65, E.PA_FP32), (66, E.PA_FP64), (130, E.PA_FP32)])
def test_session_moves_equal_the_host_moves(require_gpu, S, prec):
    """Every internal node twice, in random order.  A session's moves prune a
    path and the stale nodes beside it; the host moves score every proposal in
    full.  Same decisions and heights, and log-likelihoods that differ by
    summation at most (both sum the same terms in FP64: 1e-12)."""
    w = _gt_workload(seed=40 + S, n=4, S=S)
    eng = E.Engine.from_workload(w, E.default_options(min_len=1, seed=SEED))
    ids, st = eng.add_elements_with_trees(w.align, w.starts, w.sizes, w.children())
    assert (st == E.PA_ELEM_OK).all()
    sp, _ = _species(w)
    N, n = w.tree.N, w.C
    ch = np.zeros((n, N, 2), np.int32)
    par = np.zeros((n, N), np.int32)
    H = np.zeros((n, N))
    for c in range(n):
        ch[c], par[c], H[c] = _state(w, c)
    rates = np.stack([w.r1, w.r2], 1)
    lens = np.stack([w.sizes, w.sizes // 3], 1).astype(np.int32)
    f0, f1 = eng.loglik_lengths_split(ids, w.lengths(), lens[:, 0], lens[:, 1], precision=prec)
    ll = np.stack([f0, f1], 1)
    lz = np.full((n, 2), -1e3)           # below any tree's, so that the first moves are accepted
    prior = np.array([E.gt_prior(sp, ch[c], par[c], H[c]) for c in range(n)])
    ses = E.GtSession(eng, sp, ids, ch, par, H, w.Z, rates, ll, lz, prior)
    rng = np.random.default_rng(S)
    total = 0
    for b, v in enumerate(np.concatenate([rng.permutation(np.arange(S, N)) for _ in range(2)])):
        ind = np.full(n, b % 2, np.int32)
        a_host = eng.gt_branch_len(sp, ids, ch, par, H, w.Z, rates, int(v), ind, lens, ll, lz, prior, 0, b, precision=prec)
        a_dev = ses.branch_len(int(v), ind, lens, 0, b, precision=prec)
        np.testing.assert_array_equal(a_dev, a_host, err_msg=f"move {b} of node {v}")
        total += a_host.sum()
    h2, ll2, _, _ = ses.read()
    np.testing.assert_array_equal(h2, H)
    np.testing.assert_allclose(ll2, ll, rtol=1e-12)
    assert total > 0
    ses.close()
