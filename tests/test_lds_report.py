"""The LDS a likelihood call reports is that of the kernel it launched: a
scoring workgroup holds 16 values a node, a step of 16 bytes an internal node
(and two behind them), the work positions' own eigensystems (36 doubles each;
six under the gBGC model), and about a kilobyte of arguments."""
import numpy as np
import pytest

from phyloacc_amd import engine as E
from phyloacc_amd import synth
from test_gt_branch import SEED, _gt_workload, _species, _state

pytestmark = pytest.mark.gpu
EIG = 36 * 8


def _score(N, rs):
    return 16 * N * rs + 16 * (N // 2 + 2)


@pytest.mark.parametrize("prec,rs", [(E.PA_FP64, 8), (E.PA_FP32, 4)])
def test_scoring_calls(require_gpu, prec, rs):
    w = synth.make_workload(1, seed=4, lengths=[80, 120])
    eng = E.Engine.from_workload(w, E.default_options(min_len=1))
    ids, st = eng.add_elements(w.align, w.starts, w.sizes)
    ids = ids[st == E.PA_ELEM_OK]
    n = len(ids)
    Z = np.ones((n, eng.N), np.int32)
    eng.loglik(ids, Z, np.tile([0.4, 2.0], (n, 1)), prec)
    args = eng.loglik_stats()["lds_bytes"] - _score(eng.N, rs)
    assert 0 < args < 1280
    eng.loglik_gbgc(ids, Z, Z, np.tile([-1.5, 1.0, 0.7], (n, 1)), prec)
    assert eng.loglik_stats()["lds_bytes"] == _score(eng.N, rs) + args + 6 * EIG


@pytest.mark.parametrize("prec,rs", [(E.PA_FP64, 8), (E.PA_FP32, 4)])
def test_gene_tree_calls(require_gpu, prec, rs):
    """Own base frequencies; a history's drawn bases (one byte a thread and
    internal node) on top of a session's layout."""
    w = _gt_workload(seed=3, n=3, S=40)
    eng = E.Engine.from_workload(w, E.default_options(min_len=1, seed=SEED))
    ids, st = eng.add_elements_with_trees(w.align, w.starts, w.sizes, w.children())
    assert (st == E.PA_ELEM_OK).all()
    n, N = w.C, w.tree.N
    eng.loglik_lengths(ids, w.lengths(), prec)
    plain = eng.loglik_stats()["lds_bytes"]
    eng.loglik_lengths_pi(ids, w.lengths(), np.full(n, 0.2), prec)
    assert eng.loglik_stats()["lds_bytes"] == plain + EIG
    ch, par, H = np.zeros((n, N, 2), np.int32), np.zeros((n, N), np.int32), np.zeros((n, N))
    for c in range(n):
        ch[c], par[c], H[c] = _state(w, c)
    sp, _ = _species(w)
    rates = np.stack([w.r1, w.r2], 1)
    lens = np.stack([w.sizes, w.sizes], 1).astype(np.int32)
    ses = E.GtSession(eng, sp, ids, ch, par, H, w.Z, rates, np.zeros((n, 2)), np.zeros((n, 2)), np.zeros(n))
    ses.branch_len(w.tree.S, np.zeros(n, np.int32), lens, 0, 0, precision=prec)
    keep = eng.loglik_stats()["lds_bytes"]
    ses.close()
    eng.gt_sample_history(sp, ids, ch, par, H, w.Z, rates, lens[:, 0], 1, precision=prec)
    st = eng.loglik_stats()
    I = N // 2 + 1
    assert st["lds_bytes"] == keep + 8 * (I + 2) + I * st["block_threads"]
