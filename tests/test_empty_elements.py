"""Elements of no sites (accepted where the shortest allowed length is 0)
have no likelihood: NaN, at their own place in the results, whatever an earlier
call of the engine left in the block that results come back in."""
import numpy as np
import pytest

from phyloacc_amd import engine as E
from phyloacc_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [E.PA_FP64, E.PA_FP32])
def test_no_sites(require_gpu, prec):
    w = synth.make_gt_workload(seed=8, n_elements=5, S=6)
    sizes = w.sizes.copy()
    sizes[[1, 4]] = 0
    eng = E.Engine.from_workload(w, E.default_options(min_len=0))
    own, st = eng.add_elements_with_trees(w.align, w.starts, sizes, w.children())
    ids, st2 = eng.add_elements(w.align, w.starts, sizes)
    assert (st == E.PA_ELEM_OK).all() and (st2 == E.PA_ELEM_OK).all()
    n, empty = len(ids), np.array([1, 4])
    full = np.setdiff1d(np.arange(n), empty)
    Z, rates, L = np.ones((n, eng.N), np.int32), np.tile([0.4, 2.0], (n, 1)), w.lengths()
    lens, piA = sizes.astype(np.int32), np.full(n, 0.2)
    sel = np.tile([-1.5, 1.0, 0.7], (n, 1))
    calls = [lambda k: eng.loglik(ids[k], Z[k], rates[k], prec), lambda k: eng.loglik_gbgc(ids[k], Z[k], Z[k], sel[k], prec),
             lambda k: eng.loglik_lengths(own[k], L[k], prec), lambda k: eng.loglik_lengths_pi(own[k], L[k], piA[k], prec),
             lambda k: np.stack(eng.loglik_lengths_split(own[k], L[k], lens[k], lens[k] // 2, precision=prec), 1)]
    for call in calls:
        alone = call(full)
        assert np.isfinite(alone).all()
        got = call(np.arange(n))
        assert np.isnan(got[empty]).all()
        np.testing.assert_array_equal(got[full], alone)
        assert np.isnan(call(empty)).all()
