"""The block sizes of a scoring launch: 128 threads from eight elements a CU
on, 64 for short elements in many rounds, 256 otherwise."""
import numpy as np
import pytest

from phyloacc_amd import engine as E
from phyloacc_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [E.PA_FP64, E.PA_FP32])
@pytest.mark.parametrize("per_cu,block", [(8, 128), (65, 64)])
def test_large_calls_equal_small_ones(require_gpu, per_cu, block, prec):
    """One call over many elements against calls of 200, which 256 threads
    score.  Both sum the same FP64 terms of a few hundred patterns in another
    grouping: 1e-12 relative."""
    n = per_cu * 256 + 1                                    # an MI355X has 256 CUs
    lengths = np.random.default_rng(per_cu).integers(1, 130, n)
    w = synth.make_workload(1, seed=9, lengths=[int(x) for x in lengths])
    eng = E.Engine.from_workload(w, E.default_options(min_len=1))
    ids, st = eng.add_elements(w.align, w.starts, w.sizes)
    ids = ids[st == E.PA_ELEM_OK]
    ids = np.resize(ids, n)                                 # filtered ones replaced: the size is the point
    rng = np.random.default_rng(1)
    Z = rng.integers(0, 3, (n, eng.N)).astype(np.int32)
    rates = np.stack([rng.uniform(0.1, 0.9, n), rng.uniform(1.2, 4.0, n)], 1)
    ll = eng.loglik(ids, Z, rates, prec)
    assert eng.loglik_stats()["block_threads"] == block
    for i in list(range(0, n, 200))[:: max(1, n // 4000)]:
        k = slice(i, min(n, i + 200))
        np.testing.assert_allclose(ll[k], eng.loglik(ids[k], Z[k], rates[k], prec), rtol=1e-12)
    assert eng.loglik_stats()["block_threads"] == 256
