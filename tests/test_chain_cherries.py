"""Chains on trees whose internal nodes take more than one wave to set up: a
node's cherry bit is written by one wave of the workgroup and read by others
when the sampler's steps are built, so both must be on their own side of a
barrier.  (A cherry taken for a stored node is drawn from a partial that no
pass has written.)"""
import numpy as np
import pytest

from chain_checks import oracle_chains
from oracle import oracle_py as O
from phyloacc_amd import engine as E
from test_chain_trees import _workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block", [64, 128, 256])
@pytest.mark.parametrize("shape,S", [("balanced", 128), ("random", 66), ("random", 150)])
def test_cherries_of_large_trees(require_gpu, shape, S, block):
    """Against the oracle: the same chains, and FP64 log-likelihoods to the
    bound of the other chain tests."""
    w = _workload(shape, S, S)
    keep = [1, 4]                                      # 63 and 255 sites
    kw = dict(burnin=1, mcmc=4, adapt_freq=2, min_len=1, compress_patterns=0)
    eng = E.Engine.from_workload(w, E.default_options(**kw))
    ids, st = eng.add_elements(w.align, w.starts[keep], w.sizes[keep])
    assert (st == E.PA_ELEM_OK).all()
    kw.pop("compress_patterns")
    refs = oracle_chains(O.model_from_workload(w), O.default_options(**kw), w, keep)
    r = eng.run_chains(ids, precision=E.PA_FP64, traces=True, block_threads=block)
    assert r["stats"]["block_threads"] == block
    for k in range(len(ids)):
        for ms in range(3):
            np.testing.assert_array_equal(r["Z"][k, ms], refs[k][ms]["Z"])
            np.testing.assert_allclose(r["loglik"][k, ms], refs[k][ms]["loglik"], rtol=1e-9)
