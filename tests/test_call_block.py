"""The blocks that a likelihood call's inputs, results and device-only
eigensystems live in are kept between calls and grow when a call needs more.
Calls of every kind and size in turn on one engine, each against the same call
on an engine of its own: the same bits."""
import numpy as np
import pytest

from phyloacc_amd import engine as E
from phyloacc_amd import synth

pytestmark = pytest.mark.gpu


def _make():
    w = synth.make_gt_workload(seed=3, n_elements=12, S=9)
    eng = E.Engine.from_workload(w, E.default_options(min_len=1))
    ids, st = eng.add_elements_with_trees(w.align, w.starts, w.sizes, w.children())
    sp, st2 = eng.add_elements(w.align, w.starts, w.sizes)
    assert (st == E.PA_ELEM_OK).all() and (st2 == E.PA_ELEM_OK).all()
    return w, eng, ids, sp


def _call(kind, n, w, eng, ids, sp):
    rng = np.random.default_rng(n)
    k = np.arange(n) % len(ids)
    L, piA = w.lengths()[k], rng.uniform(0.2, 0.3, n)
    Z, B = rng.integers(0, 3, (n, eng.N)).astype(np.int32), rng.integers(0, 2, (n, eng.N)).astype(np.int32)
    lens = w.sizes[k].astype(np.int32)
    if kind == "loglik":
        return eng.loglik(sp[k], Z, np.tile([0.4, 2.0], (n, 1)))
    if kind == "gbgc":
        return eng.loglik_gbgc(sp[k], Z, B, np.tile([-1.5, 1.0, 0.7], (n, 1)))
    if kind == "lengths":
        return eng.loglik_lengths(ids[k], L)
    if kind == "pi":
        return eng.loglik_lengths_pi(ids[k], L, piA)
    return np.concatenate(eng.loglik_lengths_split(ids[k], L, lens, lens // 2, piA=piA))


@pytest.mark.parametrize("seed", [1, 2])
def test_calls_in_any_order(require_gpu, seed):
    shared = _make()
    rng = np.random.default_rng(seed)
    sizes = {"gbgc": (1, 3, 500), "loglik": (1, 40, 3000), "lengths": (2, 700), "pi": (1, 20, 900), "split": (1, 30, 600)}
    calls = [(kind, n) for kind, ns in sizes.items() for n in ns]
    for i in rng.permutation(len(calls)):
        kind, n = calls[i]
        got = _call(kind, n, *shared)
        fresh = _make()
        np.testing.assert_array_equal(got, _call(kind, n, *fresh), err_msg=f"{kind} {n}")
        fresh[1].close()
    shared[1].release_scratch()
    got = _call("gbgc", 3, *shared)
    fresh = _make()
    np.testing.assert_array_equal(got, _call("gbgc", 3, *fresh))
