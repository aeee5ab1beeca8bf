"""Chains on trees of every shape against the oracle: the pruning pass walks a
list of steps built from the tree (a node after its children, the larger
subtree first), the sampler another, and the Z update the tree's levels, so
the shapes here are those at which such lists turn: two and three leaves, a
caterpillar, a balanced tree, more than 64 internal nodes, and pattern counts
on both sides of a wave and of a workgroup."""
import numpy as np
import pytest

from chain_checks import oracle_chains
from oracle import oracle_py as O
from phyloacc_amd import engine as E
from phyloacc_amd import synth

# sites per element, one pattern each: around 64 (a wave) and 256 (the default workgroup of a small batch)
SIZES = [1, 63, 64, 65, 255, 256, 257]


def _caterpillar(S):
    kids = ["sp0", "sp1"]
    t = f"({kids[0]}:0.1,{kids[1]}:0.07)"
    for s in range(2, S):
        t = f"({t}:0.05,sp{s}:0.1)"
    return t + "r;"


def _balanced(S):
    nodes = [f"sp{s}" for s in range(S)]
    while len(nodes) > 1:
        nodes = [f"({a}:0.06,{b}:0.09)" for a, b in zip(nodes[::2], nodes[1::2])]
    return nodes[0] + "r;"


def _workload(shape, S, seed):
    rng = np.random.default_rng(seed)
    pi, Q = synth.gtr(rng)
    if shape == "random":
        text = synth.mod_text(pi, Q, synth.random_tree(S, 0.08, rng))
    else:
        tree = synth.random_tree(S, 0.08, rng)
        tree.newick = _caterpillar(S) if shape == "caterpillar" else _balanced(S)
        text = synth.mod_text(pi, Q, tree)
    t = E.parse_mod(text)
    tree = synth.Tree(S, t["children"], t["parent"], t["dist"], t["names"], "")
    sizes = np.array(SIZES)
    rates = np.where(rng.random((len(sizes), t["N"])) < 0.15, 2.5, 0.4)
    align = synth.simulate(tree, pi, Q, sizes, rates, 0.05, rng)
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)
    return synth.Workload(shape, tree, pi, Q, text, align, sizes, starts, [], [], [], rates, seed)


@pytest.mark.gpu
@pytest.mark.parametrize("ambiguous", [False, True])
@pytest.mark.parametrize("shape,S", [("random", 2), ("random", 3), ("caterpillar", 40), ("balanced", 64), ("random", 90)])
def test_chains_match_the_oracle_on_any_tree(require_gpu, shape, S, ambiguous):
    w = _workload(shape, S, 7 + S)
    rng = np.random.default_rng(S)
    if ambiguous:
        # IUPAC codes here and there, and two leaves missing from every element
        w.align = np.where(rng.random(w.align.shape) < 0.03, rng.choice(list(b"rykmsw"), w.align.shape), w.align).astype(np.uint8)
        if S > 3:
            w.align[[1, 2], 1:] = ord("-")
    kw = dict(burnin=2, mcmc=6, adapt_freq=3, min_len=1, compress_patterns=0)
    eng = E.Engine.from_workload(w, E.default_options(**kw))
    ids, st = eng.add_elements(w.align, w.starts, w.sizes)
    ok = st == E.PA_ELEM_OK
    assert ok.sum() >= len(SIZES) - 1
    ids, idx = ids[ok], np.flatnonzero(ok)
    kw.pop("compress_patterns")
    refs = oracle_chains(O.model_from_workload(w), O.default_options(**kw), w, idx)
    r = eng.run_chains(ids, precision=E.PA_FP64, traces=True)
    for k in range(len(ids)):
        for ms in range(3):
            np.testing.assert_array_equal(r["Z"][k, ms], refs[k][ms]["Z"])
            # FP64 sums over at most 257 sites and 89 nodes: the bound of the other chain tests
            np.testing.assert_allclose(r["loglik"][k, ms], refs[k][ms]["loglik"], rtol=1e-9)
            np.testing.assert_allclose(r["nrate"][k, ms], refs[k][ms]["nrate"], rtol=1e-9)
    f = eng.run_chains(ids, precision=E.PA_FP32, traces=True)
    # the state before the first draw: the same (Z, r), so the difference is the FP32 partials'
    np.testing.assert_allclose(f["loglik"][:, :, 0], r["loglik"][:, :, 0], rtol=1e-6)


@pytest.mark.gpu
def test_split_elements_score_like_whole_ones(require_gpu):
    """A scoring launch takes long elements in parts, each at least a pass of
    the workgroup's 256 patterns: elements just below, at and above one and
    two parts, alone and in a batch, against the oracle (FP64 sums in another
    order: the bound of the other likelihood tests)."""
    w = _workload("random", 40, 3)
    sizes = np.array([255, 256, 257, 511, 513, 1030])
    rng = np.random.default_rng(5)
    w.align = synth.simulate(w.tree, w.pi, w.Q, sizes, np.full((len(sizes), w.tree.N), 0.7), 0.05, rng)
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)
    eng = E.Engine.from_workload(w, E.default_options(compress_patterns=0))
    ids, st = eng.add_elements(w.align, starts, sizes)
    assert (st == E.PA_ELEM_OK).all()
    Z = np.where(rng.random((len(ids), eng.N)) < 0.2, 2, 1).astype(np.int32)
    Z[:, eng.N - 1] = 0
    rates = np.tile([0.4, 2.0], (len(ids), 1))
    m, oo = O.model_from_workload(w), O.default_options()
    ref = np.array([O.Element(m, oo, w.align, starts[k], sizes[k]).loglik(Z[k], 0.4, 2.0) for k in range(len(ids))])
    np.testing.assert_allclose(eng.loglik(ids, Z, rates, E.PA_FP64), ref, rtol=1e-9)
    np.testing.assert_allclose(eng.loglik(ids, Z, rates, E.PA_FP32), ref, rtol=1e-6)
    one = [eng.loglik(ids[k:k + 1], Z[k:k + 1], rates[k:k + 1], E.PA_FP64)[0] for k in range(len(ids))]
    np.testing.assert_allclose(one, ref, rtol=1e-9)
