"""The block sizes of scoring launches beyond those of plain calls over small
trees: 64 threads only where sixteen such workgroups fit a CU's LDS, calls with
site prefixes at each size (their table of terms lies in front of a
workgroup's stacks and is walked in steps of the block), and lists that mix
whole elements with the parts of long ones.  Each large call against calls of
60 elements, which 256 threads score: the same FP64 terms of up to 3,000
sites in another grouping, 1e-12 relative."""
import numpy as np
import pytest
import torch

from phyloacc_amd import engine as E
from phyloacc_amd import synth

pytestmark = pytest.mark.gpu
RTOL = 1e-12


def _cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


def _engine(S, lengths, own):
    rng = np.random.default_rng(S)
    pi, Q = synth.gtr(rng)
    tree = synth.random_tree(S, 0.08, rng)
    t = E.parse_mod(synth.mod_text(pi, Q, tree))
    sizes = np.asarray(lengths)
    starts = np.concatenate([[0], np.cumsum(sizes)[:-1]]).astype(np.int64)
    align = rng.choice(np.frombuffer(b"acgt-", np.uint8), size=(S, int(sizes.sum())), p=[.24, .24, .24, .24, .04])
    eng = E.Engine(S, t["children"], t["parent"], t["dist"], pi, Q, options=E.default_options(min_len=1, compress_patterns=0))
    if own:
        ids, st = eng.add_elements_with_trees(align, starts, sizes, np.tile(t["children"][None], (len(sizes), 1, 1)))
    else:
        ids, st = eng.add_elements(align, starts, sizes)
    assert (st == E.PA_ELEM_OK).all()
    return eng, ids, sizes.astype(np.int32)


def _check(eng, call, n, block):
    """call(slice) -> log-likelihoods of those rows, [rows] or [rows, 2]."""
    whole = call(slice(0, n))
    assert eng.loglik_stats()["block_threads"] == block
    for i in list(range(0, n, 60))[:: max(1, n // 1500)]:
        k = slice(i, min(n, i + 60))
        np.testing.assert_allclose(whole[k], call(k), rtol=RTOL)
    assert eng.loglik_stats()["block_threads"] == 256


@pytest.mark.parametrize("S,prec,block", [(43, E.PA_FP32, 64), (43, E.PA_FP64, 128), (90, E.PA_FP32, 128), (10, E.PA_FP64, 64)])
def test_sixty_four_threads_where_sixteen_workgroups_fit(require_gpu, S, prec, block):
    eng, ids, _ = _engine(S, np.random.default_rng(S).integers(1, 100, 40), False)
    n = 65 * _cus()
    ids = np.resize(ids, n)
    rng = np.random.default_rng(2)
    Z = rng.integers(0, 3, (n, eng.N)).astype(np.int32)
    rates = np.stack([rng.uniform(0.1, 0.9, n), rng.uniform(1.2, 4.0, n)], 1)
    _check(eng, lambda k: eng.loglik(ids[k], Z[k], rates[k], prec), n, block)


@pytest.mark.parametrize("prec", [E.PA_FP64, E.PA_FP32])
@pytest.mark.parametrize("per_cu,long,block", [(65, 0, 64), (33, 0, 128), (9, 0, 256), (9, 2900, 256)])
def test_site_prefixes(require_gpu, per_cu, long, block, prec):
    """Nine elements of 100 patterns a CU are 112 for each of eight
    workgroups, fewer than the longest element's 199."""
    eng, ids, sizes = _engine(12, list(np.random.default_rng(per_cu).integers(1, 200, 40)) + ([long] if long else []), True)
    n = per_cu * _cus()
    k = np.arange(n) % 40
    if long:
        k[[1, n // 2]] = 40
    rng = np.random.default_rng(3)
    lengths, piA = rng.exponential(0.05, (n, eng.N)), rng.uniform(0.2, 0.3, n)
    l0 = (rng.random(n) * (sizes[k] + 1)).astype(np.int32)
    l1 = (rng.random(n) * (l0 + 1)).astype(np.int32)
    _check(eng, lambda s: np.stack(eng.loglik_lengths_split(ids[k[s]], lengths[s], l0[s], l1[s], piA=piA[s], precision=prec), 1), n, block)


@pytest.mark.parametrize("prec", [E.PA_FP64, E.PA_FP32])
@pytest.mark.parametrize("longs,block", [(3, 128), (600, 256)])
def test_parts_among_whole_elements(require_gpu, longs, block, prec):
    """A few elements of many parts (each ends in a part of its own size)
    among short ones; and enough of them to raise the mean above 600."""
    eng, ids, _ = _engine(12, list(np.random.default_rng(5).integers(30, 200, 40)) + [1024, 2049, 3000], False)
    n = 9 * _cus()
    k = np.arange(n) % 40
    k[:: n // longs][:longs] = 40 + np.arange(len(k[:: n // longs][:longs])) % 3
    rng = np.random.default_rng(4)
    Z = rng.integers(0, 3, (n, eng.N)).astype(np.int32)
    rates = np.stack([rng.uniform(0.1, 0.9, n), rng.uniform(1.2, 4.0, n)], 1)
    _check(eng, lambda s: eng.loglik(ids[k[s]], Z[s], rates[s], prec), n, block)
