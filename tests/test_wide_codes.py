"""Elements whose leaf codes (species x padded patterns) take 4 GiB or more:
a code's offset does not fit 32 bits, so a launch over such arenas goes to
kernels that address a row in 64 bits.  An engine can be told to use them for
any elements; they apply the same operations in the same order, so with 256
threads, the only block size they come in, the results are the same bits, and
otherwise the FP64 sums are of the same terms in another grouping (1e-12)."""
import ctypes as C

import numpy as np
import pytest

from phyloacc_amd import engine as E
from phyloacc_amd import synth
from test_gt_branch import SEED, _gt_workload, _species, _state


def _lib():
    L = E.lib()
    L.pa_wide_codes.argtypes = [C.c_int32, C.c_int64]
    L.pa_engine_force_wide.argtypes = [C.c_void_p, C.c_int32]
    L.pa_engine_force_wide.restype = None
    return L


@pytest.mark.parametrize("S,patterns,wide", [(2, (1 << 31) - 64, 0), (2, 1 << 31, 1), (43, 99882944, 0), (43, 99883008, 1),
                                             (256, (1 << 24) - 64, 0), (256, 1 << 24, 1)])
def test_where_wide_codes_begin(S, patterns, wide):
    assert (S * patterns >= 2 ** 32) == bool(wide)
    assert _lib().pa_wide_codes(S, patterns) == wide


def _both(eng, call):
    L = _lib()
    out = []
    for on in (0, 1):
        L.pa_engine_force_wide(eng._h, on)
        out.append(call())
    L.pa_engine_force_wide(eng._h, 0)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [E.PA_FP64, E.PA_FP32])
@pytest.mark.parametrize("ambiguous", [False, True])
def test_scores(require_gpu, prec, ambiguous):
    """Whole elements, one in parts, and gBGC; a call small enough for 256
    threads and one that takes 128."""
    w = synth.make_workload(1, seed=5, lengths=[60, 63, 64, 65, 255, 256, 257, 3000])
    rng = np.random.default_rng(2)
    if ambiguous:
        w.align = np.where(rng.random(w.align.shape) < 0.03, rng.choice(list(b"rykmsw"), w.align.shape), w.align).astype(np.uint8)
    eng = E.Engine.from_workload(w, E.default_options(min_len=1, compress_patterns=0))
    ids, st = eng.add_elements(w.align, w.starts, w.sizes)
    ids = ids[st == E.PA_ELEM_OK]
    for n in (len(ids), 8 * 256 + 7):
        k = np.resize(ids[:-1], n) if n > len(ids) else ids
        Z, B = rng.integers(0, 3, (n, eng.N)).astype(np.int32), rng.integers(0, 2, (n, eng.N)).astype(np.int32)
        rates, sel = np.tile([0.4, 2.0], (n, 1)), np.tile([-1.5, 1.0, 0.7], (n, 1))
        for call in (lambda: eng.loglik(k, Z, rates, prec), lambda: eng.loglik_gbgc(k, Z, B, sel, prec)):
            a, b = _both(eng, call)
            np.testing.assert_allclose(b, a, rtol=0 if n == len(ids) else 1e-12)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [E.PA_FP64, E.PA_FP32])
def test_gene_tree_moves(require_gpu, prec):
    """Prefixes, a session's height moves, histories and a regraft with its
    candidate scores, on an engine of each kind."""
    w = _gt_workload(seed=21, n=5, S=12)
    sp, _ = _species(w)
    S, N, n = w.tree.S, w.tree.N, w.C
    lens = np.stack([w.sizes, w.sizes // 2], 1).astype(np.int32)
    rates = np.stack([w.r1, w.r2], 1)
    nodes = np.arange(S, N, dtype=np.int32)

    def moves(wide):
        eng = E.Engine.from_workload(w, E.default_options(min_len=1, seed=SEED))
        ids, st = eng.add_elements_with_trees(w.align, w.starts, w.sizes, w.children())
        assert (st == E.PA_ELEM_OK).all()
        _lib().pa_engine_force_wide(eng._h, wide)
        ch, par, H = np.zeros((n, N, 2), np.int32), np.zeros((n, N), np.int32), np.zeros((n, N))
        for c in range(n):
            ch[c], par[c], H[c] = _state(w, c)
        ll = np.stack(eng.loglik_lengths_split(ids, w.lengths(), lens[:, 0], lens[:, 1], precision=prec), 1)
        lz = np.zeros((n, 2))
        prior = np.array([E.gt_prior(sp, ch[c], par[c], H[c]) for c in range(n)])
        ind = np.zeros(n, np.int32)
        ses = E.GtSession(eng, sp, ids, ch, par, H, w.Z, rates, ll, lz, prior)
        acc, _ = ses.sweep(nodes, ind, lens, 1, 1, precision=prec)
        out = [acc] + list(ses.read())
        ses.close()
        hist = eng.gt_sample_history(sp, ids, ch, par, H, w.Z, rates, lens[:, 0], 3, precision=prec)
        out.append(hist)
        branch = np.array([b if b != np.argmax(par[c] == N) else 1 for c, b in enumerate([0, 3, S, S + 1, S + 2])], np.int32)
        out.append(eng.gt_sample_tree(sp, ids, ch, par, H, w.Z, rates, branch, ind, lens, None, ll, lz, 3, 0, precision=prec))
        return out + [ch, par, H, ll]

    for a, b in zip(moves(0), moves(1)):
        np.testing.assert_array_equal(b, a)
