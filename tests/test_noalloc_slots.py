"""The allocation-free entry point's workgroups hold the slots of the kernel
it launches, whatever the longest element: short elements beside one of 3,000
patterns, more of them than workgroups fit the device, against pa_loglik."""
import numpy as np
import pytest

from phyloacc_amd import engine as E
from phyloacc_amd import synth
from test_zz_no_alloc import _hip, _noalloc, _random_Z

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("typical", [40, 150, 400])
@pytest.mark.parametrize("prec", [E.PA_FP64, E.PA_FP32])
def test_one_long_element_among_many(require_gpu, prec, typical):
    """Mean pattern counts below 96, up to 320 and above: 64, 128 and 256
    threads.  The same terms, grouped by another block size at most."""
    hip = _hip()
    w = synth.make_workload(1, seed=31, lengths=[3000] + [typical] * 12)
    eng = E.Engine.from_workload(w, E.default_options(min_len=1, compress_patterns=0))
    ids, st = eng.add_elements(w.align, w.starts, w.sizes)
    ids = ids[st == E.PA_ELEM_OK]
    rng = np.random.default_rng(typical)
    ids = np.concatenate([ids, rng.choice(ids[1:], 5000), ids[:1]])
    Z = _random_Z(eng, ids, rng)
    rates = np.stack([rng.uniform(0.1, 0.9, len(ids)), rng.uniform(1.2, 4.0, len(ids))], 1)
    ref = eng.loglik(ids, Z, rates, prec)
    for sel in (slice(None), slice(0, 3)):
        np.testing.assert_allclose(_noalloc(eng, hip, ids[sel], Z[sel], rates[sel], prec), ref[sel], rtol=1e-12)
    eng.close()
