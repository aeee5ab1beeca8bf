"""The autotuner's candidates are different kernels: shape 1 is accepted
where a shape is set but is shape 0's kernel, so it is not timed beside it
(it took one of the three places of the second round from another block
size or shape)."""
import pytest

from phyloacc_amd import engine as E
from test_tuning import _engine


def test_shape_one_is_still_accepted():
    eng, _ = _engine(2)
    eng.set_tuning(128, 1)
    t = eng.tuning()
    assert t["block_threads"] == 128 and t["shape"] == 1 and (t["round_nodes"], t["chunk_nodes"]) == (1, 4)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [E.PA_FP32, E.PA_FP64])
def test_the_autotuner_keeps_a_shape_of_its_own(require_gpu, precision):
    for n in (4, 9, 20, 33):
        eng, ids = _engine(n, seed=n)
        assert eng.autotune(ids, precision=precision, states=8)["shape"] in (0, 2)
