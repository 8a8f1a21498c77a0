"""A training batch that does not fit the device."""
import numpy as np
import pytest

from desalm import cases
from desalm.lib import DesalmError, Solver

pytestmark = pytest.mark.gpu


def solver():
    c = cases.wavy(13, 11, 9, ng=2, itm=2, iters=(1, 2))
    s = Solver(c.params).load_case(c)
    s.ws_configure(hidden=16, samples_per_record=128, capacity=512, seed=3)
    for _ in range(3):
        s.step()
        s.ws_record()
    return s


def test_training_goes_on_after_a_batch_too_large(gpu):
    """2^30 rows need 412 GB for the inputs alone: refused by the allocator,
    and the network trains on as if nothing had been asked for."""
    a, b = solver(), solver()
    la = [a.ws_train(5, batch=64), a.ws_train(5, batch=64)]
    lb = [b.ws_train(5, batch=64)]
    with pytest.raises(DesalmError, match="out of device memory"):
        b.ws_train(5, batch=1 << 30)
    lb.append(b.ws_train(5, batch=64))
    assert np.array_equal(np.concatenate(la), np.concatenate(lb))
    assert np.array_equal(a.ws_params(), b.ws_params())
    a.close()
    b.close()
