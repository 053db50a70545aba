"""Net.fit on fewer samples than a batch takes no step: it returns a NaN per
epoch whatever the arrays are, as nothing reads them; arrays that a step would
read are still looked at first."""
import math

import pytest
import torch

from koral_amd import learn


def _net():
    net = learn.Net.__new__(learn.Net)
    net.L, net.h = None, None  # no step may be taken
    return net


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rows", [learn.NIN, 3])
def test_no_batch_no_step(dtype, rows):
    X, T = torch.zeros((rows, 10), dtype=dtype), torch.zeros((learn.NOUT, 10), dtype=dtype)
    hist = _net().fit(X, T, epochs=3, batch=11)
    assert len(hist) == 3 and all(math.isnan(h) for h in hist)


def test_a_batch_is_checked():
    X, T = torch.zeros((learn.NIN, 10)), torch.zeros((learn.NOUT, 10))
    with pytest.raises(ValueError):
        _net().fit(X.double(), T, epochs=1, batch=10)
    with pytest.raises(ValueError):
        _net().fit(X[:3], T, epochs=1, batch=10)
    with pytest.raises(ValueError):
        _net().fit(X, T[:, :9], epochs=1, batch=10)
