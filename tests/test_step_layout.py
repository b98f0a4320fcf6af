"""The host side of a step: the tokens that `Engine.execute` takes and the arrays that a step's batch is laid out in."""
import numpy as np
import pytest
import torch

from qserve_amd.serving.engine import Engine


class _Model:
    vocab = 100


def _engine():
    e = object.__new__(Engine)
    e.model = _Model()
    return e


class _OnAnotherDevice:
    """A token as a 0-dim tensor on the GPU gives it: int() works, numpy's conversion raises."""

    def __init__(self, v):
        self.v = v

    def __int__(self):
        return self.v

    def __array__(self, *args, **kwargs):
        raise TypeError("can't convert cuda:0 device type tensor to numpy")


@pytest.mark.parametrize("tokens", [[3, 99, 0], (3, 99, 0), [_OnAnotherDevice(v) for v in (3, 99, 0)], [3, _OnAnotherDevice(99), 0],
                                    [torch.tensor(3), torch.tensor(99), torch.tensor(0)], [torch.tensor([3]), 99, 0], torch.tensor([3, 99, 0]),
                                    np.array([3, 99, 0], dtype=np.int32), [np.int64(3), np.uint8(99), False], [3.0, 99.7, 0]])
def test_tokens_are_whatever_int_takes(tokens):
    ids = _engine()._token_ids(tokens)
    assert ids.dtype == np.int64 and ids.tolist() == [3, 99, 0]


@pytest.mark.parametrize("tokens", [[3, 100], [-1], [2 ** 70], [3, 2 ** 63], [_OnAnotherDevice(100)], torch.tensor([100]), [100.5]])
def test_tokens_outside_the_vocabulary_are_refused(tokens):
    with pytest.raises(ValueError, match="vocabulary"):
        _engine()._token_ids(tokens)
