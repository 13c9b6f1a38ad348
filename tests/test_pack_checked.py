"""pack_checked: an unknown action is refused, and its warning names the line that called its caller."""
import inspect
import warnings

import pytest
import torch

from fastlisaresponse_amd.batch import StorageErrorWarning, pack_checked


def _projections(h, action):
    return pack_checked(h, 10.0, "mixed", 2.5e9, action)


def _h(device):
    t = torch.arange(4096, dtype=torch.float64, device=device) * 10.0
    return torch.polar(torch.full_like(t, 1e-21), 2e-4 * t)  # slow: the estimate is over its bound


def _check(h):
    with pytest.raises(ValueError):
        _projections(h, "maybe")
    with pytest.raises(ValueError):
        _projections(h, "raise")
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        _projections(h, "off")
        line = inspect.currentframe().f_lineno + 1
        _projections(h, "warn")
    assert [w.category for w in seen] == [StorageErrorWarning]
    assert (seen[0].filename, seen[0].lineno) == (__file__, line)


def test_host_series():
    _check(_h("cpu"))


@pytest.mark.gpu
def test_device_series():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from fastlisaresponse_amd.batch import rms_frequencies
    _check(_h("cuda"))
    with pytest.raises(RuntimeError):  # a recorded gradient, as numpy refuses it
        _projections(_h("cuda").requires_grad_(), "warn")
    with pytest.raises(RuntimeError):  # an odd number of q31 words
        rms_frequencies(torch.ones(9, dtype=torch.int32, device="cuda"), [4], 10.0)
