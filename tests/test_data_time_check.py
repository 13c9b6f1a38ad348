"""The input is trimmed where it is longer than the orbits' times, in whatever order those lie."""
import types
import warnings

import numpy as np
import pytest

from fastlisaresponse_amd.response import pyResponseTDI


@pytest.mark.parametrize("t", [[0.0, 50.0, 100.0], [100.0, 50.0, 0.0], [0.0, 100.0, 50.0]])
@pytest.mark.parametrize("n,kept", [(8, 8), (11, 11), (12, 10)])
def test_trimmed_at_the_largest_time(t, n, kept):
    me = types.SimpleNamespace(dt=10.0, response_orbits=types.SimpleNamespace(t=np.array(t)))
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        out = pyResponseTDI._data_time_check(me, 0.0, n, np.arange(n))
    assert len(out) == kept and len(seen) == (kept != n)
