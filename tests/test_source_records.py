"""The source records of a plan: numbers of every kind that indexes and converts give the records of one
entry at a time, and what those refuse stays refused."""
import types
import warnings

import numpy as np
import pytest
import torch

from fastlisaresponse_amd.batch import _SOURCE_DTYPE, BatchPlan
from fastlisaresponse_amd.tables import sky_basis

N = 7
RNG = np.random.default_rng(3)
LAM, BETA = RNG.uniform(0, 6, N), RNG.uniform(-1, 1, N)
T0, SCALE = RNG.uniform(0, 1e7, N), RNG.uniform(1e-22, 1, N)


def _records(lams, betas, t0s=None, scales=None):
    plan = types.SimpleNamespace(lengths=np.full(N, 100), offsets=np.arange(N) * 100,
                                 br=types.SimpleNamespace(projections_start_ind=5, tdi_start_ind=10))
    plan._records_by_entry = lambda *a: BatchPlan._records_by_entry(plan, *a)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        return BatchPlan._records(plan, lams, betas, t0s, scales)


def _by_entry(lams, betas, t0s, scales):
    rec = np.zeros(N, dtype=_SOURCE_DTYPE)
    for s in range(N):
        k, u, v = sky_basis(lams[s], betas[s])
        rec[s]["offset"], rec[s]["num_pts"] = 100 * s, 100
        rec[s]["projections_start_ind"], rec[s]["tdi_start_ind"] = 5, 10
        rec[s]["t0"], rec[s]["scale"] = float(t0s[s]), float(scales[s])
        for c in range(3):
            rec[s]["k"][c], rec[s]["u"][c], rec[s]["v"][c] = float(k[c]), float(u[c]), float(v[c])
    return rec


def _columns(x):
    return np.stack([x, x + 1.0], axis=1)[:, 0]


FORMS = {
    "arrays": lambda x: x,
    "strided": _columns,
    "lists": lambda x: [float(v) for v in x],
    "float64 lists": list,
    "tuples": tuple,
    "tensors": torch.as_tensor,
    "float32 arrays": lambda x: x.astype(np.float32),
    "float32 tensors": lambda x: torch.as_tensor(x, dtype=torch.float32),
    "lists of float32 tensors": lambda x: list(torch.as_tensor(x, dtype=torch.float32)),
    "mixed lists": lambda x: [np.float32(x[0]), float(x[1]), x[2], 1, x[4], np.float32(x[5]), x[6]],
    "objects": lambda x: x.astype(object),
    "ints": lambda x: np.arange(N),
    "dicts": lambda x: dict(enumerate(x)),
}


@pytest.mark.parametrize("form", FORMS)
def test_every_form_is_taken_entry_by_entry(form):
    args = [FORMS[form](x) for x in (LAM, BETA, T0, SCALE)]
    assert _same(_records(*args), _by_entry(*args))


def _same(a, b):
    return a.dtype == b.dtype and a.tobytes() == b.tobytes()


@pytest.mark.parametrize("which", [2, 3])
def test_column_shaped_start_times_and_scales(which):
    args = [LAM, BETA, T0, SCALE]
    args[which] = args[which][:, None]
    assert _same(_records(*args), _by_entry(LAM, BETA, T0, SCALE))


def test_defaults():
    assert _same(_records(LAM, BETA), _by_entry(LAM, BETA, np.zeros(N), np.ones(N)))


@pytest.mark.parametrize("which,value,error", [
    (0, torch.as_tensor(LAM).requires_grad_(), RuntimeError),
    (2, [None] * N, TypeError),
    (2, np.stack([T0, T0], axis=1), TypeError),
    (1, BETA[:3], ValueError),
])
def test_refused_forms(which, value, error):
    args = [LAM, BETA, T0, SCALE]
    args[which] = value
    with pytest.raises(error):
        _records(*args)
