"""The exact stencils' two forms of the same quotients, either side of the sample position from which
the two-operation form runs: projections and TDI bitwise equal to the FP64 oracle at the last start
index of one form and the first of the other, on white noise (every bit of a quotient counts)."""
import math

import numpy as np
import pytest

from test_gpu_parity import _oracle_tables, _setup, gpu, oracle_orbits, orbits  # noqa: F401

pytestmark = pytest.mark.gpu

C_INV = 3.3356409519815204e-09
CUSTOM = [{"link": 12, "links_for_delay": [], "sign": 1},
          {"link": 31, "links_for_delay": [12, 23], "sign": 1},
          {"link": 21, "links_for_delay": [13, 32], "sign": -1}]


def _limit(h):
    return 256 if h <= 16 else 512


@pytest.mark.parametrize("order", [15, 25, 31, 35])
@pytest.mark.parametrize("side", [-1, 0])
@pytest.mark.parametrize("limit,n", [(None, 2001), (512, 100_001)])
def test_projection_either_side_of_the_limit(gpu, orbits, oracle_orbits, oracle_mod, order, side, limit,
                                             n):
    import torch
    from fastlisaresponse_amd import _capi
    from fastlisaresponse_amd.tables import sky_basis
    ow, rw, (A, deps, E), _ = _setup(gpu, orbits, order=order)
    dt, h, t0 = 10.0, (order + 1) // 2, 1.1e6
    radius, ltt = ow.extent()
    halo_lo = math.ceil((ltt + radius * C_INV) / dt) + h + 4
    # the second change of form (four reciprocals at a time) in the one-lane kernels, which take the
    # longer series
    if limit == 512 and h > 17:
        limit = 1024
    P = (limit or _limit(h)) + halo_lo - (h - 1) + side
    rng = np.random.default_rng(order + side)
    hh = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    k, u, v = sky_basis(2.2, -0.6)
    exp = oracle_mod.get_response(oracle_orbits, hh, t0 + np.arange(n) * dt, k, u, v, order, 1 / dt,
                                  A, deps, E, P, 16)
    y = torch.zeros(6 * n, dtype=torch.float64, device="cuda")
    rw.projection(y, torch.as_tensor(hh, device="cuda"), n, t0, dt, 1 / dt, k, u, v, P,
                  _capi.FLR_FLAG_ZERO_EDGES | _capi.FLR_FLAG_EXACT)
    rw.check_errors()
    np.testing.assert_array_equal(y.cpu().numpy().reshape(6, n), exp)


@pytest.mark.parametrize("order,tdi", [(25, "1st generation"), (25, "2nd generation"), (25, CUSTOM),
                                       (31, "1st generation"), (35, CUSTOM)])
@pytest.mark.parametrize("side", [-1, 0])
@pytest.mark.parametrize("limit,n", [(None, 1601), (512, 2501), (512, 170_001)])
def test_tdi_either_side_of_the_limit(gpu, orbits, oracle_orbits, oracle_mod, order, tdi, side, limit,
                                      n):
    import torch
    from fastlisaresponse_amd import _capi
    ow, rw, (A, deps, E), tabs = _setup(gpu, orbits, order=order, tdi=tdi)
    dt, h, t0 = 10.0, (order + 1) // 2, 0.0
    limit = limit or _limit(h)
    if n > 2000 and h > 17:
        limit = 1024
    chain = {"1st generation": 3, "2nd generation": 7}.get(tdi, 2) if isinstance(tdi, str) else 2
    halo_lo = math.ceil(chain * ow.extent()[1] / dt) + h + 4
    # the second change of form (four reciprocals at a time) in the split and one-lane kernels, which take
    # the longest series (any other table: past half a million samples)
    if tdi is CUSTOM and n > 100_000:
        n = 530_001
    T = limit + halo_lo - (h - 1) + side
    y = np.random.default_rng(order + side).standard_normal((6, n))
    exp = oracle_mod.get_tdi_delays(oracle_orbits, y, t0 + np.arange(n) * dt, _oracle_tables(tabs),
                                    order, 1 / dt, A, deps, E, T, 16)
    out = torch.zeros(3 * n, dtype=torch.float64, device="cuda")
    rw.tdi(out, torch.as_tensor(y.reshape(-1), device="cuda"), n, t0, dt, 1 / dt, T,
           _capi.FLR_FLAG_OVERWRITE | _capi.FLR_FLAG_ZERO_EDGES | _capi.FLR_FLAG_EXACT)
    rw.check_errors()
    np.testing.assert_array_equal(out.cpu().numpy().reshape(3, n), exp)


@pytest.mark.parametrize("tdi", ["1st generation", "2nd generation"])
@pytest.mark.parametrize("over", [0, 1])
def test_tdi_either_side_of_the_paired_window(gpu, orbits, oracle_orbits, oracle_mod, tdi, over):
    """Equal arms read paired rows of links while 1706 window samples fit, single rows past that."""
    import torch
    from fastlisaresponse_amd import _capi
    order, n, T = 25, 6000, 2000
    ow, rw, (A, deps, E), tabs = _setup(gpu, orbits, order=order, tdi=tdi)
    reach = (3 if tdi == "1st generation" else 7) * ow.extent()[1]
    dt = reach / (1706 - 256 - 2 * 17 + over - 0.5)
    assert 256 + 2 * 17 + math.ceil(reach / dt) == 1706 + over
    y = np.random.default_rng(over).standard_normal((6, n))
    exp = oracle_mod.get_tdi_delays(oracle_orbits, y, np.arange(n) * dt, _oracle_tables(tabs), order,
                                    1 / dt, A, deps, E, T, 16)
    out = torch.zeros(3 * n, dtype=torch.float64, device="cuda")
    rw.tdi(out, torch.as_tensor(y.reshape(-1), device="cuda"), n, 0.0, dt, 1 / dt, T,
           _capi.FLR_FLAG_OVERWRITE | _capi.FLR_FLAG_ZERO_EDGES | _capi.FLR_FLAG_EXACT)
    rw.check_errors()
    np.testing.assert_array_equal(out.cpu().numpy().reshape(3, n), exp)
