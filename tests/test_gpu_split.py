"""The split kernels of short series (flr_split.hip: a sample's work shared by a workgroup's waves)
against the oracle (exact form, bitwise) and against the one-lane kernels of the batch launches (fast
form, the same operations in the same order: bitwise), at lengths that leave one lane, one sample short
of and past a 64-sample tile, and at every dispatch: equal and unequal arms, both stock tables, a table
of more units than one round holds, other orders, accumulation, A, E, T, given sample times, windows
that overflow."""
import numpy as np
import pytest

from test_gpu_parity import _oracle_tables, _setup, gpu, oracle_orbits, orbits  # noqa: F401

pytestmark = pytest.mark.gpu

LONG = [{"link": l, "links_for_delay": d, "sign": s} for l, d, s in
        [(12, [], 1), (23, [12], 1), (31, [12, 23], 1), (13, [], -1), (32, [13], -1),
         (21, [13, 32], -0.5)] + [(13, [31] * (k % 5), 0.25 * k) for k in range(1, 14)]]  # 57 units
P, T = 780, 1000


@pytest.mark.parametrize("n", [2 * P + 1, 2 * P + 63, 2 * P + 64, 2 * P + 65, 3001])
@pytest.mark.parametrize("order", [15, 25, 31])
@pytest.mark.parametrize("times", [False, True])
def test_projection(gpu, orbits, oracle_orbits, oracle_mod, n, order, times):
    import torch
    from fastlisaresponse_amd import _capi
    from fastlisaresponse_amd.tables import sky_basis
    _, rw, (A, deps, E), _ = _setup(gpu, orbits, order=order)
    dt, t0 = 10.0, 1.1e6
    rng = np.random.default_rng(n)
    h = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    k, u, v = sky_basis(0.7, 0.4)
    t = t0 + np.arange(n) * dt
    exp = oracle_mod.get_response(oracle_orbits, h, t, k, u, v, order, 0.1, A, deps, E, P, 4)
    y = torch.full((6 * n,), 7.0, dtype=torch.float64, device="cuda")
    kw = dict(t_data=torch.as_tensor(t, device="cuda")) if times else {}
    rw.projection(y, torch.as_tensor(h, device="cuda"), n, t0, dt, 0.1, k, u, v, P,
                  _capi.FLR_FLAG_ZERO_EDGES | _capi.FLR_FLAG_EXACT, **kw)
    rw.check_errors()
    np.testing.assert_array_equal(y.cpu().numpy().reshape(6, n), exp)


@pytest.mark.parametrize("n", [2 * T + 1, 2 * T + 64, 2 * T + 65, 4003])
@pytest.mark.parametrize("order,tdi", [(25, "1st generation"), (25, "2nd generation"), (25, LONG),
                                       (15, "2nd generation"), (31, LONG)])
def test_tdi(gpu, orbits, oracle_orbits, oracle_mod, n, order, tdi):
    import torch
    from fastlisaresponse_amd import _capi
    _, rw, (A, deps, E), tabs = _setup(gpu, orbits, order=order, tdi=tdi)
    dt = 10.0
    rng = np.random.default_rng(n)
    y, pre = rng.standard_normal((6, n)), rng.standard_normal(3 * n)
    t = np.arange(n) * dt
    yd = torch.as_tensor(y.reshape(-1), device="cuda")
    args = (oracle_orbits, y, t, _oracle_tables(tabs), order, 0.1, A, deps, E, T, 4)
    exp = oracle_mod.get_tdi_delays(*args)
    for flags in (0, _capi.FLR_FLAG_AET):
        out = torch.full((3 * n,), 7.0, dtype=torch.float64, device="cuda")
        rw.tdi(out, yd, n, 0.0, dt, 0.1, T, flags | _capi.FLR_FLAG_OVERWRITE |
               _capi.FLR_FLAG_ZERO_EDGES | _capi.FLR_FLAG_EXACT)
        rw.check_errors()
        want = np.stack(oracle_mod.aet(*exp)) if flags else exp
        np.testing.assert_array_equal(out.cpu().numpy().reshape(3, n), want)
    out = torch.as_tensor(pre.copy(), device="cuda")  # accumulated, with given times
    rw.tdi(out, yd, n, 0.0, dt, 0.1, T, _capi.FLR_FLAG_EXACT, t_arr=torch.as_tensor(t, device="cuda"))
    rw.check_errors()
    np.testing.assert_array_equal(out.cpu().numpy().reshape(3, n),
                                  oracle_mod.get_tdi_delays(*args, delayed_links=pre))


@pytest.mark.parametrize("tdi", ["1st generation", "2nd generation", LONG])
@pytest.mark.parametrize("exact", [True, False])
def test_same_bits_as_the_one_lane_kernels(gpu, orbits, tdi, exact):
    import torch
    from fastlisaresponse_amd import pyResponseTDI
    from fastlisaresponse_amd.batch import BatchedResponse
    n = 5003
    g = torch.Generator().manual_seed(3)
    h = torch.view_as_complex(torch.randn(n, 2, generator=g, dtype=torch.float64)).cuda()
    for chan in ("XYZ", "AET"):
        r = pyResponseTDI(0.1, n, tdi=tdi, orbits=orbits, tdi_chan=chan, exact=exact)
        r.get_projections(h, 1.2, 0.3)
        got = torch.stack(r.get_tdi_delays())
        r.check_errors()
        plan = BatchedResponse(0.1, tdi=tdi, orbits=orbits, tdi_chan=chan,
                               exact=exact).plan(h, [n], [1.2], [0.3])
        plan.run()
        plan.check_errors()
        assert torch.equal(r.y_gw, plan.projections(0))
        assert torch.equal(got, plan.out_all.view(3, n))


def test_window_errors_are_latched(gpu, orbits):
    import torch
    from fastlisaresponse_amd._capi import FLRError
    from fastlisaresponse_amd.tables import sky_basis
    _, rw, _, _ = _setup(gpu, orbits, tdi="2nd generation")
    n, dt = 3000, 10.0
    y = torch.zeros(6 * n, dtype=torch.float64, device="cuda")
    h = torch.zeros(n, dtype=torch.complex128, device="cuda")
    k, u, v = sky_basis(0.1, 0.2)
    late = torch.arange(n, dtype=torch.float64, device="cuda") * dt
    late[1:] += 1.0e6  # a jump no window of the tile holds
    for times in (None, late):
        rw.projection(y, h, n, 0.0, dt, 0.1, k, u, v, 780 if times is not None else 5, 0,
                      t_data=times)
        with pytest.raises(FLRError):
            rw.check_errors()
        out = torch.zeros(3 * n, dtype=torch.float64, device="cuda")
        rw.tdi(out, y, n, 0.0, dt, 0.1, 1000 if times is not None else 5, 0, t_arr=times)
        with pytest.raises(FLRError):
            rw.check_errors()
