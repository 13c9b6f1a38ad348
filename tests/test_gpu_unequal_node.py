"""The 1024-sample tiles of the mixed form with unequal arms follow the orbit node that a tile spans: the
null channel T, which shows the delays' errors first, against the TDI with extended-precision delays."""
import numpy as np
import pytest

from conftest import YRSID_SI, gb_waveform, rel_l2
from test_gpu_unequal import NTH, wobbly_orbits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_gpu():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _cartwheel():
    from fastlisaresponse_amd.orbits import CartwheelOrbits
    o = CartwheelOrbits(t_max=1.2 * YRSID_SI)
    o.configure(linear_interp_setup=True)
    return o


def _plan(torch, orbits, h, n, dt, t0, tdi):
    from fastlisaresponse_amd.batch import BatchedResponse
    br = BatchedResponse(1 / dt, tdi=tdi, orbits=orbits, precision="mixed-c128", t_buffer=max(1e4, 1e3 * dt))
    return br.plan(torch.as_tensor(h, device="cuda"), [n], [1.2], [0.3], [t0])


@pytest.mark.parametrize("make,f0,t0,dt,tdi", [
    (_cartwheel, 2e-3, 2e6, 10.0, "2nd generation"),
    (_cartwheel, 2e-3, 1.5e7, 10.0, "2nd generation"),
    (_cartwheel, 2e-3, 2e6, 10.0, "1st generation"),
    (_cartwheel, 2e-3, 2e6, 5.0, "2nd generation"),
    # arms whose slopes change by 1.5e-12 s/s at the nodes
    (lambda: wobbly_orbits(3e-8, 1e5), 4e-3, 2e6, 10.0, "2nd generation"),
])
def test_null_channel_of_long_tiles(torch_gpu, oracle_mod, make, f0, t0, dt, tdi):
    torch = torch_gpu
    orbits, n = make(), 1 << 17
    T = int(1e4 / dt)
    h = gb_waveform(n, dt, f=f0, fdot=1e-16, t0=t0)
    oo = oracle_mod.OracleOrbits(*orbits.pycppdetector_args)
    y, _ = oracle_mod.response_pipeline(oo, h, 1.2, 0.3, dt, 25, tdi, t0=t0, x_base=orbits.x_base,
                                        nthreads=NTH)
    y = np.asarray(y).reshape(6, -1)
    ext = oracle_mod.tdi_extended_delays(oo, y, t0, dt, tdi, tdi_start=T, chan="AET")[2, T:-T]
    plan = _plan(torch, orbits, h, n, dt, t0, tdi)
    assert plan.launch_shape[0] == 1024
    plan.run()
    plan.check_errors()
    got = plan.channels(0)[2].double().cpu().numpy()[T:-T]
    # the outputs' float32 rounding and, in the one group of 256 samples that the node lies in, the
    # distance from two lines of their closest one: up to 4e-9 of T in 64 bits for these sources (a line
    # through the whole tile: 2.7e-8, and 1.2e-8 through one of half the length)
    rounding = rel_l2(ext.astype(np.float32), ext)
    assert rel_l2(got, ext) <= np.hypot(rounding, 6e-9), (rel_l2(got, ext), rounding)


@pytest.mark.parametrize("dt,window", [(10.0, 1024), (15.0, 512)])
def test_long_tiles_span_one_node_at_most(torch_gpu, dt, window):
    n = 20_000
    plan = _plan(torch_gpu, _cartwheel(), gb_waveform(n, dt), n, dt, 0.0, "2nd generation")
    assert plan.launch_shape[0] == window


@pytest.mark.parametrize("chan", ["AET", "XYZ"])
def test_inner_products_of_long_tiles_around_large_kinks(torch_gpu, chan):
    """Where the samples around a node are done once for each side of it, every sample meets the data
    once: the sums against those of the stored outputs, up to their float32 rounding."""
    from fastlisaresponse_amd.batch import BatchedResponse
    torch = torch_gpu
    n, dt, t0 = 1 << 17, 10.0, 2e6
    h = torch.as_tensor(gb_waveform(n, dt, f=4e-3, fdot=1e-16, t0=t0), device="cuda")
    br = BatchedResponse(1 / dt, orbits=wobbly_orbits(3e-8, 1e5), tdi_chan=chan, precision="mixed-c128")
    plan = br.plan(h, [n], [1.2], [0.3], [t0])
    assert plan.launch_shape[0] == 1024
    plan.run()
    T = br.tdi_start_ind
    g = torch.Generator(device="cuda").manual_seed(4)
    data = torch.randn(plan.out_all.shape, generator=g, device="cuda") * plan.out_all.abs().max()
    sums = plan.inner_products(data)[0]
    plan.check_errors()
    out = plan.out_all.view(3, n).double()[:, T:n - T]
    d = data.view(3, n).double()[:, T:n - T]
    hh, dd = out.square().sum(1), d.square().sum(1)
    assert bool(((sums[:, 1] - hh).abs() <= 2.0 ** -23 * hh).all())
    assert bool(((sums[:, 0] - (d * out).sum(1)).abs() <= 2.0 ** -24 * (dd * hh).sqrt()).all())
