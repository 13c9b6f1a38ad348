"""Inner products of one source are the same bits alone, in any batch and at any launch shape: their window
follows the response and the sampling alone (flr_capi.hip: inner_passes)."""
import numpy as np
import pytest

from conftest import YRSID_SI, gb_waveform

pytestmark = pytest.mark.gpu

LENGTHS = [700_001, 20_011, 150_000]


@pytest.fixture(scope="module")
def torch_gpu():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("cls_name", ["EqualArmlengthOrbits", "CartwheelOrbits"])
@pytest.mark.parametrize("tdi,dt", [("2nd generation", 10.0), ("1st generation", 5.0)])
def test_sums_alone_and_in_a_batch(torch_gpu, cls_name, tdi, dt):
    import fastlisaresponse_amd.orbits as orbits_mod
    from fastlisaresponse_amd.autotune import apply
    from fastlisaresponse_amd.batch import BatchedResponse
    torch = torch_gpu
    orbits = getattr(orbits_mod, cls_name)(t_max=0.5 * YRSID_SI)
    orbits.configure(linear_interp_setup=True)
    br = BatchedResponse(1 / dt, tdi=tdi, orbits=orbits, precision="mixed-c128")
    hs = [torch.as_tensor(gb_waveform(n, dt, f=4e-3, phi0=0.1 * s), device="cuda")
          for s, n in enumerate(LENGTHS)]
    lam, beta = [0.3, 1.3, 2.3], [0.2, -0.4, 0.9]
    plan = br.plan(torch.cat(hs), LENGTHS, lam, beta)
    g = torch.Generator(device="cuda").manual_seed(9)
    data = torch.randn(plan.out_all.shape, generator=g, device="cuda") * 1e-21
    sums = plan.inner_products(data).clone()
    windows = {plan.launch_shape[0]}
    for s, n in enumerate(LENGTHS):
        o = 3 * int(plan.offsets[s])
        one = br.plan(hs[s], [n], lam[s:s + 1], beta[s:s + 1])
        windows.add(one.launch_shape[0])
        part = data[o:o + 3 * n].clone()
        assert torch.equal(one.inner_products(part)[0], sums[s]), s
    if cls_name == "EqualArmlengthOrbits":
        assert len(windows) > 1  # the runs' windows differ
    for window in (256, 512, 1024):
        apply(plan, window, 16)
        assert torch.equal(plan.inner_products(data), sums), window
        plan.run()
    plan.check_errors()
    # and the sums are those of the stored outputs, up to their float32 rounding
    for s, n in enumerate(LENGTHS):
        T = br.tdi_start_ind
        h = torch.stack(plan.channels(s)).double()[:, T:n - T]
        hh = h.square().sum(1)
        assert bool(((sums[s, :, 1] - hh).abs() <= 2.0 ** -23 * hh).all()), s
