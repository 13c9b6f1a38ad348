"""The launch window that a mixed fused batch takes by itself (flr_capi.hip: auto_passes). Equal arms:
whatever the sizes make it, the outputs are those of every explicit window, bit for bit. Unequal arms:
it follows the orbits and the sampling alone, so that a source gives the same bits alone and in a batch,
and those of the explicit window of that length."""
import numpy as np
import pytest

from conftest import YRSID_SI, check_mixed, gb_waveform, unequal_arms

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_gpu():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _plan(torch, cls, precision, tdi, chan, dt, lengths, **kw):
    from fastlisaresponse_amd.batch import BatchedResponse, pack_mixed, pack_q31
    orb = cls(t_max=0.5 * YRSID_SI)
    br = BatchedResponse(1 / dt, tdi=tdi, orbits=orb, tdi_chan=chan, precision=precision,
                         storage_check="off", **kw)
    h = torch.as_tensor(np.concatenate([gb_waveform(n, dt, f=4e-3, phi0=0.1 * s)
                                        for s, n in enumerate(lengths)]), device="cuda")
    scales = None
    if precision != "mixed-c128":
        h, scales = (pack_mixed if precision == "mixed" else pack_q31)(h, lengths)
    return br.plan(h, lengths, [0.3 + s for s in range(len(lengths))], [0.2] * len(lengths),
                   scales=scales)


@pytest.mark.parametrize("precision", ["mixed-c128", "mixed", "mixed-q31"])
@pytest.mark.parametrize("tdi,chan,dt", [("2nd generation", "AET", 10.0),
                                         ("1st generation", "XYZ", 5.0)])
def test_equal_arms_any_size(torch_gpu, precision, tdi, chan, dt):
    torch = torch_gpu
    from fastlisaresponse_amd import EqualArmlengthOrbits
    from fastlisaresponse_amd.autotune import apply
    seen = set()
    for lengths in ([9001], [60001, 5003], [300_001], [700_001, 20_000], [1_400_003]):
        plan = _plan(torch, EqualArmlengthOrbits, precision, tdi, chan, dt, lengths)
        seen.add(plan.launch_shape[0])
        plan.run()
        plan.check_errors()
        got = plan.out_all.clone()
        for window in (256, 512, 1024):
            apply(plan, window, 32)
            plan.out_all.fill_(float("nan"))
            plan.run()
            plan.check_errors()
            assert torch.equal(plan.out_all, got), (lengths, window)
    assert len(seen) > 1  # the sizes span the rule


def test_unequal_arms_alone_and_in_a_batch(torch_gpu):
    torch = torch_gpu
    from fastlisaresponse_amd import CartwheelOrbits
    from fastlisaresponse_amd.autotune import apply
    lengths = [9001, 700_001, 40_001]
    plan = _plan(torch, CartwheelOrbits, "mixed-c128", "2nd generation", "AET", 10.0, lengths)
    plan.run()
    plan.check_errors()
    for s, n in enumerate(lengths):
        o = sum(lengths[:s])
        one = plan.br.plan(plan.h_all[o:o + n].clone(), [n], [0.3 + s], [0.2])
        assert one.launch_shape[0] == plan.launch_shape[0]
        one.run()
        one.check_errors()
        assert torch.equal(one.out_all, plan.out_all[3 * o:3 * (o + n)]), s
    got = plan.out_all.clone()
    apply(plan, plan.launch_shape[0], 16)
    plan.run()
    plan.check_errors()
    assert torch.equal(plan.out_all, got)


@pytest.mark.parametrize("cls_name", ["EqualArmlengthOrbits", "CartwheelOrbits"])
@pytest.mark.parametrize("tdi,dt", [("2nd generation", 15.0), ("2nd generation", 8.0),
                                    ("2nd generation", 6.5), ("2nd generation", 4.2),
                                    ("1st generation", 7.0)])
def test_filters_of_every_length(torch_gpu, oracle_mod, cls_name, tdi, dt):
    """Composite filters of 11 to 14 matrix steps against the oracle, on input as fast as order 25
    interpolates well."""
    import fastlisaresponse_amd.orbits as orbits_mod
    torch = torch_gpu
    orbits = getattr(orbits_mod, cls_name)(t_max=1.2 * YRSID_SI)
    orbits.configure(linear_interp_setup=True)
    oo = oracle_mod.OracleOrbits(*orbits.pycppdetector_args)
    n, t0 = 9000, 1.0e6
    f = 0.1 / dt
    h = gb_waveform(n, dt, 1e-21, f, 1e-17, 0.7, 0.2, 0.4, t0=t0)
    from fastlisaresponse_amd.batch import BatchedResponse
    br = BatchedResponse(1.0 / dt, tdi=tdi, orbits=orbits, tdi_chan="XYZ", precision="mixed-c128",
                         t_buffer=1000.0 * dt)
    plan = br.plan(torch.as_tensor(h, device="cuda"), [n], [0.9], [-0.4], [t0])
    plan.run()
    plan.check_errors()
    y, exp = oracle_mod.response_pipeline(oo, h, 0.9, -0.4, dt, 25, tdi, t0=t0, tdi_chan="XYZ",
                                          x_base=orbits.x_base, nthreads=8,
                                     t_buffer=1000.0 * dt)
    got = torch.stack(plan.channels(0)).cpu().numpy().astype(np.float64)
    # the outputs' float32 rounding, and positions within 1e-8 samples (times 2 pi f dt = 0.63) in each
    # of up to 16 units of the projections' size
    T = br.tdi_start_ind
    units = 16 if tdi == "2nd generation" else 8
    size = np.sqrt(np.mean(y[:, T:-T] ** 2)) / np.sqrt(np.mean(exp[:, T:-T] ** 2))
    check_mixed(oracle_mod, oo, got, y, exp, t0, dt, tdi, "XYZ", 2.0 ** -24 + 0.63e-8 * units * size, T,
                (), unequal_arms(orbits))
