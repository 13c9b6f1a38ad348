"""The launch window of a bound mixed plan: BatchPlan.rebind keeps it, whatever the new start times, so
that captured runs and inner products, which hold the tile length and the tile count, keep replaying
the bound sources (flr_capi.hip: flr_fused_bind). With equal arms the start times decide whether every
tile passes the composite filters' test as a whole, here at 0 s but not at 3.5e7 s."""
import numpy as np
import pytest

from conftest import gb_waveform

pytestmark = pytest.mark.gpu

LENGTHS = [90_001, 5_003, 40_011]
EARLY, LATE = 0.0, 3.5e7


@pytest.fixture(scope="module")
def torch_gpu():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _plan(torch, t0, orbits):
    from fastlisaresponse_amd.batch import BatchedResponse
    h = torch.as_tensor(np.concatenate([gb_waveform(n, 10.0, f=4e-3, phi0=0.1 * s)
                                        for s, n in enumerate(LENGTHS)]), device="cuda")
    br = BatchedResponse(0.1, tdi="2nd generation", orbits=orbits, precision="mixed-c128")
    return br.plan(h, LENGTHS, [0.3, 1.3, 2.3], [0.2, -0.4, 0.9], [t0] * 3)


def _shape(plan):
    import ctypes

    from fastlisaresponse_amd._capi import check, lib
    tile, grid = ctypes.c_int(), ctypes.c_int()
    check(lib().flr_batch_launch(plan._h, ctypes.byref(tile), ctypes.byref(grid)))
    return tile.value, grid.value


def _rebind(plan, t0):
    plan.rebind([2.0, 0.5, 4.0], [0.1, 0.7, -0.2], [t0] * 3)


def _capture(torch, call):
    call()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call()
    return g


@pytest.fixture(scope="module")
def orbits():
    from fastlisaresponse_amd import EqualArmlengthOrbits
    o = EqualArmlengthOrbits()
    o.configure(linear_interp_setup=True)
    return o


@pytest.mark.parametrize("first,then", [(LATE, EARLY), (EARLY, LATE)])
def test_rebind_keeps_the_window(torch_gpu, orbits, first, then):
    torch = torch_gpu
    plan = _plan(torch, first, orbits)
    shape = _shape(plan)
    _rebind(plan, then)
    assert _shape(plan) == shape
    plan.run()
    plan.check_errors()
    fresh = _plan(torch, then, orbits)
    _rebind(fresh, then)
    fresh.run()
    fresh.check_errors()
    assert torch.equal(plan.out_all, fresh.out_all)


def test_graphs_replay_the_rebound_sources(torch_gpu, orbits):
    torch = torch_gpu
    plan = _plan(torch, LATE, orbits)
    g = torch.Generator(device="cuda").manual_seed(5)
    data = torch.randn(plan.out_all.shape, generator=g, device="cuda") * 1e-21
    sums = torch.empty((3, 3, 4), dtype=torch.float64, device="cuda")
    runs = _capture(torch, plan.run)
    inner = _capture(torch, lambda: plan.inner_products(data, sums))
    _rebind(plan, EARLY)
    fresh = _plan(torch, EARLY, orbits)
    _rebind(fresh, EARLY)
    fresh.run()
    want = fresh.inner_products(data).clone()
    for rep in range(3):
        plan.out_all.fill_(float("nan"))
        sums.fill_(float("nan"))
        torch.cuda.synchronize()
        runs.replay()
        inner.replay()
        torch.cuda.synchronize()
        assert torch.equal(plan.out_all, fresh.out_all), rep
        # (d|h) and (h|h): sums of up to 9e4 products, each within 2^-53 of sqrt((d|d) (h|h))
        dd = torch.stack([data[3 * o:3 * (o + n)].view(3, n).double().square().sum(1)
                          for o, n in zip(plan.offsets, LENGTHS)])
        size = torch.stack([(dd * want[..., 1]).sqrt(), want[..., 1]], dim=-1)
        assert bool(((sums - want)[..., :2].abs() <= 9e4 * 2.0 ** -53 * size).all()), rep
        # eager work between the replays
        assert torch.equal(plan.inner_products(data), sums)
    plan.check_errors()


def test_a_replay_without_its_proof_reports(torch_gpu, orbits):
    """A run captured where every tile passes the filters' test holds no per-sample stencils: replayed
    with sources that need them it writes NaN and latches an error, and an eager run is right."""
    torch = torch_gpu
    plan = _plan(torch, EARLY, orbits)
    runs = _capture(torch, plan.run)
    _rebind(plan, LATE)
    runs.replay()
    torch.cuda.synchronize()
    assert bool(plan.out_all.isnan().any())
    with pytest.raises(RuntimeError):
        plan.check_errors()
    plan.run()
    plan.check_errors()
    assert not bool(plan.out_all.isnan().any())


@pytest.mark.parametrize("lengths", [[9_001], [90_001, 5_003, 40_011], [700_001, 20_000]])
def test_window_of_any_start_time(torch_gpu, orbits, lengths):
    """The rule counts tiles: plans of the same sources take the same window at any start time, and their
    outputs are those of every explicit window."""
    from fastlisaresponse_amd.autotune import apply
    from fastlisaresponse_amd.batch import BatchedResponse
    torch = torch_gpu
    br = BatchedResponse(0.1, tdi="2nd generation", orbits=orbits, precision="mixed-c128")
    m = len(lengths)
    h = torch.as_tensor(np.concatenate([gb_waveform(n, 10.0, f=4e-3) for n in lengths]), device="cuda")
    shapes = set()
    for t0 in (EARLY, LATE, 2.8e8):
        plan = br.plan(h, lengths, [0.3] * m, [0.2] * m, [t0] * m)
        shapes.add(_shape(plan))
        plan.run()
        plan.check_errors()
        got = plan.out_all.clone()
        for window in (256, 512, 1024):
            apply(plan, window, 32)
            plan.run()
            plan.check_errors()
            assert torch.equal(plan.out_all, got), (t0, window)
    assert len(shapes) == 1


@pytest.mark.parametrize("lengths,dt,window", [([8_552] * 48, 7.0, 512), ([74_783] * 8, 10.0, 512),
                                               ([131_072] * 32, 10.0, 1024), ([9_001], 10.0, 256),
                                               ([131_072] * 32, 5.3, 1024)])
def test_window_by_the_computed_tiles(torch_gpu, orbits, lengths, dt, window):
    """Tiles in the zeroed edges count nothing, and 512 samples are left only for a tenth or more."""
    from fastlisaresponse_amd.batch import BatchedResponse
    torch = torch_gpu
    br = BatchedResponse(1 / dt, tdi="2nd generation", orbits=orbits, precision="mixed-c128")
    m = len(lengths)
    h = torch.zeros(sum(lengths), dtype=torch.complex128, device="cuda")
    plan = br.plan(h, lengths, [0.3] * m, [0.2] * m)
    assert _shape(plan)[0] == window
