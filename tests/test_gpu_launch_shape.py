"""BatchPlan.launch_shape is the shape that the library runs."""
import pytest

from conftest import gb_waveform

pytestmark = pytest.mark.gpu


def test_follows_the_library():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from fastlisaresponse_amd import EqualArmlengthOrbits
    from fastlisaresponse_amd._capi import check, lib
    from fastlisaresponse_amd.autotune import apply
    from fastlisaresponse_amd.batch import BatchedResponse
    orbits = EqualArmlengthOrbits()
    orbits.configure(linear_interp_setup=True)
    h = torch.as_tensor(gb_waveform(9_001, 10.0), device="cuda")
    plan = BatchedResponse(0.1, orbits=orbits, precision="mixed-c128").plan(h, [9_001], [0.3], [0.2])
    assert plan.launch_shape == (256, 32)
    apply(plan, 1024, 8)
    assert plan.launch_shape == (1024, 8)
    check(lib().flr_batch_set_launch(plan._h, 512, 0))
    assert plan.launch_shape == (512, 8)
    plan.rebind([1.0], [0.1], [3.5e7])
    assert plan.launch_shape == (512, 8)
    fp = BatchedResponse(0.1, orbits=orbits).plan(h, [9_001], [0.3], [0.2])
    assert fp.launch_shape == (256, 32)
