"""The 8-byte formats of series with NaN, infinities, zeros and tiny amplitudes, as torch's own division
and rounding store them."""
import pytest
import torch

from fastlisaresponse_amd.batch import pack_mixed, pack_q31

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")
SERIES = {
    "NaN in one part": [1 + 2j, complex(NAN, 1.0), complex(-3.0, NAN), 2 - 1j],
    "infinite": [1 + 2j, complex(INF, 1.0), complex(-3.0, -INF), 2 - 1j],
    "NaN and infinite": [1 + 2j, complex(INF, NAN), 0j, 2 - 1j],
    "zeros": [0j, -0j, complex(-0.0, 0.0)],
    "tiny": [1e-300 + 2e-301j, -3e-300j, 5e-301 + 0j],
    "huge": [1e300 + 2e299j, -3e300j, 5e299 + 0j],
}


def _reference(h, q31):
    if q31:
        x = torch.view_as_real(h)
        top = float(x.abs().max())
        top = top if top > 0.0 else 1.0
        full = float(2 ** 31 - 1)
        return torch.round(x.reshape(-1) * (full / top)), top / full
    top = float(h.abs().max())
    top = top if top > 0.0 else 1.0
    return (h / top).to(torch.complex64), top


@pytest.mark.parametrize("name", SERIES)
def test_complex64(name):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    h = torch.tensor(SERIES[name], dtype=torch.complex128, device="cuda")
    got, scales = pack_mixed(h, [len(h)])
    want, top = _reference(h, False)
    assert torch.equal(torch.tensor(scales), torch.tensor([top]))
    assert torch.allclose(torch.view_as_real(got), torch.view_as_real(want), rtol=0.0, atol=0.0,
                          equal_nan=True), (got, want)


@pytest.mark.parametrize("name", ["zeros", "tiny", "huge"])
def test_q31(name):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    h = torch.tensor(SERIES[name], dtype=torch.complex128, device="cuda")
    got, scales = pack_q31(h, [len(h)])
    want, scale = _reference(h, True)
    assert scales == [scale] and torch.equal(got, want.to(torch.int32))
