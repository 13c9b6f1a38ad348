"""The packed series' statistics and 8-byte conversions on the GPU (flr_series_stats,
flr_series_pack) against the same quantities from plain torch operations: scales and stored
samples bit for bit (the same maximum, one product per component, one rounding), the RMS
frequencies to the rounding of a sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHUNK = 4096  # samples per workgroup of the kernels


@pytest.fixture(scope="module")
def torch_gpu():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _series(torch, lengths, seed):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(sum(lengths), 2, generator=g, dtype=torch.float64)
    amp = torch.repeat_interleave(10.0 ** torch.arange(-23.0, -23.0 + len(lengths)),
                                  torch.tensor(lengths))
    return torch.view_as_complex(h * amp[:, None]).cuda()


def _by_torch(torch, h, n, q31):
    """One source in plain torch: (stored, scale)."""
    if q31:
        seg = torch.view_as_real(h)
        s = float(seg.abs().max()) if n else 1.0
        s = s if s > 0.0 else 1.0
        full = float(2 ** 31 - 1)
        return torch.round(seg.reshape(-1) * (full / s)).to(torch.int32), s / full
    s = float(h.abs().max())
    s = s if s > 0.0 else 1.0
    return (h / s).to(torch.complex64), s


@pytest.mark.parametrize("lengths", [[1], [2], [255], [CHUNK], [CHUNK + 1], [3 * CHUNK - 1],
                                     [1, CHUNK, 5, 2 * CHUNK + 17, 300], [1 << 20]])
def test_pack_matches_torch(torch_gpu, lengths):
    torch = torch_gpu
    from fastlisaresponse_amd.batch import pack_mixed, pack_q31, rms_frequencies
    h = _series(torch, lengths, 5)
    for q31, pack in ((False, pack_mixed), (True, pack_q31)):
        stored, scales = pack(h, lengths)
        o = 0
        for s, n in enumerate(lengths):
            exp, sc = _by_torch(torch, h[o:o + n], n, q31)
            per = 2 if q31 else 1
            assert scales[s] == sc
            assert torch.equal(stored[per * o:per * (o + n)], exp)
            o += n
        # sums of up to 2^20 terms in another order: 2^20 * 2^-53 relative at most
        np.testing.assert_allclose(rms_frequencies(stored, lengths, 10.0),
                                   rms_frequencies(stored.cpu(), lengths, 10.0), rtol=1e-9)
    np.testing.assert_allclose(rms_frequencies(h, lengths, 10.0),
                               rms_frequencies(h.cpu(), lengths, 10.0), rtol=1e-9)


def test_pack_special_values_and_views(torch_gpu):
    torch = torch_gpu
    from fastlisaresponse_amd.batch import pack_mixed, pack_q31
    h = _series(torch, [3 * CHUNK], 7)
    zero = torch.zeros(100, dtype=torch.complex128, device="cuda")
    assert pack_mixed(zero, [100])[1] == [1.0]
    assert pack_q31(zero, [100])[1] == [1.0 / float(2 ** 31 - 1)]
    # a NaN anywhere leaves no maximum: scale 1, as torch's max
    bad = h.clone()
    bad[CHUNK + 3] = complex(float("nan"), 0.0)
    stored, scales = pack_mixed(bad, [bad.numel()])
    exp, sc = _by_torch(torch, bad, bad.numel(), False)
    assert scales == [sc] == [1.0]
    assert torch.equal(torch.nan_to_num(torch.view_as_real(stored)),
                       torch.nan_to_num(torch.view_as_real(exp)))
    # a conjugated view and a strided one hold other values than their storage
    for view in (h.conj(), h[::3]):
        stored, scales = pack_mixed(view, [view.numel()])
        exp, sc = _by_torch(torch, view.resolve_conj().contiguous(), view.numel(), False)
        assert scales == [sc] and torch.equal(stored, exp)
    # an empty source takes scale 1
    assert pack_mixed(h, [0, h.numel()])[1][0] == 1.0


def test_dropin_packs_and_guards_in_one_pass(torch_gpu):
    torch = torch_gpu
    from fastlisaresponse_amd import EqualArmlengthOrbits, pyResponseTDI
    from fastlisaresponse_amd.batch import StorageErrorWarning
    orb = EqualArmlengthOrbits(t_max=1.0e7)
    n = 20011
    t = torch.arange(n, dtype=torch.float64, device="cuda") * 10.0
    for precision in ("mixed", "mixed-q31"):
        r = pyResponseTDI(0.1, n, orbits=orb, tdi_chan="AET", precision=precision)
        h = 1e-21 * torch.exp(2j * np.pi * 5e-3 * t)
        r.get_projections(h, 0.4, 0.2)
        exp, sc = _by_torch(torch, h, n, precision == "mixed-q31")
        assert torch.equal(r._mixed[0], exp) and r._mixed[1] == sc
        with pytest.warns(StorageErrorWarning):
            r.get_projections(1e-21 * torch.exp(2j * np.pi * 1e-4 * t), 0.4, 0.2)
        r.storage_check = "raise"
        with pytest.raises(ValueError, match="storage error"):
            r.get_projections(1e-21 * torch.exp(2j * np.pi * 1e-4 * t), 0.4, 0.2)
