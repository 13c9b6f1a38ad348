"""GBWave's number of samples, len(arange(0, T yr, dt)), without making the array (CPU)."""
import numpy as np
import pytest

from conftest import YRSID_SI


@pytest.mark.parametrize("dt", [0.1, 2.5, 5.0, 10.0, 15.0, 1 / 3])
def test_count_is_that_of_arange(dt):
    from fastlisaresponse_amd.waveforms import num_samples
    rng = np.random.default_rng(int(10 * dt))
    spans = [0.0, dt / 2, dt] + [n * dt for n in rng.integers(1, 300_000, 300)]
    spans += list(rng.uniform(0, 1e5 * dt, 100)) + [np.nextafter(1000 * dt, s) for s in (0, 1e9)]
    for span in spans:
        T = span / YRSID_SI
        assert num_samples(T, dt) == len(np.arange(0.0, T * YRSID_SI, dt)), (span, dt)


def test_one_record_is_the_tables():
    """The record GBWave packs from plain numbers, byte for byte gb_table's."""
    from fastlisaresponse_amd import waveforms as w
    rng = np.random.default_rng(4)
    for _ in range(200):
        A, f, fdot = 10 ** rng.uniform(-23, -20), 10 ** rng.uniform(-4, -1), 10 ** rng.uniform(-20, -14)
        iota, phi0, psi = (float(x) for x in rng.uniform(0, 6.3, 3))
        rec, _ = w.gb_table(np.array([[A, f, fdot, iota, phi0, psi]]), [1234])
        assert w.gb_record(A, f, fdot, iota, phi0, psi, 1234) == rec.tobytes()
