"""The exact stencils' two-operation quotients (csrc/flr_quotient.hpp) against a / b, bit for bit,
compiled for the host with g++ from the header the device code includes (no GPU needed).

Denominators are those of a stencil, F = j + e and G = j + (1 - e), e a multiple of the spacing of
doubles at the smallest position the form is used from; the reciprocal seed is the exact quotient
with errors up to 2^-22 planted. Numerators: random ones, and the hardest ones there are -- for a
denominator B (an odd integer times a power of two) a numerator A whose quotient lies 1 / (B M) of
itself from the midpoint M of two doubles, the least distance possible. A form without the
correction l (one product by the reciprocal) fails on both."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "lisa-on-gpu_amd", "csrc")

SHIM = r"""
static thread_local double seed_error;
#define FLR_HOST_DEVICE
#define FLR_RCP_SEED(x) ((1.0 / (x)) * (1.0 + seed_error))
#include "flr_quotient.hpp"
extern "C" int min_position(int h) { return flr::exact2_min_position(h); }
extern "C" int min_position4(int h) { return flr::exact4_min_position(h); }
// the same through recip_quad, each pair beside the one n/2 further on (parts: div_recip too, which
// order 25 takes)
extern "C" long check4(const double *a, const double *F, const double *G, const double *err, long n,
                       int parts)
{
    long wrong = 0;
    for (long i = 0; i + n / 2 < n; ++i) {
        seed_error = err[i];
        const long k = i + n / 2;
        flr::Recip f1, g1, f2, g2;
        flr::recip_quad(F[i], G[i], F[k], G[k], f1, g1, f2, g2);
        if (parts) {
            wrong += flr::div_recip(a[i], f1) != a[i] / F[i];
            wrong += flr::div_recip(a[i], g1) != a[i] / G[i];
            wrong += flr::div_recip(a[k], f2) != a[k] / F[k];
            wrong += flr::div_recip(a[k], g2) != a[k] / G[k];
        }
        wrong += flr::div_recip_y(a[i], F[i], f1) != a[i] / F[i];
        wrong += flr::div_recip_y(a[i], G[i], g1) != a[i] / G[i];
        wrong += flr::div_recip_y(a[k], F[k], f2) != a[k] / F[k];
        wrong += flr::div_recip_y(a[k], G[k], g2) != a[k] / G[k];
    }
    return wrong;
}
// wrong[0]: quotients of div_recip and div_recip_y that differ from a / b; wrong[1]: those of y a alone
extern "C" void check(const double *a, const double *F, const double *G, const double *err, long n,
                      long *wrong)
{
    wrong[0] = wrong[1] = 0;
    for (long i = 0; i < n; ++i) {
        seed_error = err[i];
        flr::Recip rF, rG;
        flr::recip_pair(F[i], G[i], rF, rG);
        wrong[0] += flr::div_recip(a[i], rF) != a[i] / F[i];
        wrong[0] += flr::div_recip(a[i], rG) != a[i] / G[i];
        wrong[0] += flr::div_recip_y(a[i], F[i], rF) != a[i] / F[i];
        wrong[0] += flr::div_recip_y(a[i], G[i], rG) != a[i] / G[i];
        wrong[1] += a[i] * rF.y != a[i] / F[i];
    }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("quotient")
    src = d / "shim.cpp"
    src.write_text(SHIM)
    so = d / "libshim.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC, str(src),
                    "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


def _check(lib, a, F, G, err):
    a, F, G, err = (np.ascontiguousarray(x, dtype=np.float64) for x in (a, F, G, err))
    wrong = (ctypes.c_long * 2)()
    lib.check(*(ctypes.c_void_p(x.ctypes.data) for x in (a, F, G, err)), ctypes.c_long(len(a)),
              wrong)
    return wrong[0], wrong[1]


def _check4(lib, a, F, G, err, h):
    a, F, G, err = (np.ascontiguousarray(x, dtype=np.float64) for x in (a, F, G, err))
    lib.check4.restype = ctypes.c_long
    return lib.check4(*(ctypes.c_void_p(x.ctypes.data) for x in (a, F, G, err)),
                      ctypes.c_long(len(a)), h <= 14)


def _denominators(rng, h, pos, n):
    """j + e, j + (1 - e) for j = 1 .. h-1 and e a multiple of ulp(pos) = 2^(log2(pos) - 52)."""
    bits = 52 - (pos.bit_length() - 1)
    e = rng.integers(0, 1 << bits, n).astype(np.float64) * 2.0 ** -bits
    j = rng.integers(1, h, n).astype(np.float64)
    F, G = j + e, j + (1.0 - e)
    assert np.array_equal(F - j, e)  # the sums are exact
    return F, G, bits


@pytest.mark.parametrize("h", [2, 8, 13, 16, 17, 20])
def test_random_numerators(lib, h):
    rng = np.random.default_rng(h)
    n = 400_000
    F, G, _ = _denominators(rng, h, lib.min_position(h), n)
    a = rng.standard_normal(n) * 10.0 ** rng.uniform(-30, 5, n)
    err = rng.uniform(-1, 1, n) * 2.0 ** -22
    two_ops, one_op = _check(lib, a, F, G, err)
    assert two_ops == 0
    assert one_op > n // 20  # the test can tell
    F, G, _ = _denominators(rng, h, lib.min_position4(h), n)  # from its own least position
    assert _check4(lib, a, F, G, err, h) == 0


@pytest.mark.parametrize("h,four", [(13, False), (16, False), (20, False), (13, True), (16, True), (20, True)])
def test_hardest_numerators(lib, h, four):
    rng = np.random.default_rng(100 + h)
    n = 20_000
    F, _, bits = _denominators(rng, h, (lib.min_position4 if four else lib.min_position)(h), n)
    a, Fk, Gk = [], [], []
    for f in F:
        B = int(f * 2.0 ** bits)
        B >>= (B & -B).bit_length() - 1
        s = B.bit_length() + 1  # quotient A 2^s / B near a 54-bit odd M
        if s < 3:
            continue
        inv = pow(B, -1, 1 << s)
        for r in (inv, (1 << s) - inv):  # B M = +-1 modulo 2^s
            M = r + ((int(rng.integers(1, 1 << 20)) | (1 << 20)) << s)
            drop = M.bit_length() - 54
            M = r + (((M >> s) >> drop) << s) if drop > 0 else M
            if not (1 << 53) <= M < (1 << 54):
                M = r + (((1 << 53) >> s) + 1 << s)
            if not ((1 << 53) <= M < (1 << 54)) or M % 2 == 0:
                continue
            A = (B * M + (1 if (B * M + 1) % (1 << s) == 0 else -1)) >> s
            if A >= 1 << 53:
                continue
            a.append(float(A))
            Fk.append(float(f))
            Gk.append(2.0 * np.floor(f) + 1.0 - f)
    assert len(a) > 2000
    err = rng.uniform(-1, 1, len(a)) * 2.0 ** -22
    if four:
        assert _check4(lib, np.array(a), np.array(Fk), np.array(Gk), err, h) == 0
        return
    two_ops, _ = _check(lib, np.array(a), np.array(Fk), np.array(Gk), err)
    assert two_ops == 0
