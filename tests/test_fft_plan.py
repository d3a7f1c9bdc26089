"""Radices 9, 10 and 15 of the HIP butterflies against the DFT definition, and
the radix plans of every length the transforms take, on the CPU."""
import ctypes as C
import os

import numpy as np
import pytest

import powerllel_channel_sycl_amd as pll

_LIB = os.path.join(os.path.dirname(pll.LIB_PATH), "libpll_selftest.so")


@pytest.mark.parametrize("radix", [9, 10, 15])
@pytest.mark.parametrize("sign", [-1, 1])
def test_butterfly_matches_dft_definition(radix, sign):
    lib = C.CDLL(_LIB)
    D = np.ctypeslib.ndpointer(dtype=np.float64, flags="C_CONTIGUOUS")
    lib.pll_selftest_dft.argtypes = [C.c_int, C.c_int, D, D]
    rng = np.random.default_rng(radix * 7 + sign)
    z = rng.standard_normal(radix) + 1j * rng.standard_normal(radix)
    inp, out = np.empty(2 * radix), np.empty(2 * radix)
    inp[0::2], inp[1::2] = z.real, z.imag
    assert lib.pll_selftest_dft(radix, sign, inp, out) == 0
    n = np.arange(radix, dtype=np.longdouble)
    w = np.exp(1j * np.mod(np.outer(n, n), radix) * (sign * 2 * np.pi / np.longdouble(radix)))
    ref = w @ z.astype(np.clongdouble)
    assert np.max(np.abs(out[0::2] + 1j * out[1::2] - ref)) < 4e-15 * np.max(np.abs(ref))


def _smooth(n):
    for p in (2, 3, 5):
        while n % p == 0:
            n //= p
    return n == 1


def test_every_length_has_a_plan():
    lib = C.CDLL(_LIB)
    rad = (C.c_int * 8)()
    for n in filter(_smooth, range(2, 4097)):
        k = lib.pll_selftest_plan(n, 1024, rad)
        got = list(rad[:k])
        assert k >= 1 and int(np.prod(got)) == n, (n, got)
        assert set(got) <= {2, 3, 4, 5, 6, 8, 9, 10, 12, 15, 16} and n // min(got) <= 1024, (n, got)
    assert lib.pll_selftest_plan(7, 1024, rad) == 0
