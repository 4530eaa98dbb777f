"""The sine and cosine of the 16-bit forms' positional encoding
(sailor_amd/csrc/pe_sincos.h), built for the host from the same source, against
64-bit values.  The bounds are the header's: half an ulp of the result (3.0e-8
below 1) for the last rounding, at most as much for those before it, and 1.9e-9 for
the polynomial; rms as of the library's sine, 1.8e-8."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sailor_amd",
                    "csrc")


@pytest.fixture(scope="module")
def sincos(tmp_path_factory):
    d = tmp_path_factory.mktemp("pe_sincos")
    src = d / "pe.cpp"
    src.write_text("""
#define SAILOR_PE_FN static inline
#include "pe_sincos.h"
extern "C" void pe(const float* x, float* s, float* c, int n) {
  for (int i = 0; i < n; ++i) sailor::pe_sincos(x[i], s[i], c[i]);
}
""")
    so = str(d / "pe.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC,
                    str(src), "-o", so], check=True)
    fn = ctypes.CDLL(so).pe
    p = np.ctypeslib.ndpointer(np.float32, flags="C_CONTIGUOUS")
    fn.argtypes = [p, p, p, ctypes.c_int]

    def run(x):
        x = np.ascontiguousarray(x, np.float32)
        s, c = np.empty_like(x), np.empty_like(x)
        fn(x, s, c, x.size)
        return s, c
    return run


@pytest.mark.parametrize("limit", [1e-3, 1.0, 32.0, 512.0, 8192.0])
def test_errors_against_64_bits(sincos, limit):
    rng = np.random.default_rng(int(limit * 1000))
    x = rng.uniform(-limit, limit, 400000).astype(np.float32)
    # and the neighbourhood of every multiple of pi/4, where signs and the
    # choice of polynomial change
    k = np.unique(rng.integers(0, int(limit / (np.pi / 4)) + 1, 20000))
    near = (k * (np.pi / 4)).astype(np.float32)
    x = np.concatenate([x, near, np.nextafter(near, np.float32(np.inf)), -near])
    x = x[np.abs(x) <= 8192.0]
    for got, want in zip(sincos(x), (np.sin(x.astype(np.float64)), np.cos(x.astype(np.float64)))):
        err = np.abs(got.astype(np.float64) - want)
        print(f"|x| <= {limit}: rms {np.sqrt((err ** 2).mean()):.2e}, max {err.max():.2e}")
        assert err.max() <= 6.6e-8 and np.sqrt((err ** 2).mean()) <= 1.8e-8


def test_special_values(sincos):
    s, c = sincos(np.float32([0.0, -0.0, 2.0 ** -30, -(2.0 ** -30)]))
    assert np.array_equal(s, np.float32([0.0, 0.0, 2.0 ** -30, -(2.0 ** -30)]))
    assert np.array_equal(c, np.ones(4, np.float32))
