"""The controller's correctly rounded root (csrc/crpow.hpp, cr_root) on the CPU."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HEADER = os.path.join(HERE, "..", "ode_prototyping_amd", "csrc", "crpow.hpp")

SOURCE = """
#include "%s"
#include <quadmath.h>
extern "C" void roots(const double* x, long n, int k, double* root, double* pow, double* quad) {
  const double y = 1.0 / k;
  for (long i = 0; i < n; ++i) {
    root[i] = odehip::cr_root(x[i], y, k);
    pow[i] = odehip::cr_pow(x[i], y);
    quad[i] = static_cast<double>(powq(static_cast<__float128>(x[i]), static_cast<__float128>(y)));
  }
}
"""


@pytest.fixture(scope="module")
def roots(tmp_path_factory):
    d = tmp_path_factory.mktemp("root")
    src, so = str(d / "root.cpp"), str(d / "root.so")
    with open(src, "w") as f:
        f.write(SOURCE % HEADER)
    subprocess.run(["g++", "-std=c++20", "-O2", "-ffp-contract=off", "-fPIC", "-shared", src,
                    "-lquadmath", "-o", so], check=True)
    fn = ctypes.CDLL(so).roots
    p = ctypes.POINTER(ctypes.c_double)

    def call(x, k):
        out = [np.empty_like(x) for _ in range(3)]
        fn(x.ctypes.data_as(p), ctypes.c_long(x.size), k, *[o.ctypes.data_as(p) for o in out])
        return out
    return call


@pytest.mark.parametrize("k", [2, 3, 5, 6, 8, 9, 13, 21])
def test_root_equals_pow_and_binary128(roots, k):
    """Scaled errors as a controller meets them, the whole range, neighbours of 1, and
    exact powers: the same double as cr_pow and as binary128's pow rounded."""
    rng = np.random.default_rng(k)
    x = np.concatenate([np.exp(rng.uniform(-25.0, 10.0, 2000)),
                        np.exp2(rng.uniform(-1021.0, 1023.0, 1000)),
                        1.0 + rng.uniform(-1e-9, 1e-9, 500), [1.0, 0.38, 1e-300, 1e300],
                        np.arange(1.0, 6.0) ** min(k, 9)])
    root, pw, quad = roots(np.ascontiguousarray(x), k)
    assert np.array_equal(root, pw)
    assert np.array_equal(root, quad)


def test_root_special_inputs(roots):
    x = np.array([0.0, 5e-324, np.inf, np.nan, -1.0])
    root, pw, _ = roots(x, 6)
    assert np.array_equal(root, pw, equal_nan=True)
