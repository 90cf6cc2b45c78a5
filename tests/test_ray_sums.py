"""The samples' positions a whole segment ahead (csrc/ray_sums.h), compiled for the host: equal
to the running sum p = p + d, each addition rounded, over binades, zero and long marches."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spimagine_amd", "csrc")
PROGRAM = r"""
#include <cmath>
#include <cstdint>
#include <cstring>
#define __device__
#define __forceinline__ inline
static inline uint32_t __float_as_uint(float v) { uint32_t u; std::memcpy(&u, &v, 4); return u; }
static inline float __uint_as_float(uint32_t u) { float v; std::memcpy(&v, &u, 4); return v; }
static inline float __builtin_amdgcn_rcpf(float v) { return 1.0f / v; }
#include "ray_sums.h"
extern "C" void sums(const float* p, const float* d, const uint32_t* n, float* out, int count) {
    for (int i = 0; i < count; ++i) out[i] = spr::sum_n(p[i], d[i], n[i]);
}
"""


@pytest.fixture(scope="module")
def sum_n(tmp_path_factory):
    at = tmp_path_factory.mktemp("sums")
    (at / "sums.cpp").write_text(PROGRAM)
    lib = str(at / "sums.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-mfma", "-ffp-contract=off", "-shared", "-fPIC",
                           "-I", CSRC, "-o", lib, str(at / "sums.cpp")])
    f = ctypes.CDLL(lib).sums

    def call(p, d, n):
        p, d = np.ascontiguousarray(p, np.float32), np.ascontiguousarray(d, np.float32)
        n, out = np.ascontiguousarray(n, np.uint32), np.empty(len(p), np.float32)
        f(*[ctypes.c_void_p(a.ctypes.data) for a in (p, d, n, out)], ctypes.c_int(len(p)))
        return out
    return call


def running(p, d, n):
    q = p.copy()
    for k in range(int(n.max())):
        q = np.where(k < n, q + d, q)
    return q


@pytest.mark.parametrize("reach", [1.1, 40.])
def test_sums_over_binades_and_zero(sum_n, reach):
    rng = np.random.default_rng(int(reach))
    m = 20000
    p = rng.uniform(-reach, reach, m).astype(np.float32)
    p[::5] = (rng.integers(0, 64, p[::5].size) / 64.).astype(np.float32)  # powers of two among them
    d = (rng.uniform(-1, 1, m) * reach * 2. ** -rng.integers(1, 13, m)).astype(np.float32)
    u = d.view(np.uint32)
    u[::2] &= ~((1 << rng.integers(0, 20, u[::2].size)) - 1).astype(np.uint32)  # few bits: ties
    d[::11] = 0.
    n = rng.integers(0, 2000, m)
    n[::3] = rng.integers(0, 40, n[::3].size)
    np.testing.assert_array_equal(sum_n(p, d, n).view(np.uint32), running(p, d, n).view(np.uint32))


# past 2^24 steps a count less three has no float32 of its own
@pytest.mark.parametrize("p,d,n", [(-7.9, 1.7e-6, (1 << 24) + 8), (.4, 3e-9, 3 << 23),
                                   (9.5, -7.3e-7, (1 << 24) + 2048), (-.9, 5.2e-8, 5 << 22)])
def test_sums_of_long_marches(sum_n, p, d, n):
    p, d = np.float32(p), np.float32(d)
    steps = np.full(n + 1, d, np.float32)
    steps[0] = p
    want = np.add.accumulate(steps, dtype=np.float32)[-1]
    got = sum_n([p], [d], [n])[0]
    assert got == want, (got, want)
