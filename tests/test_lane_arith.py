"""The 28-bit lane arithmetic of the G1 kernels (csrc/fp_lane28.hpp) compiled for the host: the
bounds that its comments state, at their edges, against Python integers.  No GPU is needed."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import pyg1 as G

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zk-hillclimb_amd", "csrc")
SHIM = r"""
#define FDEV __host__ __device__ inline
#include "fp_lane28.hpp"
static f28_t in(const int32_t* p) { f28_t r; for (int i = 0; i < 14; i++) r.v[i] = p[i]; return r; }
extern "C" {
void store_point(uint32_t* w, const int32_t* x, const int32_t* y, const int32_t* z, int inf) {
    g28_store(w, g28_t{in(x), in(y), in(z)}, inf != 0);
}
void copy_point(uint32_t* w) { bool inf; const g28_t a = g28_load(w, inf); g28_store(w, a, inf); }
int is_zero(const int32_t* x) { return f28_zero(in(x)); }
uint32_t from_words(int32_t* r, const uint32_t* w) {
    uint32_t any;
    const f28_t t = f28_from_words(w, any);
    for (int i = 0; i < 14; i++) r[i] = t.v[i];
    return any;
}
void to_words(uint32_t* w, const int32_t* x) { f28_to_words(w, in(x)); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("lane")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-x", "hip", "--cuda-host-only",
                    "--offload-arch=gfx950", "-O1", "-fPIC", "-shared", "-I", CSRC, str(d / "shim.cpp"), "-o",
                    str(d / "shim.so")], check=True, capture_output=True)
    return ctypes.CDLL(str(d / "shim.so"))


def limbs(v):
    """14 limbs of 28 bits, the top one signed"""
    return np.array([(v >> (28 * i)) & 0xFFFFFFF for i in range(13)] + [v >> 364], np.int32)


def value(w):
    return sum(int(w[i]) << (28 * i) for i in range(14))


def ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def test_stored_points_keep_their_bounds(lib):
    """x, y below 45 p and z below 36 p with carried nonnegative limbs (the row form's bounds),
    the same residue: negative values, and values that are only copied, however often."""
    rng = np.random.default_rng(28)
    rnd = lambda lo, hi: int(lo * G.P) + int.from_bytes(rng.bytes(64), "little") % int((hi - lo) * G.P)
    pts = [(rnd(-17, 45), rnd(-17, 45), rnd(-1, 36)) for _ in range(200)]
    pts += [(-17 * G.P + 1, 45 * G.P - 1, 36 * G.P - 1), (0, -1, 0), (-1, 0, -G.P + 1), (45 * G.P - 1, 1, -1)]
    for x, y, z in pts:
        for inf in (0, 1):
            w = np.zeros(48, np.uint32)
            lib.store_point(ptr(w), ptr(limbs(x)), ptr(limbs(y)), ptr(limbs(z)), inf)
            for _ in range(4):
                for v, k, bound in ((x, 0, 45), (y, 1, 45), (z, 2, 36)):
                    c = w[16 * k:16 * k + 16]
                    assert (c[:13] < 1 << 28).all()
                    assert value(c) < bound * G.P and (value(c) - v) % G.P == 0
                assert w[14] == inf and not w[15] and not w[30:32].any() and not w[46:48].any()
                lib.copy_point(ptr(w))


def test_zero_test_range(lib):
    """f28_zero over (-32 p, 64 p): every multiple of p there, and nothing beside one."""
    for j in range(-31, 64):
        assert lib.is_zero(ptr(limbs(j * G.P))), j
        for d in (-1, 1, 1 << 28, -(1 << 200)):
            assert not lib.is_zero(ptr(limbs(j * G.P + d))), (j, d)


def test_words_of_a_coordinate(lib):
    """Canonical words to R' = 2^392 residues below 3 p, and any value in (-45 p, 45 p) back to
    canonical words: 0, 1, p - 1, single bits, multiples of p and random ones."""
    rng = np.random.default_rng(144)
    vals = [0, 1, G.P - 1, G.P - 2, 1 << 380] + [1 << i for i in range(0, 380, 7)]
    vals += [int.from_bytes(rng.bytes(48), "little") % G.P for _ in range(100)]
    for v in vals:
        w, t = G.limbs12(v), np.zeros(14, np.int32)
        assert (lib.from_words(ptr(t), ptr(w)) != 0) == (v != 0)
        assert 0 <= value(t) < 3 * G.P and (value(t) - (v << 8)) % G.P == 0 and (t[:13] < 1 << 28).all()
        for j in (-44, -17, -1, 0, 1, 36, 44):
            x = v * (1 << 8) % G.P + j * G.P
            back = np.zeros(12, np.uint32)
            lib.to_words(ptr(back), ptr(limbs(x)))
            assert np.array_equal(back, w), (v, j)
