"""exp_nonpositive (nvr_attention.h), compiled for the host from the header's own
text, against the oracle's expf, bit for bit: every float from -87 to -128 (the
results that are subnormal or round to zero), one in 41 of the rest from -0 to
-infinity, and NaN."""
import ctypes
import os
import re
import subprocess

import numpy as np

import oracle as ora

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-rs_amd", "csrc")

SHIM = """#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#define __device__
#define __forceinline__ inline
static float __uint_as_float(uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }
"""
LOOP = """
extern "C" void run(const float* x, float* y, size_t n) { for (size_t i = 0; i < n; ++i) y[i] = exp_nonpositive(x[i]); }
"""


def _function(header: str, name: str) -> str:
    return re.search(rf"^__device__ __forceinline__ float {name}\(.*?(?:}}  //[^\n]*|^}})$",
                     open(os.path.join(CSRC, header)).read(), re.S | re.M).group(0)


def test_exp_nonpositive_has_the_bits_of_expf(tmp_path):
    source, lib = tmp_path / "exp.cpp", tmp_path / "exp.so"
    source.write_text(SHIM + _function("nvr_device.h", "pow2i") + "\n" + _function("nvr_attention.h", "exp_nonpositive")
                      + LOOP)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-o", lib, source], check=True)
    run = ctypes.CDLL(str(lib)).run
    run.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]

    first, last = (int(np.float32(x).view(np.uint32)) for x in (-87.0, -128.0))
    bits = np.concatenate([np.arange(0x80000000, 0xFF800001, 41, dtype=np.uint32),
                           np.arange(first, last + 1, dtype=np.uint32),
                           np.array([0x80000000, 0xFF800000, 0x7FC00000, 0xFFC00000], np.uint32)])
    x = bits.view(np.float32)
    got = np.empty_like(x)
    run(x.ctypes.data, got.ctypes.data, x.size)
    want = np.asarray(ora.expf_array(x), np.float32)
    nan = np.isnan(want)
    assert nan.sum() == 2 and np.isnan(got[nan]).all()
    assert (want == 0).any() and ((want > 0) & (want < 2.0 ** -126)).any()
    assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))
