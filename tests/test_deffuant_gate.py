"""The short form of the Deffuant gate (csrc/deffuant_gate.hpp), compiled for
the CPU, against the gate's own operations: IEEE division and abm_expf."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "deffuant_gate.hpp"
#include <cstring>

static float value(uint32_t b) { float f; memcpy(&f, &b, 4); return f; }
static int32_t bits(float f) { int32_t b; memcpy(&b, &f, 4); return b; }
// an estimate of 1 / d that is `off` steps from the rounded one, where it may be
static float estimate(float d, int off) {
  return value((uint32_t)(bits(1.0f / d) + ((bits(d) & 0x7fffff) == 0x7fffff ? 0 : off)));
}

// Largest distance in float32 steps between the quotients over the floats
// [lo, hi] (bit patterns), every `stride`-th.
extern "C" int32_t quotients(uint32_t lo, uint32_t hi, uint32_t stride) {
  int32_t worst = 0;
#pragma omp parallel for reduction(max : worst)
  for (int64_t b = lo; b <= (int64_t)hi; b += stride) {
    const float x = value((uint32_t)b);
    const int32_t d = bits(abm::div_gate_scale(x)) - bits(x / abm::kGateScale);
    const int32_t e = bits(abm::div_gate_scale(-x)) - bits(-x / abm::kGateScale);
    const int32_t m = (d < 0 ? -d : d) | (e < 0 ? -e : e);
    worst = m > worst ? m : worst;
  }
  return worst;
}

// Reciprocals of [lo, hi] that differ from 1 / d, from estimates up to 1 ulp off.
extern "C" int64_t reciprocals(uint32_t lo, uint32_t hi, uint32_t stride) {
  int64_t bad = 0;
#pragma omp parallel for reduction(+ : bad)
  for (int64_t b = lo; b <= (int64_t)hi; b += stride) {
    const float d = value((uint32_t)b), want = 1.0f / d;
    for (int off = -1; off <= 1; ++off)
      bad += abm::inv_rounded(d, estimate(d, off)) != want;
  }
  return bad;
}

// Gates of +-[lo, hi] whose short form differs.
extern "C" int64_t gates(uint32_t lo, uint32_t hi, uint32_t stride) {
  int64_t bad = 0;
#pragma omp parallel for reduction(+ : bad)
  for (int64_t b = lo; b <= (int64_t)hi; b += stride)
    for (int sign = 0; sign < 2; ++sign) {
      const float num = sign ? -value((uint32_t)b) : value((uint32_t)b);
      const float want = abm::gate(num, 0.0f);
      for (int off = -1; off <= 1; ++off) {
        const float g = abm::gate_short(num, [off](float d) { return estimate(d, off); });
        bad += bits(g) != bits(want);
      }
    }
  return bad;
}
"""


def _bits(x):
    import numpy as np

    return int(np.float32(x).view(np.uint32))


def _power(e):
    return (e + 127) << 23


@pytest.fixture(scope="module")
def gate(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("needs a host C++ compiler")
    d = tmp_path_factory.mktemp("gate")
    src, so = d / "gate.cpp", d / "gate.so"
    src.write_text(SOURCE)
    subprocess.run([cxx, "-std=c++17", "-O3", "-march=native", "-ffp-contract=off", "-fopenmp",
                    "-shared", "-fPIC", "-I", os.path.join(REPO, "jaxabm_amd", "csrc"), str(src),
                    "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    for f in (lib.quotients, lib.reciprocals, lib.gates):
        f.argtypes = [C.c_uint32] * 3
    lib.reciprocals.restype = lib.gates.restype = C.c_int64
    return lib


def test_quotient_is_the_rounded_one(gate):
    """Every float of [2^-105, 2^-103) and [2^-8, 1.6], and every 31st between
    (the operations scale exactly there); below, one step off at most."""
    assert gate.quotients(_power(-105), _power(-103), 1) == 0
    assert gate.quotients(_power(-103), _power(-8), 31) == 0
    assert gate.quotients(_power(-8), _bits(1.6), 1) == 0
    assert gate.quotients(0, _power(-105), 31) == 1


@pytest.mark.parametrize("exponent", [0, 1, 24, 60, 86, 119])
def test_reciprocal_is_the_rounded_one(gate, exponent):
    assert gate.reciprocals(_power(exponent), _power(exponent + 1) - 1, 1) == 0


def test_short_gate_has_the_same_bits(gate):
    """Every |eps - |d|| of [2^-8, 1.2], the end of the short form, and every
    31st below."""
    assert gate.gates(_power(-8), _bits(1.2), 1) == 0
    assert gate.gates(0, _power(-8), 31) == 0
