"""The library's plan of a convolution (csrc/mmnb_conv_plan.h), built for the host and
called from Python."""
import ctypes
import functools
import shutil
import subprocess
import tempfile
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "onnx_runtime_dart_amd" / "csrc"
SHIM = """
#include "mmnb_conv_plan.h"
extern "C" void plan(int64_t P, int64_t K, int64_t N, int64_t z, int64_t cus, int64_t *o) {
  const mmnb::ConvPlan p = mmnb::conv_plan(P, K, N, z, cus);
  const int64_t v[] = {p.taps, p.nw, p.nper, p.pt, p.cw, p.threads, p.gx, p.gy, p.step};
  for (int i = 0; i < 9; i++) o[i] = v[i];
}
"""
FIELDS = "taps nw nper pt cw threads gx gy step".split()


@functools.lru_cache(None)
def _lib():
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    d = Path(tempfile.mkdtemp(prefix="conv_plan"))
    (d / "plan.cpp").write_text(SHIM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-I", str(CSRC),
                    str(d / "plan.cpp"), "-o", str(d / "plan.so")], check=True)
    return ctypes.CDLL(str(d / "plan.so"))


def plan(P, K, N, z, cus=256):
    out = (ctypes.c_int64 * 9)()
    _lib().plan(*(ctypes.c_int64(v) for v in (P, K, N, z, cus)), out)
    return dict(zip(FIELDS, out))
