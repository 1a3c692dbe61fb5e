"""lut_rest (csrc/wr_math.h), the two values of the LW look-up table that the FP64 kernels evaluate instead of loading.

The function's own source is compiled for the CPU, with the hardware's reciprocal estimate replaced by 1 / x off by a
given relative error, and must give the oracle's table (the device's, by the same operations) bit for bit at every index."""
import ctypes as C
import re
import subprocess
from pathlib import Path

import numpy as np
import pytest

from oracle import pyoracle

HEADER = Path(__file__).resolve().parents[1] / "woof_nam_amd" / "csrc" / "wr_math.h"
NTBL = 10000


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    m = re.search(r"__device__ __forceinline__ void lut_rest\(.*?\n}\n", HEADER.read_text(), re.S)
    d = tmp_path_factory.mktemp("lut_rest")
    (d / "lut.cpp").write_text("""
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_rcp estimate
static double off;
static double estimate(double x) { return (1.0 / x) * (1.0 + off); }
""" + m.group(0) + """
extern "C" void run(double err, int ntbl, const double *e, double *tfn, double *tau)
{
    off = err;
    for (int i = 1; i <= ntbl; ++i) lut_rest(i, ntbl, e[i], tfn[i], tau[i]);
}
""")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-w", "-shared", "-fPIC", "-o", str(d / "lut.so"),
                    str(d / "lut.cpp")], check=True)
    return C.CDLL(str(d / "lut.so"))


# the reciprocal's documented error is far below 2^-22; two Newton steps take that to rounding
@pytest.mark.parametrize("err", [0.0, 2.0 ** -22, -2.0 ** -22, 2.0 ** -24, -2.0 ** -24, 2.0 ** -27, -2.0 ** -30])
def test_every_index_equals_the_table(lib, err):
    e, tfn, tau = (np.ascontiguousarray(x, dtype=np.float64) for x in pyoracle.lw_tables())
    got = np.zeros((2, NTBL + 1))
    dp = C.POINTER(C.c_double)
    lib.run(C.c_double(err), NTBL, e.ctypes.data_as(dp), got[0].ctypes.data_as(dp), got[1].ctypes.data_as(dp))
    for g, ref in ((got[0], tfn), (got[1], tau)):
        assert np.array_equal(g[1:].view(np.int64), ref[1:].view(np.int64))
