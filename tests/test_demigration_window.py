"""The sample window of a trace that an image tile reaches
(seisfat2d_amd/csrc/kdm_window.h), compiled for the host: it holds exactly the
samples of the record among the tile's time indices, for least and greatest
traveltime sums up to "not reached" values whose index lies beyond 32 bits."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INT_MAX = 2**31 - 1


@pytest.fixture(scope="module")
def window(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    tmp = tmp_path_factory.mktemp("window")
    src, so = tmp / "w.cpp", tmp / "w.so"
    src.write_text('#include "kdm_window.h"\n'
                   'extern "C" void window(int lo, int hi, int nt, int* out) {\n'
                   '  const seisfat::SampleWindow w = seisfat::sample_window(lo, hi, nt);\n'
                   '  out[0] = w.first;\n  out[1] = w.len;\n}\n')
    # a signed wrap ends the process
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fsanitize-undefined-trap-on-error", "-shared",
                    "-fPIC", "-I", os.path.join(ROOT, "seisfat2d_amd", "csrc"), "-o", str(so), str(src)], check=True)
    f = C.CDLL(str(so)).window

    def call(lo, hi, nt):
        out = (C.c_int * 2)()
        f(lo, hi, nt, out)
        return out[0], out[1]
    return call


def index(x, dt, nt):
    """A node's time index as the kernels take it: the floor of the float
    quotient, saturated (nt for an infinite one), -1 for every negative one."""
    with np.errstate(over="ignore"):
        v = np.floor(np.float32(x) / np.float32(dt))
    return nt if np.isinf(v) else int(min(max(float(v), -1.0), INT_MAX))


@pytest.mark.parametrize("dt", [4e-3, 9e-4, 1e-5])
@pytest.mark.parametrize("nt", [1, 400, 16384])
def test_window_holds_the_records_samples(window, nt, dt):
    end = nt * dt
    least = [-1.0, -0.4 * dt, 0.0, 0.4 * dt, 0.5 * end, end - 0.6 * dt]
    greatest = least + [end + 0.6 * dt, 2.0**31 * dt, 2.0**32 * dt, 2e6, 1e9, 1e30, 3e38, np.inf]
    for lo in least:
        for hi in greatest:
            if hi < lo:
                continue
            i, j = index(lo, dt, nt), index(hi, dt, nt)
            first, n = window(i, j, nt)
            samples = [k for k in (max(i, 0), min(j, nt - 1)) if 0 <= k < nt and i <= k <= j]
            if not samples:
                assert n <= 0, (lo, hi)
            else:
                assert (first, first + n - 1) == (samples[0], samples[-1]), (lo, hi)
                assert first >= 0 and first + n <= nt
