"""The kernels' two shortened roundings (quant_one in nh_device.h, round_digits
in nh_forward.hip), compiled from the library's source with g++, against
roundf: every one of the 2^32 floats, and every float of the digits' range."""
import os
import shutil
import subprocess

import pytest

from test_span_runs import SRC, _grab

MAIN = r"""
int main() {
    long bad = 0, digits = 0;
#pragma omp parallel for schedule(static) reduction(+ : bad, digits)
    for (long b = 0; b < (1L << 32); ++b) {
        const uint32_t u = (uint32_t)b;
        float v;
        std::memcpy(&v, &u, 4);
        // (v.round().clamp(-128, 127) as the kernels take it: a NaN gives -128)
        const float r = roundf(v);
        const int8_t want = r >= 127.0f ? 127 : r >= -128.0f ? (int8_t)(int)r : -128;
        bad += quant_one(v, 1.0f) != want;
        if (v >= 0.0f && v < 4194304.0f) {
            bad += round_digits(v) != (int32_t)r;
            ++digits;
        }
    }
    std::printf("%ld of the digits' floats, %ld differ\n", digits, bad);
    return bad != 0 || digits < 1000000000L;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_float(tmp_path):
    dev = open(os.path.join(os.path.dirname(SRC), "nh_device.h")).read()
    code = "".join([
        "#include <cmath>\n#include <cstdint>\n#include <cstdio>\n#include <cstring>\n",
        _grab(dev, "__device__ __forceinline__ int8_t quant_one("),
        _grab(open(SRC).read(), "__device__ __forceinline__ int32_t round_digits(", "}\n"),
        MAIN,
    ]).replace("__device__ __forceinline__", "inline")
    cpp, exe = tmp_path / "round.cpp", tmp_path / "round"
    cpp.write_text(code)
    subprocess.run(["g++", "-O2", "-std=c++17", "-fopenmp", "-ffp-contract=off", str(cpp), "-o", str(exe)], check=True,
                   capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=115)
    assert r.returncode == 0, r.stdout + r.stderr
