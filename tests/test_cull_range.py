"""The FP32 cull over the range of a double, on the host: wherever it gives a
verdict it is the FP64 test's, and at ordinary sizes it nearly always does."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))

# What the device headers need of the HIP runtime in a host program.
HIP = """#pragma once
#include <cmath>
#include <cstddef>
#include <cstdint>
#define __device__
#define __forceinline__ inline
#define __noinline__
struct alignas(16) uint4 { unsigned x, y, z, w; };
"""


def test_every_verdict_is_the_fp64_tests(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    exe = str(tmp_path / "cull32")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-Wno-unknown-pragmas",
                    "-I", str(tmp_path), os.path.join(HERE, "cpp", "test_cull32.cpp"), "-o", exe],
                   check=True)
    pairs = 20000
    out = subprocess.run([exe, str(pairs)], check=True, stdout=subprocess.PIPE, text=True).stdout
    rows = [[float(x) for x in line.split()] for line in out.splitlines()]
    assert rows[0][0] == -320 and rows[-1][0] > 300 and any(r[0] == 0 for r in rows)
    for exponent, sure, unsure, wrong in rows:
        assert sure + unsure + wrong == pairs
        assert wrong == 0, "sizes of 1e%g: %d wrong verdicts" % (exponent, wrong)
        if abs(exponent) <= 20:
            assert sure > 0.999 * pairs
