"""CPU checks of the index helpers of csrc/common.h at the limits of the
integer range.  A coordinate beyond it, or infinite, converts to the nearest
integer on the GPU, so that first taps of INT_MIN and INT_MAX do occur (a
diverged displacement under extrapolation).

The helpers are compiled for the host from the header itself."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
IMIN, IMAX = -2 ** 31, 2 ** 31 - 1


@pytest.fixture(scope="module")
def helpers(tmp_path_factory):
    """Runs a C++ expression over lines of integers a[0], a[1], ... on the
    host; signed overflow traps."""
    gxx = shutil.which("g++")
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    if gxx is None or not os.path.isdir(os.path.join(rocm, "include", "hip")):
        pytest.skip("needs g++ and the HIP headers")
    tmp = tmp_path_factory.mktemp("helpers")

    def run(expression, args):
        args = np.ascontiguousarray(args, dtype=np.int64)
        src, exe = tmp / "h.cpp", tmp / "h"
        src.write_text('#include "common.h"\n#include <cstdio>\nusing namespace ni_amd;\n'
                       f"int main() {{ long long a[{args.shape[1]}];\n"
                       f"  while (fread(a, sizeof a, 1, stdin) == 1) {{ long long r = {expression};\n"
                       "    fwrite(&r, sizeof r, 1, stdout); }\n  return 0; }\n")
        subprocess.run([gxx, "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-fsanitize=signed-integer-overflow",
                        "-fsanitize-undefined-trap-on-error", "-I", os.path.join(ROOT, "nitorch_amd", "csrc"),
                        "-I", os.path.join(rocm, "include"), str(src), "-o", str(exe)], check=True)
        done = subprocess.run([str(exe)], input=args.tobytes(), capture_output=True)
        assert done.returncode == 0, "the helper overflowed"
        return np.frombuffer(done.stdout, np.int64)
    return run


def test_axis_inside(helpers):
    firsts = [IMIN, IMIN + 1, IMIN + 64, -2, -1, 0, 1, 5, 60, 64, IMAX - 64, IMAX - 8, IMAX - 1, IMAX]
    args = np.array([(f, e, n) for f in firsts for e in (1, 2, 3, 4, 8, 17, 64) for n in (1, 2, 3, 8, 64, 65, IMAX)])
    out = helpers("axis_inside((int)a[0], (int)a[1], (int)a[2])", args)
    first, extent, n = args.T
    assert np.array_equal(out.astype(bool), (first >= 0) & (first + extent <= n))
