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


def fold_reference(bound, i, n):
    """Index and sign of voxel i under a bound's periodic extension, from the
    definition, in exact integers."""
    if 0 <= i < n:
        return i, 1
    if bound == 0:
        return min(max(i, 0), n - 1), 1
    if bound == 1:
        k = i % (2 * n - 2) if n > 1 else 0
        return (k, 1) if k < n else (2 * n - 2 - k, 1)
    if bound in (2, 4):
        k = i % (2 * n)
        return (k, 1) if k < n else (2 * n - 1 - k, 1 if bound == 2 else -1)
    if bound == 3:
        if n == 1:
            return 0, 1
        k = i % (2 * n + 2)
        if k in (n, 2 * n + 1):
            return 0, 0
        return (k, 1) if k < n else (2 * n - k, -1)
    return (i % n, 1) if bound == 5 else (0, 0)


@pytest.mark.parametrize("width", [32, 64])
def test_fold(helpers, width):
    lo, hi = -2 ** (width - 1), 2 ** (width - 1) - 1
    ends = list(range(70)) + [97, 100, 1000, 65535, 10 ** 6]
    at = sorted(set([lo + e for e in ends] + [hi - e for e in ends] + list(range(-200, 201))))
    args = np.array([(b, i, n) for b in range(9) for n in list(range(1, 13)) + [16, 30, 32, 62, 97, 181, 2 ** 30 + 1]
                     for i in at])
    kind = "int" if width == 32 else "int64_t"
    out = helpers(f"({{ int s; long long j = fold<{kind}>((int)a[0], ({kind})a[1], ({kind})a[2], s);"
                  " j * 4 + s + 1; })", args)
    ref = [4 * j + s + 1 for j, s in (fold_reference(*(int(v) for v in row)) for row in args)]
    assert np.array_equal(out, np.array(ref))
    n = args[:, 2]
    assert ((out >> 2 >= 0) & (out >> 2 < n)).all()


def test_tap_at(helpers):
    args = np.array([(f, t) for f in (IMIN, -1, 0, 7, IMAX - 7, IMAX) for t in range(8)])
    out = helpers("tap_at((int)a[0], (int)a[1])", args)
    assert np.array_equal(out, (args.sum(1) + 2 ** 31) % 2 ** 32 - 2 ** 31)


def test_place_in(helpers):
    """The range test of the first-tap bins."""
    at = [IMIN, IMIN + 1, IMIN + 8, -9, -8, -1, 0, 1, 7, 23, 24, 183, 184, IMAX - 8, IMAX - 7, IMAX - 1, IMAX]
    args = np.array([(i, 8, n) for i in at for n in (8, 32, 192, 2 ** 20)])
    out = helpers("place_in((int)a[0], (int)a[1], (int)a[2])", args)
    place = args[:, 0] + args[:, 1]
    assert np.array_equal(out, np.where((place >= 0) & (place < args[:, 2]), place, -1))


def test_bound_signs(helpers):
    args = np.array([(b, i, 5) for b in range(9) for i in range(-40, 41)])
    sign = helpers("({ int s; fold<int>((int)a[0], (int)a[1], (int)a[2], s); (long long)s; })", args).reshape(9, -1)
    named = helpers("bound_signs((int)a[0])", np.arange(9)[:, None])
    assert np.array_equal(named.astype(bool), (sign != 1).any(1))
