"""The plain FP64 form's lanes per pixel and lanes in use (plain64_shape, host arithmetic): at every
size and depth where all shapes were timed, the rule takes one within a tenth of the fastest."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tinypt_amd", "csrc")
SHAPES = [(0, 64), (1, 64), (1, 32), (1, 16)]  # lanes per pixel one or four, lanes in use
# (levels of the deepest tree, pixels): ms of each shape on MI355X
TIMED = {
    (3, 4096): (5.12, 2.79, 2.48, 2.20), (3, 8281): (5.11, 2.84, 2.51, 2.50), (3, 12544): (5.14, 2.90, 2.88, 3.55),
    (3, 16384): (5.42, 2.90, 2.95, 4.08), (3, 23104): (5.29, 3.16, 4.17, 4.88), (3, 32761): (5.47, 3.28, 4.48, 6.22),
    (3, 46225): (4.10, 3.76, 4.50, 6.24), (3, 65536): (3.16, 3.28, 4.97, 7.35), (3, 262144): (1.49, 2.90, 4.20, 5.99),
    (6, 4096): (7.61, 4.55, 3.79, 3.45), (6, 8281): (7.62, 4.68, 4.11, 3.79), (6, 16384): (7.91, 4.76, 4.37, 4.64),
    (6, 23104): (8.13, 5.03, 4.14, 4.87), (6, 32761): (8.69, 5.02, 4.95, 5.87), (6, 46225): (6.32, 4.02, 4.41, 5.75),
    (6, 65536): (4.97, 3.71, 5.18, 6.73), (6, 131044): (2.57, 2.31, 3.30, 5.03), (6, 262144): (1.75, 3.03, 3.92, 5.39),
    (13, 8281): (14.65, 9.53, 7.73, 6.22), (13, 16384): (16.14, 9.78, 7.99, 7.44), (13, 23104): (17.52, 10.18, 7.96, 7.34),
    (13, 32761): (18.36, 10.17, 8.45, 9.11), (13, 46225): (14.64, 8.51, 7.05, 8.69), (13, 65536): (11.56, 7.05, 9.69, 12.07),
    (13, 131044): (5.39, 4.13, 5.33, 7.64), (13, 196249): (4.29, 4.55, 6.06, 8.53), (13, 262144): (3.43, 5.99, 7.26, 8.19),
    (17, 8281): (22.88, 14.67, 11.39, 9.04), (17, 16384): (26.35, 16.13, 12.58, 10.56), (17, 32761): (32.38, 17.43, 13.59, 12.66),
    (17, 46225): (24.82, 15.08, 11.41, 12.41), (17, 65536): (19.01, 11.94, 14.55, 17.41), (17, 196249): (8.22, 7.36, 8.96, 12.09),
    (17, 262144): (6.25, 9.81, 11.24, 11.77),
}


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("shape")
    src, exe = str(d / "shape.cpp"), str(d / "shape")
    with open(src, "w") as f:
        f.write('#include "plain64_shape.h"\n#include <cstdio>\n#include <cstdlib>\n'
                "int main(int, char** a) {\n"
                "  const auto s = tpt::plain64_shape(atoi(a[1]), atoll(a[2]));\n"
                '  printf("%d %d %d\\n", s.quads, s.lanes, s.mixed);\n}\n')
    subprocess.run([shutil.which("g++") or "g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, src, "-o", exe], check=True)
    return lambda depth, n: tuple(int(x) for x in subprocess.check_output([exe, str(depth), str(n)]).split())


@pytest.mark.parametrize("depth,pixels", sorted(TIMED))
def test_the_shape_taken_is_among_the_fastest(rule, depth, pixels):
    ms = dict(zip(SHAPES, TIMED[depth, pixels]))
    assert ms[rule(depth, pixels)[:2]] <= 1.1 * min(ms.values())


@pytest.mark.parametrize("depth", [0, 1, 4, 5, 6, 11, 16, 17, 63])
def test_shapes_are_ones_the_kernel_takes(rule, depth):
    for n in (1, 8192, 8193, 16384, 16385, 32768, 32769, 49152, 49153, 196608, 196609, 2**28):
        quads, lanes, mixed = rule(depth, n)
        assert (quads, lanes) in SHAPES and mixed == (depth >= 6)
