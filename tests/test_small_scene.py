"""Which scenes the small-scene kernels take (small_scene.h, host arithmetic).  They address a scene's
nodes and triangles where these lie in the scene's own arrays, by 32-bit signed byte offsets, so a
small flattened tree behind the large trees of meshes that no instance uses has to stay with the
kernels for device memory."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tinypt_amd", "csrc")


@pytest.fixture(scope="module")
def asked(tmp_path_factory):
    d = tmp_path_factory.mktemp("small")
    src, exe = str(d / "small.cpp"), str(d / "small")
    with open(src, "w") as f:
        f.write('#include "small_scene.h"\n#include <cstdio>\n#include <cstdlib>\n'
                "int main(int, char** a) {\n"
                "  auto n = [&](int i) { return (uint32_t)strtoul(a[i], nullptr, 10); };\n"
                "  tpt::SmallScene m{};\n"
                "  m.node0 = n(1); m.n_nodes = n(2); m.tri0 = n(3); m.n_tris = n(4);\n"
                '  printf("%d\\n", (int)tpt::small_scene_addressable(m));\n}\n')
    subprocess.run([shutil.which("g++") or "g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, src, "-o", exe], check=True)
    return lambda *v: subprocess.check_output([exe] + [str(x) for x in v]).strip() == b"1"


@pytest.mark.parametrize("first,count,size,nodes", [(19_173_961, 12, 112, True), (44_739_242, 36, 48, False)])
def test_scenes_beyond_signed_offsets_are_not_small(asked, first, count, size, nodes):
    args = (lambda k: (k, count, 0, 36)) if nodes else (lambda k: (0, 12, k, count))
    last = (2**31 - 1) // size - count  # the last place from which every byte offset is below 2^31
    assert first - count <= last < first
    assert asked(*args(0)) and asked(*args(last))
    for k in (last + 1, first, 2 * first, 2**25 if nodes else 2**28 - 1, 2**32 - 1):
        assert not asked(*args(k))
