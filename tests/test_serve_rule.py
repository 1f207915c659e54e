"""Where a serving step from a slot map runs its decodes (csrc/kdn_serve_rule.hpp), on the host."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kernel-deltanet_amd", "csrc")

# tokens, slots, heads, d_v -> beside the prefill on the auxiliary stream
CASES = [
    ((9, 9, 16, 64), 0), ((9, 8192, 16, 64), 0),            # a few decodes, whatever the pool's size
    ((100, 100, 4, 64), 0), ((224, 224, 16, 64), 0),        # decodes alone
    ((512, 512, 16, 64), 1),                                # enough of them that the events do not show
    ((309, 10, 16, 64), 0),                                 # a few decodes and a prefill of 300
    ((524, 225, 16, 64), 1), ((924, 226, 4, 64), 1),        # many decodes and one or two short prefills
    ((160, 100, 16, 64), 1), ((160, 100, 16, 16), 0),       # the same; a quarter of the bytes in narrow states
    ((1024, 2, 1, 16), 0), ((1025, 2, 1, 16), 1),           # long steps as with host offsets
]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text('#include <cstdio>\n#include <cstdlib>\n#include "kdn_serve_rule.hpp"\n'
                                "int main(int, char** a) {\n  printf(\"%d\\n\", (int)kdn::slot_decode_beside(atoll(a[1]), atoll(a[2]), "
                                "atoll(a[3]), 512, atoi(a[4])));\n}\n")
    subprocess.run([cxx, "-std=c++17", "-I", CSRC, "-o", str(d / "rule"), str(d / "rule.cpp")], check=True)
    return lambda *sizes: int(subprocess.run([str(d / "rule")] + [str(s) for s in sizes], capture_output=True, text=True,
                                             check=True).stdout)


@pytest.mark.parametrize("sizes,beside", CASES)
def test_decode_beside(rule, sizes, beside):
    assert rule(*sizes) == beside
