"""No kernel of the built library uses scratch (spilled registers, private arrays), read from the code objects' notes."""
import os
import re
import subprocess

import pytest

from kdn import build as kbuild

LLVM = "/opt/rocm/llvm/bin"
EM_AMDGPU = 224


def code_objects(lib, tmp):
    """The gfx950 ELF images of the library's fat binary, as files."""
    fat = os.path.join(tmp, "fat.bin")
    subprocess.run([os.path.join(LLVM, "llvm-objcopy"), f"--dump-section=.hip_fatbin={fat}", lib, os.path.join(tmp, "copy.so")],
                   check=True)
    data = open(fat, "rb").read()
    at = [m.start() for m in re.finditer(b"\x7fELF", data) if int.from_bytes(data[m.start() + 18:m.start() + 20], "little") == EM_AMDGPU]
    for i, (lo, hi) in enumerate(zip(at, at[1:] + [len(data)])):
        path = os.path.join(tmp, f"{i}.co")
        with open(path, "wb") as f:
            f.write(data[lo:hi])
        yield path


def test_no_kernel_uses_scratch(tmp_path):
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "llvm-readelf")]
    if not os.path.exists(kbuild.OUT) or not all(os.path.exists(t) for t in tools):
        pytest.skip("needs the built library and LLVM's binary tools")
    found, scratch = 0, {}
    for path in code_objects(kbuild.OUT, str(tmp_path)):
        notes = subprocess.run([tools[1], "--notes", path], capture_output=True, text=True, check=True).stdout
        names = re.findall(r"^\s+\.name:\s+(_Z\S+)", notes, re.M)
        sizes = [int(v) for v in re.findall(r"\.private_segment_fixed_size:\s*(\d+)", notes)]
        assert len(names) == len(sizes)
        found += len(names)
        scratch.update({n: v for n, v in zip(names, sizes) if v})
    assert found > 200
    assert scratch == {}
