"""What the compiled GEMM kernels of libnova_hip.so have to hold that no run of
them shows for certain: read from the code objects built in this tree."""
import glob
import os
import re
import shutil
import subprocess

import pytest

import nova_hip as nh

LLVM = "/opt/rocm/llvm/bin/"


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    """The library's gfx950 code objects, each with its kernels' names."""
    d = tmp_path_factory.mktemp("code")
    so = shutil.copy(os.path.join(os.path.dirname(nh.__file__), "libnova_hip.so"), d)
    subprocess.run([LLVM + "llvm-objdump", "--offloading", so], check=True, capture_output=True)
    out = []
    for f in sorted(glob.glob(str(d / "*gfx950*"))):
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", f], check=True, capture_output=True,
                               text=True).stdout
        out.append((f, notes, re.findall(r"\.name:\s+(_Z\w+)\n", notes)))
    return out


def _instructions(objects, pattern):
    """(kernel, its instructions) for each kernel whose name matches."""
    for f, _, names in objects:
        names = [n for n in names if re.search(pattern, n)]
        if not names:
            continue
        text = subprocess.run([LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr",
                               "--disassemble-symbols=" + ",".join(names), f], check=True,
                              capture_output=True, text=True).stdout
        for part in re.split(r"^<(?=_Z)", text, flags=re.M)[1:]:
            name, _, body = part.partition(">:")
            yield name, [line.split("//")[0].strip() for line in body.splitlines() if line.strip()]


def test_gemm_loads_are_inside_the_range_check(objects):
    """A buffer load's scalar offset need not count towards its range check, so
    the register-staged GEMM kernels leave it at zero: every byte a load
    addresses is in its address operand and its immediate offset."""
    seen = 0
    for name, ins in _instructions(objects, "gemm_unaligned|gemm_small"):
        for i in ins:
            if i.startswith("buffer_load"):
                seen += 1
                assert re.search(r"s\[\d+:\d+\], 0( |$)", i), (name, i)
    assert seen > 100
