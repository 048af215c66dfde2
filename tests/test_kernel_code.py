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


def _registers(text):
    """The vector registers an operand list names, as ("v" or "a", number)."""
    out = set()
    for kind, lo, hi, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", text):
        out.update((kind, n) for n in (range(int(lo), int(hi) + 1) if lo else [int(one)]))
    return out


def test_no_register_is_touched_while_an_lds_read_is_on_its_way_into_it(objects):
    """The LDS reads of these kernels are inline assembly, whose latency the
    compiler does not see: a copy or a spill of such a register that it places
    ahead of the kernel's own lgkmcnt wait would take the value of before."""
    reads = 0
    for name, ins in _instructions(objects, "gemm_f32_split|gemm_ring|gemm_pers"):
        pending = []  # one set of registers per LDS (or scalar) operation in flight, oldest first
        for i in ins:
            op, _, args = i.partition(" ")
            wait = re.search(r"lgkmcnt\((\d+)\)", i) if op == "s_waitcnt" else None
            if wait:
                n = int(wait.group(1))
                pending = pending[-n:] if n else []
            elif op in ("s_branch", "s_endpgm"):
                pending = []
            elif pending:
                busy = _registers(args) & set().union(*pending)
                assert not busy, (name, i, busy)
            if op.startswith("ds_read"):
                reads += 1
                pending.append(_registers(args.split(", v")[0]))
            elif op.startswith(("ds_", "s_load", "s_buffer_load")):
                pending.append(set())
    assert reads > 1000


def _resources(objects, pattern):
    """(kernel, what its code object says of a resource) for each match."""
    for _, notes, _ in objects:
        for block in re.split(r"\n  - \.agpr_count:", notes)[1:]:
            name = re.search(r"\.name:\s+(_Z\w+)\n", block).group(1)
            if re.search(pattern, name):
                yield name, lambda key: int(re.search(rf"\.{key}:\s+(\d+)\n", block).group(1))


def test_ring_and_split_kernels_spill_no_vector_register(objects):
    """A spill is memory traffic in the loops whose DMA waits are counted by
    hand, and a chance for the compiler to store a register too early (above)."""
    seen = 0
    for name, of in _resources(objects, "gemm_f32_split|gemm_ring|gemm_pers|gemm_unaligned"):
        seen += 1
        assert of("vgpr_spill_count") == 0 and of("private_segment_fixed_size") == 0, name
    assert seen > 50


# Tile (64 TM x 64 TN), stages, K groups -> workgroups per CU that the choice of
# a form and the tile order count on.
PER_CU = {("ring", 4, 3, 2, 1): 1, ("ring", 4, 2, 3, 1): 1, ("ring", 2, 2, 2, 2): 1,
          ("ring", 1, 2, 3, 1): 2, ("ring", 1, 1, 3, 1): 3, ("ring", 1, 1, 4, 2): 1,
          ("ring", 1, 1, 2, 1): 4, ("ring", 1, 2, 2, 1): 3,
          ("f32_split", 4, 3, 2, 1): 1, ("f32_split", 3, 4, 2, 1): 1, ("f32_split", 3, 3, 2, 1): 1,
          ("f32_split", 4, 2, 2, 1): 1, ("f32_split", 2, 2, 2, 1): 2, ("f32_split", 1, 1, 3, 1): 3}


def test_as_many_workgroups_fit_a_cu_as_the_form_tables_say(objects):
    """By LDS (160 KB) and by vector registers (512 per lane of a SIMD)."""
    seen = 0
    for name, of in _resources(objects, "gemm_f32_split|gemm_ring"):
        kind = "ring" if "gemm_ring" in name else "f32_split"
        tm, tn, stages, rest = map(int, re.findall(r"Li(\d+)E", name)[1 if kind == "ring" else 0:])
        want = PER_CU[kind, tm, tn, stages, rest if kind == "ring" else 1]
        waves = of("max_flat_workgroup_size") // 64 // 4  # per SIMD
        registers = -(-of("vgpr_count") // 8) * 8
        fit = min(160 * 1024 // of("group_segment_fixed_size"), 512 // registers // waves)
        assert fit >= want, (name, fit, want)
        seen += 1
    assert seen == 88
