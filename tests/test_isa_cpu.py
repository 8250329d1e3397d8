"""CPU: what the compiler made of the kernels, from their gfx950 assembly.

The persistent kernel's scan writes tile_heavy, its shading reads it in the
same launch.  A scalar load there could be served from a line the scalar cache
already holds: no fence between the stages reaches that cache.
"""
import re
import subprocess
from pathlib import Path

import pytest

from minirender_amd import build

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    out = tmp_path_factory.mktemp("isa") / "kernels.s"
    subprocess.run([build.HIPCC, *build.COMMON, "-x", "hip", "--cuda-device-only", "-S",
                    str(build.CSRC / "kernels.hip"), "-o", str(out)], check=True, capture_output=True)
    return out.read_text()


def regs(op):
    """Scalar registers of an operand: s5, s[10:11]."""
    m = re.fullmatch(r"s\[(\d+):(\d+)\]|s(\d+)", op)
    if not m:
        return set()
    return {int(m[3])} if m[3] else set(range(int(m[1]), int(m[2]) + 1))


def scalar_reads_of(body, offset):
    """Scalar loads through the pointer at `offset` of the kernel's argument
    (within a basic block, following the pointer through scalar additions),
    and whether the pointer was loaded at all."""
    pointer, found, bad = set(), False, []
    for line in body.splitlines():
        if line.startswith((".LBB", "; %bb")):
            pointer = set()
        op, _, rest = line.strip().replace("\t", " ").partition(" ")
        args = [a.strip() for a in rest.split(";")[0].split(",")]
        if op.startswith("s_load_dword"):
            base, first = regs(args[1]), int(args[2], 0) if re.fullmatch(r"0x[0-9a-f]+|\d+", args[2]) else -1
            if base & pointer:
                bad.append(line.strip())
            dst = sorted(regs(args[0]))
            pointer -= set(dst)
            at = (offset - first) // 4
            if first >= 0 and 0 <= at < len(dst) - 1:
                pointer |= {dst[at], dst[at + 1]}
                found = True
        elif op.startswith("s_") and args and regs(args[0]):
            moves = op in ("s_add_u32", "s_addc_u32", "s_mov_b32", "s_mov_b64")
            tainted = moves and any(regs(a) & pointer for a in args[1:])
            pointer -= regs(args[0])
            if tainted:
                pointer |= regs(args[0])
    return bad, found


def test_persistent_shading_reads_tile_flags_by_vector_loads(assembly, tmp_path):
    src = tmp_path / "offset.cpp"
    src.write_text('#include <cstddef>\n#include <cstdio>\n#include "pipeline.h"\n'
                   'int main() { printf("%zu %d", offsetof(mr::BatchArgs, tile_heavy), (int)mr::kPShade); }\n')
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{build.CSRC}",
                    str(src), "-o", str(tmp_path / "offset")], check=True)
    offset, stage = map(int, subprocess.run([str(tmp_path / "offset")], capture_output=True, text=True,
                                            check=True).stdout.split())
    name = re.search(rf"^(\S*persist_stage\S*Li{stage}E\S*):", assembly, re.M).group(1)
    body = assembly[assembly.index(f"\n{name}:"):]
    bad, found = scalar_reads_of(body[:body.index(".Lfunc_end")], offset)
    assert found
    assert not bad, bad


@pytest.mark.parametrize("kernel", ["k_geom", "k_front"])
def test_geometry_takes_no_maxima_to_memory(assembly, kernel):
    """Geometry adds to counters only: a direct list is a length and its items
    (a bounding box of it, kept by atomic maxima on one line per job, was read
    by nothing)."""
    names = re.findall(rf"^(_ZN2mr\S*{kernel}\S*):", assembly, re.M)
    assert names
    for name in names:
        body = assembly[assembly.index(f"\n{name}:"):]
        body = body[:body.index(".Lfunc_end")]
        assert "global_atomic_add" in body or "ILb1E" in name  # (small batches count nothing)
        assert not re.findall(r"(?:global|flat)_atomic_u?max\S*", body)
