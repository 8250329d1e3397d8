"""CPU: the host side of a batch (context.cpp) with stand-ins for the HIP
runtime and the kernel launchers (tests/cpu/host_check.cpp)."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "minirender_amd" / "csrc"


@pytest.fixture(scope="module")
def host_bin(tmp_path_factory):
    out = tmp_path_factory.mktemp("host") / "host_check"
    subprocess.run(["g++", "-w", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{CSRC}", str(ROOT / "tests" / "cpu" / "host_check.cpp"),
                    str(CSRC / "context.cpp"), "-o", str(out), "-lpthread"], check=True)
    return out


def run(host_bin, what):
    r = subprocess.run([str(host_bin), what], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "ok"


def test_general_batches_find_their_counters_zero(host_bin):
    run(host_bin, "clean")


def test_launches_counts_every_kernel(host_bin):
    run(host_bin, "launches")


def test_small_batches_are_those_that_gain(host_bin):
    """Triangles in no order, too many of them for a job's tiles, batches of
    many tests take the general kernels; frames of few tiles are shared out in
    row bands."""
    run(host_bin, "small")


def test_large_loose_triangles_take_the_small_kernels(host_bin):
    """Loose triangles are held to a limit by their size: the general kernels
    bin each for every tile, which costs more the larger they are."""
    run(host_bin, "scatter")


def test_small_batches_by_tile_size(host_bin):
    """8-pixel tiles test regions with one wavefront, 32-pixel tiles draw four
    times the pixels each: limits of their own."""
    run(host_bin, "tiles")


def test_graphs_are_updated_to_the_same_kernels(host_bin):
    """An instantiated graph takes another batch's parameters only when that
    batch launches the same kernels."""
    run(host_bin, "graphs")
