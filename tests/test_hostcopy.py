"""The pinned-ring copies (pathtracer_amd/csrc/hostcopy.cpp) on the CPU, against
stand-ins for the HIP calls (tests/hostcopy_sim.cpp): bytes both ways around the
chunk sizes, and which memory goes through the ring: the caller's pageable one. Memory
that the runtime knows (page-locked, managed or on a device) is copied by the runtime
in one piece; copying threads would only slow it down, or could not reach it."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
SIZES = [1, (128 << 10) - 1, 128 << 10, (2 << 20) + 1, 5 << 20, (33 << 20) + 7]


@pytest.fixture(scope="module")
def sim(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not Path("/opt/rocm/include/hip/hip_runtime.h").exists():
        pytest.skip("g++ or the HIP headers not found")
    exe = tmp_path_factory.mktemp("hc") / "hostcopy_sim"
    csrc = ROOT / "pathtracer_amd" / "csrc"
    subprocess.run([gxx, "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-isystem", "/opt/rocm/include", "-I", str(csrc),
                    str(ROOT / "tests" / "hostcopy_sim.cpp"), str(csrc / "hostcopy.cpp"), "-o", str(exe), "-pthread"],
                   check=True, timeout=120)
    return exe


def run(sim, *args):
    r = subprocess.run([str(sim), *map(str, args)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr


@pytest.mark.parametrize("kind", ["pageable", "pinned", "device", "managed"])
def test_bytes_and_way(sim, kind):
    for n in SIZES:
        run(sim, kind, n)


@pytest.mark.parametrize("kind", ["pageable", "pinned"])
def test_stream_of_another_device_than_the_current_one(sim, kind):
    for n in SIZES:
        run(sim, kind, n, 1)
