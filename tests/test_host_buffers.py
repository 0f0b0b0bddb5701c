"""The library's device buffers at the limits of memory and under capture, with
hipMalloc and hipFree replaced by counters and the kernels by checks of their
buffers: tests/host_buffers.cpp, compiled for the host with the library's own
sources."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_device_buffers(tmp_path):
    csrc = ROOT / "vectorvisualization_amd" / "csrc"
    exe = tmp_path / "host_buffers"
    # the launchers that no check reaches stay undefined
    subprocess.run(["g++", "-std=c++17", "-no-pie", "-fno-pie", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{ROOT / 'include'}", f"-I{csrc}", str(ROOT / "tests" / "host_buffers.cpp"),
                    "-Wl,--unresolved-symbols=ignore-all", "-o", str(exe)], check=True,
                   timeout=300)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr
