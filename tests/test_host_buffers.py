"""The context's device buffers at the limits of memory and under capture, with
hipMalloc and hipFree replaced by counters: tests/host_buffers.cpp, compiled
for the host against the library's own header."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_context_buffers(tmp_path):
    exe = tmp_path / "host_buffers"
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'vectorvisualization_amd' / 'csrc'}", str(ROOT / "tests" / "host_buffers.cpp"), "-o",
                    str(exe)], check=True, timeout=300)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
