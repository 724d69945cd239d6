"""CPU: the host side of synchronous transfers where no memory can be pinned or
the stream cannot be asked whether it is captured (tests/cxx/host_stage.cpp, over
a stub runtime)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_transfers_without_pinned_memory(tmp_path):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    exe = str(tmp_path / "host_stage")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unused-result", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(rocm, "include"),
                    os.path.join(HERE, "cxx", "host_stage.cpp"), os.path.join(ROOT, "xmp_amd", "csrc", "api.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "host stage ok" in r.stdout, r.stdout + r.stderr
