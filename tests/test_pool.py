"""CPU: the buffer pool over a stand-in for the HIP allocator (a host program)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pool(tmp_path):
    exe = str(tmp_path / "pool")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", exe,
                    os.path.join(ROOT, "tests", "host", "pool.cpp"),
                    os.path.join(ROOT, "amcl3d_amd", "csrc", "pool.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
