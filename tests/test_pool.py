"""CPU test of the caching pool's rules (csrc/pool.hpp, plain host code):
reuse by size, the bound and what it evicts, room made when memory runs out,
several threads at once."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pool_rules(tmp_path):
    exe = str(tmp_path / "pool_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "idrs-package_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "pool_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
