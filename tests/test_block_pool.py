"""CPU: the block pool of a context (plato_amd/csrc/block_pool.hpp, the code the library
compiles) driven by several threads at once under g++'s thread sanitizer."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_pool_under_threads(tmp_path):
    exe = tmp_path / "test_block_pool"
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-fsanitize=thread", "-pthread",
                    "-I", os.path.join(ROOT, "plato_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "test_block_pool.cc"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "shared blocks: 0, left: 0, kept: 0, used: 0" in r.stdout
