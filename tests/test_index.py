"""The kernels' index arithmetic (pocket-engine_amd/csrc/pkv_index.h), built
for the host and checked against the bounds of what it indexes
(tests/index_check.cpp says which)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_index_arithmetic_on_the_host(tmp_path):
    exe = str(tmp_path / "index_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-fsanitize=undefined",
                    "-fno-sanitize-recover=all", os.path.join(HERE, "index_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0 and r.stdout.rstrip().endswith("ok"), r.stdout + r.stderr
