"""The device blocks kept for the next states (burn_automata_amd/csrc/npa_blocks.hpp), over a host allocator with a
budget: reuse, bounds, what is given back where an allocation finds no memory, and threads."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_kept_blocks(tmp_path):
    exe = tmp_path / "check_blocks"
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-Wall", "-Wextra", "-Werror", "-o", str(exe),
                    os.path.join(ROOT, "tests", "native", "check_blocks.cpp")], check=True)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=120)
    assert r.returncode == 0 and "blocks ok" in r.stdout, r.stdout
