"""The locality order of host layouts on the CPU: a permutation, compact, the same from any run, and made without a data
race (its threads share one array of marks)."""
import os
import subprocess

import pytest

from conftest import REPO

HOST = os.path.join(REPO, "tests", "host")


def build(tmp_path, *flags):
    exe = str(tmp_path / "order_check")
    subprocess.run(["g++", "-O2", "-std=c++17", *flags, "-I", os.path.join(REPO, "include"), "-I",
                    os.path.join(REPO, "shallow-water-eric_amd", "csrc"), "-o", exe,
                    os.path.join(HOST, "order_check.cpp"), "-lpthread"], check=True)
    return exe


def test_order_is_a_compact_permutation(tmp_path):
    out = subprocess.run([build(tmp_path), "401", "4"], capture_output=True, text=True)
    print(out.stdout)
    assert out.returncode == 0
    longest, mean = out.stdout.split()[1:3]
    # a halo longer than 512 rows sends the mesh to the gather kernels; a 16 x 16 patch of this graph borders on 66
    assert int(longest) <= 512 and float(mean) < 2 * 66


def test_order_without_a_data_race(tmp_path):
    """300 x 300 rows: above the 32,768 from which parts are bisected side by side."""
    trivial = tmp_path / "t.cpp"
    trivial.write_text("int main() { return 0; }\n")
    exe = str(tmp_path / "t")
    ok = subprocess.run(["g++", "-fsanitize=thread", "-o", exe, str(trivial)], capture_output=True)
    if ok.returncode or subprocess.run([exe], capture_output=True).returncode:
        pytest.skip("no thread sanitizer here")
    exe = build(tmp_path, "-g", "-fsanitize=thread")
    out = subprocess.run([exe, "300"], capture_output=True, text=True, env=dict(os.environ, TSAN_OPTIONS="exitcode=66"))
    assert out.returncode == 0, out.stderr[-3000:]
    assert out.stdout.startswith("ok")
