"""The (schedule, search) pairs of a batch (csrc/batch_pairs.h) on the CPU: a C++ check program compiled with g++ holds
that each pair is another launch, that only allowed ones are listed, and which one is taken without timing."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)


def test_batch_pairs(tmp_path):
    exe = str(tmp_path / "batch_pairs_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", f"-I{REPO}/vapoursynth-zipcu_amd/csrc", f"-I{REPO}/include",
                    os.path.join(HERE, "cpp", "batch_pairs_check.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "batch pairs: ok" in out.stdout
