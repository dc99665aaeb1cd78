"""The screened search's geometry (csrc/screen_geom.h) on the CPU: a C++ check program compiled with g++ walks the
loads of every plan as the kernel does."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "vapoursynth-zipcu_amd", "csrc")


def test_screen_geometry_reads_in_bounds(tmp_path):
    exe = str(tmp_path / "screen_geom_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Wextra", f"-I{CSRC}",
                    os.path.join(HERE, "cpp", "screen_geom_check.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "screen geometry: ok" in out.stdout
