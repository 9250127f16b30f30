"""The wavefront's edge selection (prep_selec_wave) against the reference's quickselect (prep_selec), both
compiled for the CPU: the same value and the same array afterwards, with ties, infinities, NaN, constant
and sorted arrays, lengths from 4 to 502."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_wave_selection_equals_selec(tmp_path):
    exe = tmp_path / "selec_wave"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I",
                    os.path.join(os.path.dirname(HERE), "simple3.0_amd", "csrc"),
                    os.path.join(HERE, "selec_wave.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe), "800"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout == "0 of 800 differ\n", r.stdout + r.stderr
