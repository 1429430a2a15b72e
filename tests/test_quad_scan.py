"""The indices the quad walks of Fluids, Boids and Clouds load, on the CPU: the walks' own stepping
(csrc/rtp_quad_scan.hpp) compiled for the host."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "realtimeparticles_amd", "csrc")


def test_quads_load_inside_their_buffers(tmp_path):
    exe = str(tmp_path / "quad_scan")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "cpp", "quad_scan.cpp")], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
