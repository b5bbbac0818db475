"""Source codes of the triangular solves over chains (xs_strip.h): the LDS
places that a step reads for them, in workgroups of four and of eight waves."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_code_points_into_the_lds_arrays(tmp_path):
    exe = str(tmp_path / "strip_codes")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(HERE, "hostsim"), "-o", exe,
                    os.path.join(HERE, "hostsim", "strip_codes.cpp")], check=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and int(p.stdout) == 0, (p.stdout, p.stderr)
