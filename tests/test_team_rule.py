"""Rules of the one-kernel PCG solve that need no GPU: a C++ program over
idp_amd/csrc/team_rule.hpp."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_team_rules(tmp_path):
    exe = tmp_path / "team_rule"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-O1", os.path.join(HERE, "cpp", "team_rule.cpp"), "-o",
                    str(exe)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
