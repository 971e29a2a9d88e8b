"""The P6 sub-step's linear system (csrc/react_solve.hpp) built for the CPU with the sanitizers' checks of every index,
over random records with and without the neutrons, against long double."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def build_and_run(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wno-unknown-pragmas", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", os.path.join(HERE, name + ".cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout


def test_the_system_is_solved_within_its_arrays(tmp_path):
    out = dict(line.split() for line in build_and_run(tmp_path, "react_solve").splitlines())
    # 1e-16 a rounding, a few hundred roundings, and the systems' condition (derivatives over five decades)
    assert set(out) == {"9", "10"} and all(float(v) <= 1e-10 for v in out.values()), out
