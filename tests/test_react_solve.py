"""P6's host side and linear system without a device: the sub-step's system (csrc/react_solve.hpp) built for the CPU with
the sanitizers' checks of every index, over random records with and without the neutrons, against long double; and the
launches of worlds with different records, over a stand-in for the HIP runtime (tests/host/fake_hip.hpp)."""
import os
import subprocess

from helpers import HOST, host_program, run_host


def test_the_system_is_solved_within_its_arrays(tmp_path):
    exe = str(tmp_path / "react_solve")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wno-unknown-pragmas", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", os.path.join(HOST, "react_solve.cpp"), "-o", exe], check=True)
    out = dict(line.split() for line in run_host(exe).splitlines())
    # 1e-16 a rounding, a few hundred roundings, and the systems' condition (derivatives over five decades)
    assert set(out) == {"9", "10"} and all(float(v) <= 1e-10 for v in out.values()), out


def test_no_world_lowers_the_lds_limit_of_another(tmp_path):
    run_host(host_program(tmp_path, "react_launch", ["react.hip", "util.cpp"]))
