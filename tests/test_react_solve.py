"""P6's host side and arithmetic without a device: the temperature factor and the sub-step's system (csrc/react_solve.hpp) built for the CPU with
the sanitizers' checks of every index, over random records with and without the neutrons, against long double; and the
launches of worlds with different records, over a stand-in for the HIP runtime (tests/host/fake_hip.hpp)."""
import os
import subprocess

from helpers import HOST, WORLD_SOURCES, host_program, run_host


def test_factor_and_system_within_their_arrays(tmp_path):
    exe = str(tmp_path / "react_solve")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wno-unknown-pragmas", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", os.path.join(HOST, "react_solve.cpp"), "-o", exe], check=True)
    out = dict(line.split() for line in run_host(exe).splitlines())
    # 1e-16 a rounding, a few hundred roundings, and the systems' condition (derivatives over five decades)
    assert set(out) == {"factor", "9", "10"} and all(float(out[k]) <= 1e-10 for k in ("9", "10")), out
    # ln(T / T_thr) to two roundings of 1.1e-16 over a node's 0.0036, times ln f's step of up to 0.14 a node (9e-15), and
    # ln f itself, up to 95, to two roundings of 7e-15
    assert float(out["factor"]) <= 2.5e-14, out


def test_no_world_lowers_the_lds_limit_of_another(tmp_path):
    run_host(host_program(tmp_path, "react_launch", ["react.hip", "util.cpp"]))


def test_the_report_is_summed_on_the_device(tmp_path):
    run_host(host_program(tmp_path, "react_report", WORLD_SOURCES))
