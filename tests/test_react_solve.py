"""P6's host side and linear system without a device: the sub-step's system (csrc/react_solve.hpp) built for the CPU with
the sanitizers' checks of every index, over random records with and without the neutrons, against long double; and the
launches of worlds with different records, over a stand-in for the HIP runtime (tests/host/fake_hip.hpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
HOST = os.path.join(HERE, "host")
CSRC = os.path.join(HERE, os.pardir, "sandbox_reactions_amd", "csrc")


def run(exe):
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    return r.stdout


def test_the_system_is_solved_within_its_arrays(tmp_path):
    exe = str(tmp_path / "react_solve")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wno-unknown-pragmas", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", os.path.join(HOST, "react_solve.cpp"), "-o", exe], check=True)
    out = dict(line.split() for line in run(exe).splitlines())
    # 1e-16 a rounding, a few hundred roundings, and the systems' condition (derivatives over five decades)
    assert set(out) == {"9", "10"} and all(float(v) <= 1e-10 for v in out.values()), out


def host_program(tmp_path, name, sources):
    """A program of the library's host code alone (no device code) and the stand-in runtime."""
    from sandbox_reactions_amd.build import HIPCC
    objs = []
    for src in [os.path.join(HOST, name + ".cpp")] + [os.path.join(CSRC, s) for s in sources]:
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "--cuda-host-only", "-O1", "-std=c++17", "-w",
                        "-c", src, "-o", objs[-1]], check=True)
    exe = str(tmp_path / name)
    subprocess.run([HIPCC, "-o", exe] + objs + ["-lpthread", "-Wl,--unresolved-symbols=ignore-all"], check=True)
    return exe


def test_no_world_lowers_the_lds_limit_of_another(tmp_path):
    run(host_program(tmp_path, "react_launch", ["react.hip", "util.cpp"]))
