"""Kernels behind a guard that is up follow no pointer: they end whatever the
pairs of the iteration that raised it look like.  On the CPU (the kernels
compiled against the HIP subset in cpu_emu)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_no_walk_behind_the_guard(tmp_path):
    from cpu_emu import build as emu_build

    exe = tmp_path / "guarded_walk"
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-fno-fast-math", "-U_FORTIFY_SOURCE",
                    "-D_FORTIFY_SOURCE=0", "-w", "-pthread", "-I", os.path.join(HERE, "cpu_emu", "include"),
                    "-I", emu_build.CSRC, "-I", os.path.join(emu_build.ROOT, "include"),
                    "-x", "c++", os.path.join(emu_build.CSRC, "fl_kernels.hip"), "-x", "none",
                    os.path.join(HERE, "cpu_emu", "emu.cpp"), os.path.join(HERE, "cpp", "guarded_walk.cpp"),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
