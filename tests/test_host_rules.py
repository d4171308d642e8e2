"""Host rules of the engine, checked on the CPU by small programs over its headers (tests/cpp)."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "lbm-topopt_amd", "csrc")


def run_program(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
                    os.path.join(ROOT, "tests", "cpp", name + ".cpp"), "-o", exe], check=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "RESULT OK" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]


def test_grouped_sweeps_read_the_right_states(tmp_path):
    run_program(tmp_path, "sweep_groups_check")


def test_checkpoint_count_streams():
    """lbmx_checkpoint_simulate counts a schedule without holding lists of its steps."""
    code = ("import resource, lbmx\n"
            "lbmx.checkpoint_simulate(48, 1000)\n"
            "a = resource.getrusage(resource.RUSAGE_SELF).ru_maxrss\n"
            "lbmx.checkpoint_simulate(48, 300000)\n"
            "print(resource.getrusage(resource.RUSAGE_SELF).ru_maxrss - a)\n")
    env = dict(os.environ, PYTHONPATH=os.path.join(ROOT, "lbm-topopt_amd"))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stderr[-2000:]
    assert int(r.stdout.split()[-1]) < 8 * 1024  # KiB; 300000 steps in lists take tens of MiB


def test_cone_kernel_choice(tmp_path):
    run_program(tmp_path, "cone_shape_check")


def test_steps_shape(tmp_path):
    run_program(tmp_path, "steps_shape_check")
