"""The multi-RHS schedule on the CPU (drivers/multi_schedule.cpp): executed as
the kernels read it, against the leaves, and its checks against damage that
keeps every total.  Stacks wider than a stage-1 group (2,048 columns) leave
slots that the t sum adds."""
import os
import re
import subprocess

import numpy as np
import pytest

from conftest import ROOT
from test_multi_groups import odd_matrix
from test_multi_wide import ND, WIDE
from test_schedule_replay import big_rank_matrix, write_format1

LIBDIR = os.path.join(ROOT, "hacapk_hmvm_amd")


@pytest.fixture(scope="module")
def driver(H, tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("drv") / "multi_schedule")
    subprocess.run(["g++", "-std=c++17", "-O2", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(LIBDIR, "csrc"),
                    os.path.join(ROOT, "tests", "drivers", "multi_schedule.cpp"), "-o", exe, "-L" + LIBDIR, "-lhmvm_hip",
                    "-Wl,-rpath," + LIBDIR], check=True)
    return exe


def matrix_file(H, tmp_path, kind):
    path = str(tmp_path / "m.bin")
    if kind == "wide":
        write_format1(path, ND, WIDE + [(2, 33, 65, 900, 1, 0), (2, 17, 9, 950, 20, 0)], np.random.default_rng(1))
    elif kind == "odd":
        odd_matrix(H, path, 2100)
    else:
        big_rank_matrix(H, path)
    return path


@pytest.mark.parametrize("kind", ["wide", "odd", "big"])
@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("t_mode", [-1, 0, 1, 2, 3])
@pytest.mark.parametrize("window", [0, 1])
def test_replay_and_damage(H, driver, tmp_path, kind, storage, t_mode, window):
    r = subprocess.run([driver, matrix_file(H, tmp_path, kind), str(storage), str(t_mode), str(window)],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    assert "MISSED" not in r.stdout
    counts = dict(re.findall(r"(windows|tsum|slots) (\d+)", r.stdout))
    assert (int(counts["tsum"]) > 0) == (kind == "wide") and (int(counts["windows"]) > 1) == (window > 0)
    damaged = r.stdout.count("\n") - 1 - r.stdout.count("nothing to damage")
    assert damaged >= (6 if kind != "big" else 5), r.stdout
