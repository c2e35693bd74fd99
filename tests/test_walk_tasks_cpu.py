"""The scheduling of cut traversals, run on the CPU with a thread for each wave (walk_tasks_model.cpp):
whichever classes of blocks are placed on the device and however full the tables get, every wave ends and
each group has the result and the counts that it has alone."""

import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pytreegrav_amd", "csrc")

pytestmark = pytest.mark.skipif(not shutil.which("g++"), reason="g++ not available")


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("tasks") / "model")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", CSRC, os.path.join(HERE, "walk_tasks_model.cpp"),
                    "-o", exe], check=True)

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stdout + r.stderr
        return [int(v) for v in re.findall(r"\d+", r.stdout)]

    return run


# all classes; one missing, as when another walk's waiting waves hold an XCD; a single running wave
@pytest.mark.parametrize("classes,per", [(0xFF, 2), (0x7F, 2), (0xFE, 1), (0x10, 1), (0x81, 3)])
@pytest.mark.parametrize("groups", [1, 100])
def test_every_task_is_walked_whichever_blocks_run(model, classes, per, groups):
    assert model(classes, per, groups) == [0, 0]


# tables of tasks, of stack entries and of groups too small for all groups at once, and for the largest
# group alone (a level of larger budgets, or several)
@pytest.mark.parametrize("tcount,ecap,gcount,largest,level", [(64, 4096, 512, 90, 0), (4096, 128, 512, 90, 0),
                                                              (4096, 4096, 3, 90, 0), (257, 4096, 512, 2000, 1),
                                                              (61, 64, 2, 5000, 2), (4096, 200, 512, 3000, 1),
                                                              (16, 32, 1, 40000, 3)])
@pytest.mark.parametrize("classes,per", [(0xFF, 2), (0x08, 1)])
def test_full_tables_change_no_result(model, tcount, ecap, gcount, largest, level, classes, per):
    for _ in range(3):
        back, deepest = model(classes, per, 700, largest, tcount, ecap, gcount)
        assert back > 0 and deepest >= level
