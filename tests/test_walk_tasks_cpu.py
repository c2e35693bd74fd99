"""The scheduling of cut traversals, run on the CPU with a thread for each wave (walk_tasks_model.cpp):
whichever classes of blocks are placed on the device, every task is walked once and every wave ends."""

import os
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
    return exe


# all classes; one missing, as when another walk's waiting waves hold an XCD; a single running wave
@pytest.mark.parametrize("classes,per", [(0xFF, 2), (0x7F, 2), (0xFE, 1), (0x10, 1), (0x81, 3)])
@pytest.mark.parametrize("groups", [1, 100])
def test_every_task_is_walked_whichever_blocks_run(model, classes, per, groups):
    r = subprocess.run([model, str(classes), str(per), str(groups)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
