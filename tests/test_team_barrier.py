"""The ePIE team's barrier hands every workgroup the values of its own barrier, in whatever order the
workgroups announce and read: checked over all orders on the host, with the flag words the kernel uses
(ptyk_team.h)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")


def _run(tmp_path, *defines):
    exe = tmp_path / "team_barrier"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", *defines, f"-I{ROOT / 'ptychopy_amd' / 'csrc'}",
                    str(ROOT / "tests" / "seam" / "team_barrier.cpp"), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True)


def test_every_order_gives_the_values_of_the_awaited_barrier(tmp_path):
    r = _run(tmp_path)
    assert r.returncode == 0 and int(r.stdout.split()[0]) > 1000, r.stdout


def test_one_word_a_workgroup_would_not(tmp_path):
    """The check finds the fault of a single word: a late reader gets the next barrier's value."""
    r = _run(tmp_path, "-DONE_WORD")
    assert r.returncode == 1 and "gives" in r.stdout, r.stdout


def test_teams_get_their_place_in_the_order_they_come(tmp_path):
    """A large team is not overtaken for ever by small ones that fit beside what others hold."""
    exe = tmp_path / "team_slots"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-pthread", f"-I{ROOT / 'ptychopy_amd' / 'csrc'}",
                    str(ROOT / "tests" / "seam" / "team_slots.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
