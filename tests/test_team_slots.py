"""The slots in which a team of wavefronts keeps its lists (cuhnsw_amd/csrc/team_slots.h): whatever the order in which the wavefronts'
accesses happen, a list has one writer, and none outlives the level it was made for."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def run(tmp_path_factory):
  def compiled(name):
    out = str(tmp_path_factory.mktemp("team_harness") / name)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-I" + os.path.join(ROOT, "cuhnsw_amd", "csrc"),
                           os.path.join(ROOT, "tests", "team_harness", name + ".cpp"), "-o", out])
    return lambda *args: [int(x) for x in subprocess.check_output([out] + [str(a) for a in args]).split()]
  return compiled


def test_a_list_has_one_writer_and_one_level(run):
  slots = run("slots")
  states, clashes, stale = slots(0)
  assert states > 1000 and (clashes, stale) == (0, 0)
  # (the walk does find the two writers where a level's end stores to slots that were free when it looked)
  assert slots(1)[1] > 0


def test_a_list_of_any_length_that_a_row_can_have_keeps_its_slot(run):
  """Rows of 64 ids have lists of up to eight eights."""
  assert run("words")() == [0, 0]
