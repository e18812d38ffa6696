"""Saves that do not finish, and files that change under a reader: nothing but a whole index is ever accepted, and no
process dies of it.  (Host code, compiled here; the engine with a GPU writes and reads through the same classes.)"""
import os
import shutil
import subprocess
import tempfile
import time

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
  out = str(tmp_path_factory.mktemp("file_harness") / "file_faults")
  src = os.path.join(ROOT, "cuhnsw_amd", "csrc")
  subprocess.check_call(["g++", "-std=c++17", "-O1", "-I" + src, os.path.join(ROOT, "tests", "file_harness", "file_faults.cpp"),
                         os.path.join(src, "index_file.cpp"), "-o", out])
  return out


@pytest.fixture(params=["tmp", "shm"])
def path(request, tmp_path):
  """A file on a disk's file system and one in memory (they are written in different ways)."""
  if request.param == "tmp":
    yield str(tmp_path / "index.hnsw")
    return
  if not os.access("/dev/shm", os.W_OK):
    pytest.skip("no file system in memory")
  folder = tempfile.mkdtemp(prefix="cuhnsw_test_", dir="/dev/shm")
  yield os.path.join(folder, "index.hnsw")
  shutil.rmtree(folder)


def call(harness, *args):
  r = subprocess.run([harness] + list(args), capture_output=True, text=True, check=False)
  assert r.returncode == 0, (args, r.returncode)   # (a negative status: a signal ended the process)
  return r.stdout.strip()


@pytest.mark.parametrize("mode", ["throw", "die"])
@pytest.mark.parametrize("before", ["nothing", "an index"])
def test_an_unfinished_save_leaves_nothing_that_loads(harness, path, mode, before):
  if before == "an index":
    call(harness, "write", path, "1")
    assert call(harness, "read", path) == "1 1"
  call(harness, mode, path, "2")
  assert call(harness, "read", path).startswith("refused: index file:")
  call(harness, "write", path, "3")                # and the path is as good as before
  assert call(harness, "read", path) == "3 3"


def test_a_file_saved_over_while_it_is_read_is_refused(harness, path):
  call(harness, "write", path, "1")
  time.sleep(0.05)                                 # (a file's time stamp moves in steps of a few milliseconds)
  assert call(harness, "overtaken", path, "2") == "refused: index file: written to while it was read"
  assert call(harness, "read", path) == "2 2"


def test_a_file_cut_off_while_it_is_written_does_not_end_the_process(harness, path):
  """(Through a mapping an ordinary store to what is no longer there would be a bus error.)"""
  call(harness, "cut", path, "1")                  # refused, or written as far as it goes: but it returns
  call(harness, "write", path, "2")
  assert call(harness, "read", path) == "2 2"
