"""Set and tag of the visited filter name the id, whatever the number of sets and of elements, and none looks like an empty
entry: a search takes a tag that is there for a node it has met."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def places(tmp_path_factory):
  out = str(tmp_path_factory.mktemp("filter_harness") / "filter_places")
  subprocess.check_call(["g++", "-std=c++17", "-O2", "-I" + os.path.join(ROOT, "cuhnsw_amd", "csrc"),
                         os.path.join(ROOT, "tests", "filter_harness", "filter_places.cpp"), "-o", out])
  return lambda *args: [int(x) for x in subprocess.check_output([out] + [str(a) for a in args]).split()]


@pytest.mark.parametrize("sets,n", [
    (1, 1), (260, 100_000), (260, 1 << 24), (261, (1 << 24) - 1),   # the fewest sets, the longest stretches
    (512, 1_183_514), (568, 10_000_000), (569, 1 << 24), (1023, 1 << 24), (16384, 1 << 24),
    (260, (1 << 24) + 1), (568, 30_000_000), (3000, 1 << 25),       # ids of more than 24 bits
])
def test_every_id_has_a_place_of_its_own(places, sets, n):
  got, outside, shared, as_empty = places(sets, n)
  assert got >= max(sets, 260) and (outside, shared, as_empty) == (0, 0, 0)


def test_a_filter_that_would_need_too_many_sets_is_none(places):
  assert places(260, 2_000_000_000, 1 << 20)[0] == 0
