"""Which batches and builds go by teams of wavefronts: a wavefront alone gives the same answers and the same file, so that nothing
else says which of the two it was."""
import numpy as np
import pytest

from helpers import gauss_mixture
from test_gpu_search import _device_search, _engine, _levels

pytestmark = pytest.mark.gpu


def _built(tmp_path, n, d, dist, entries=0, max_m0=32, efc=80):
  e = _engine(tmp_path, dist_type=dist, max_m=16, max_m0=max_m0, ef_construction=efc, heuristic_coef=0.0)
  e.set_tunable("filter_entries", entries)
  e.set_data(gauss_mixture(n, d, seed=1, normalise=dist == "dot"))
  e.set_random_levels(_levels(n, 1 / np.log(16), 2))
  e.build_graph()
  return e


# (256 CUs: the wavefronts that the GPU holds of a kernel of 128 registers are four teams of four, or two of eight, on each; long rows
# take 256 registers: half as many; and their bytes in all.  And a wavefront alone where teams are the slower way: short searches, long
# ones on a GPU that many teams share, teams of four on rows of 129 to 256 elements but for a middle range)
@pytest.mark.parametrize("d,dist,ef,teams", [
    (50, "dot", 300, {1: 8, 256: 8, 257: 8, 512: 8, 513: 4, 768: 4, 1024: 4, 1025: 0}),
    (50, "dot", 31, {1: 0, 64: 0, 512: 0, 1024: 0}),
    (50, "dot", 32, {1: 8, 256: 8, 257: 0, 513: 0}),
    (50, "dot", 512, {64: 8, 512: 8, 1024: 4}),
    (50, "dot", 930, {8: 8, 64: 8, 65: 0, 300: 0}),
    (50, "dot", 1000, {8: 8, 9: 0, 256: 0}),
    (128, "l2", 128, {1: 8, 256: 8, 512: 8, 513: 4, 1024: 4, 1025: 0}),
    (100, "l2", 50, {1: 8, 64: 8, 256: 8, 257: 0, 513: 0}),
    (100, "dot", 450, {512: 8, 513: 0, 1024: 0}),
    (180, "l2", 200, {1: 8, 256: 8, 512: 8, 513: 4, 768: 4, 769: 0, 1024: 0}),
    (180, "l2", 60, {1: 8, 64: 8, 65: 0, 512: 0, 700: 0}),
    (180, "dot", 100, {65: 8, 512: 8, 513: 0}),
    (180, "dot", 330, {512: 8, 513: 0}),
    (300, "l2", 150, {1: 8, 256: 8, 257: 4, 512: 4, 513: 0}),
    (300, "l2", 39, {1: 0, 300: 0}),
    (960, "l2", 150, {1: 8, 186: 8, 187: 4, 293: 4, 294: 0}),
])
def test_batches_that_leave_the_machine_idle_go_by_teams(tmp_path, d, dist, ef, teams):
  e = _built(tmp_path, 2000, d, dist)
  q = gauss_mixture(1025, d, seed=3, normalise=dist == "dot")
  got = {}
  for nq in teams:
    _device_search(e, q[:nq], 10, ef)
    got[nq] = e.last_search_team
  assert got == teams
  e.set_tunable("filter_entries", 16384)
  _device_search(e, q[:1], 10, ef)
  assert e.last_search_team == 0


@pytest.mark.parametrize("d,dist", [(50, "dot"), (128, "l2"), (180, "l2"), (300, "l2")])
def test_small_batches_of_a_build_go_by_teams(tmp_path, d, dist):
  # (batches grow with the index: of 3 000 nodes all have at most 1 024)
  assert _built(tmp_path, 3000, d, dist).last_build_team_batches > 5
  assert _built(tmp_path, 3000, d, dist, entries=16384).last_build_team_batches == 0
  assert _built(tmp_path, 3000, d, dist, max_m0=65).last_build_team_batches == 0
