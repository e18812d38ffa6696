"""Builds by teams of wavefronts on rows too long for registers: the node's row and, in its place, those of the selection's picks lie in
LDS that the whole team reads."""
import numpy as np
import pytest

from helpers import gauss_mixture
from test_gpu_search import _engine, _levels

pytestmark = pytest.mark.gpu


def test_index_of_long_rows_built_by_teams_is_the_one_built_without(tmp_path):
  """A short search: the selection begins soon after the team has."""
  n, d = 1200, 960
  x, levels, files = gauss_mixture(n, d, seed=5), _levels(n, 1.0 / np.log(16), 6), []
  for entries in (0, 16384):
    e = _engine(tmp_path, dist_type="l2", max_m=16, max_m0=32, ef_construction=12, heuristic_coef=0.0)
    e.set_tunable("filter_entries", entries)
    e.set_data(x)
    e.set_random_levels(levels)
    e.build_graph()
    assert (e.last_build_team_batches > 0) == (entries == 0)
    p = tmp_path / "b.idx"
    e.save_index(str(p))
    files.append(p.read_bytes())
  assert files[0] == files[1]
