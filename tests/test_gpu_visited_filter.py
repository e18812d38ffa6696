"""What the visited filter forgets, and whatever its size, changes nothing: the same index file, the same answers -- also where
the answer, which lies over the filter, is longer than that."""
import hashlib

import numpy as np
import pytest

from helpers import gauss_mixture, integer_vectors
from test_gpu_search import _check_parity, _engine, _levels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,dist", [(50, "dot"), (100, "l2"), (300, "l2")])
def test_builds_are_the_same_whatever_the_filter(tmp_path, d, dist):
  """(Small filters lose nodes between the candidates of one batch, which then lists them twice and may put them back.)"""
  n, mult = 6000, 1 / np.log(12)
  x, levels = gauss_mixture(n, d, seed=5, normalise=dist == "dot"), _levels(n, mult, 6)
  files = set()
  for entries in (0, 1040, 1100, 1500, 4096, 16384):
    e = _engine(tmp_path, dist_type=dist, max_m=12, max_m0=24, ef_construction=200, heuristic_coef=0.0)
    e.set_tunable("filter_entries", entries)
    e.set_data(x)
    e.set_random_levels(levels)
    e.build_graph()
    p = str(tmp_path / "b.idx")
    e.save_index(p)
    with open(p, "rb") as f:
      files.add(hashlib.sha256(f.read()).hexdigest())
  assert len(files) == 1


@pytest.mark.parametrize("ints", [False, True])
def test_answers_of_every_length_over_the_filter(oracle, tmp_path, ints):
  n, d, mult = 4000, 40, 1 / np.log(8)
  x = integer_vectors(n, d, seed=7, hi=12) if ints else gauss_mixture(n, d, seed=7)
  q = integer_vectors(50, d, seed=8, hi=12) if ints else gauss_mixture(50, d, seed=8)
  dist = "l2" if ints else "dot"
  ix = oracle.OracleIndex(dist).build(x, _levels(n, mult, 9), 8, 16, 80, mult)
  p = str(tmp_path / "s.idx")
  ix.save(p)
  e = _engine(tmp_path, dist_type=dist, max_m=8, max_m0=16)
  e.load_index(p)
  for entries, k, ef in ((0, 1, 40), (0, 100, 128), (1040, 173, 300), (1040, 174, 300), (1040, 512, 512), (0, 1000, 1000)):
    e.set_tunable("filter_entries", entries)
    e.set_tunable("fast_path", 2)
    _check_parity(oracle, ix, e, q, k, ef, counters=False)
