"""The sorted set in registers at the edges of every size it is built for (64 entries per register of each lane: ef up to
512), filled to the last entry and one short of it, with distances that are all different and with integer data, where
equal keys meet at the set's end; and builds whose candidate sets have these sizes."""
import numpy as np
import pytest

from helpers import gauss_mixture, integer_vectors
from test_gpu_search import _check_parity, _engine, _levels

pytestmark = pytest.mark.gpu

EDGES = [63, 64, 65, 191, 192, 193, 255, 256, 257, 319, 320, 321, 383, 384, 385, 447, 448, 449, 511, 512]


@pytest.mark.parametrize("d,ints", [(50, False), (100, False), (12, True), (70, True)])
def test_search_at_the_edges_of_a_set(oracle, tmp_path, d, ints):
  n, mult = 3000, 1 / np.log(8)
  x = integer_vectors(n, d, seed=3, hi=9) if ints else gauss_mixture(n, d, seed=3)
  q = integer_vectors(60, d, seed=4, hi=9) if ints else gauss_mixture(60, d, seed=4)
  dist = "l2" if ints else "dot"
  ix = oracle.OracleIndex(dist).build(x, _levels(n, mult, 5), 8, 16, 60, mult)
  p = str(tmp_path / "s.idx")
  ix.save(p)
  e = _engine(tmp_path, dist_type=dist, max_m=8, max_m0=16)
  e.load_index(p)
  for ef in EDGES:
    _check_parity(oracle, ix, e, q, min(ef, 10 if ef % 2 else ef), ef, counters=False)


@pytest.mark.parametrize("efc", [64, 150, 192, 200, 256, 300, 384, 448, 449])
def test_build_with_every_set_size(oracle, tmp_path, efc):
  n, d, mult = 2500, 40, 1 / np.log(8)
  x, levels = integer_vectors(n, d, seed=6, hi=30), _levels(n, mult, 7)
  files = []
  for literal in (0, 1):  # (the literal queues place equal keys by their own rule: only the set's build is compared, below)
    e = _engine(tmp_path, dist_type="l2", max_m=8, max_m0=16, ef_construction=efc, heuristic_coef=0.0)
    e.set_data(x)
    e.set_random_levels(levels)
    e.set_tunable("build_literal", literal)
    e.build_graph()
    p = str(tmp_path / ("b%d.idx" % literal))
    e.save_index(p)
    ix = oracle.OracleIndex("l2").load(p)
    assert ix.validate() == 0
    files.append(ix)
  q = integer_vectors(100, d, seed=8, hi=30)
  gt, _ = oracle.bruteforce(x, q, 10, "l2")
  rec = [np.mean([len(set(a) & set(b)) / 10 for a, b in zip(ix.search(q, 10, 100)[0], gt)]) for ix in files]
  assert rec[0] >= rec[1] - 0.02
