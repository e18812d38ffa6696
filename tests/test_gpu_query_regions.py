"""Batches of three rounds of wavefronts and more: the longest fifth first, the others by region, each chiplet's share of
them in a queue of its own.  Every query is answered, once, as the oracle answers it, whatever the numbers of queries, slots
and regions; also where all queries are one (a single region, a single length) and where few are left to share out."""
import numpy as np
import pytest

from helpers import gauss_mixture
from test_gpu_search import _device_search, _engine, _levels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,dist,max_m", [(40, "dot", 4), (100, "l2", 8), (300, "l2", 4)])
def test_queries_by_region(oracle, tmp_path, d, dist, max_m):
  n, k = 3000, 10
  mult = 1 / np.log(max_m)
  x = gauss_mixture(n, d, seed=21, normalise=dist == "dot")
  ix = oracle.OracleIndex(dist).build(x, _levels(n, mult, 22), max_m, 2 * max_m, 60, mult)
  p = str(tmp_path / "i.idx")
  ix.save(p)
  e = _engine(tmp_path, dist_type=dist, max_m=max_m, max_m0=2 * max_m)
  e.load_index(p)
  pool = gauss_mixture(3001, d, seed=23, normalise=dist == "dot")
  same = np.repeat(pool[:1], 700, axis=0)
  for slots, q in ((1, pool[:3]), (1, pool[:31]), (7, pool[:31]), (20, pool[:333]), (100, pool), (100, same),
                   (64, np.concatenate([same[:500], pool[:300]]))):
    e.set_tunable("search_slots", slots)
    for ef in (40, 200):
      o_ids, o_d, o_f, o_cnt = ix.search(q, k, ef, counters=True)
      for order in (2, 0):  # 2: whatever the size of batch and index
        e.set_tunable("query_order", order)
        g_ids, g_d, g_f, stats = _device_search(e, q, k, ef)
        assert (g_f == o_f).all() and (g_ids == o_ids).all() and (g_d == o_d).all()
        assert (stats[:, 1:] == o_cnt[:, 1:4]).all()


@pytest.mark.parametrize("mult", [1 / np.log(24), 1 / np.log(3), 0.0])
def test_levels_of_another_thickness(oracle, tmp_path, mult):
  """The level that stands for the regions goes by the levels the nodes have, not by max_m: many, few, none above 0."""
  n, d, k, ef = 3000, 24, 10, 80
  x = gauss_mixture(n, d, seed=31)
  ix = oracle.OracleIndex("dot").build(x, _levels(n, mult, 32), 12, 24, 60, max(mult, 0.1))
  p = str(tmp_path / "i.idx")
  ix.save(p)
  e = _engine(tmp_path, dist_type="dot", max_m=12, max_m0=24)
  e.load_index(p)
  q = gauss_mixture(2000, d, seed=33)
  o_ids, o_d, o_f, o_cnt = ix.search(q, k, ef, counters=True)
  e.set_tunable("search_slots", 64)
  for order in (1, 2, 3):
    e.set_tunable("query_order", order)
    g_ids, g_d, g_f, stats = _device_search(e, q, k, ef)
    assert (g_f == o_f).all() and (g_ids == o_ids).all() and (g_d == o_d).all()
    assert (stats[:, 1:] == o_cnt[:, 1:4]).all()
