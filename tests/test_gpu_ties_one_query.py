"""Equal keys in searches of one query, which run alone in the instance for idle machines: there the offers of an
evaluation enter a full set together, unless equal keys forbid it.  (The index is loaded anew for each query: one that was
handed over would send the next ones another way.)"""
import numpy as np
import pytest

from helpers import graph_cut_between_equals, integer_vectors
from test_gpu_search import _device_search, _engine, _levels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ef", [129, 150, 300, 500])
@pytest.mark.parametrize("d", [8, 100, 200, 300])
def test_a_cut_between_two_equal_keys(oracle, tmp_path, d, ef):
  rng = np.random.default_rng(31 * d + ef)
  e = _engine(tmp_path, dist_type="l2", max_m=32, max_m0=64)
  for case in range(12):
    coordinates, rows = graph_cut_between_equals(rng, ef, width=64)
    x = np.zeros((len(rows), d), np.float32)
    x[:, case % d] = coordinates
    links0 = np.zeros((len(rows), 1 + 64), np.uint32)
    for i, nb in enumerate(rows):
      links0[i, 0] = len(nb)
      links0[i, 1:1 + len(nb)] = nb
    ix = oracle.OracleIndex("l2").from_arrays(x, np.zeros(len(rows), np.int32), links0, np.zeros(0, np.uint32),
                                              max_m=32, max_m0=64, maxlevel=0, enterpoint=0)
    p = str(tmp_path / "c.idx")
    ix.save(p)
    q = np.zeros((1, d), np.float32)
    for k in (5, ef):
      o_ids, o_d, o_f, o_cnt = ix.search(q, k, ef, counters=True)
      assert o_ids[0, 0] == len(rows) - 1
      e.load_index(p)
      g_ids, g_d, g_f, stats = _device_search(e, q, k, ef)
      assert (g_f == o_f).all() and (g_ids == o_ids).all() and (g_d == o_d).all(), case
      assert (stats[:, 1:] == o_cnt[:, 1:4]).all()


@pytest.mark.parametrize("d,hi", [(12, 40), (70, 40), (160, 219)])
def test_integer_data_one_query_at_a_time(oracle, tmp_path, d, hi):
  n, k, mult = 3000, 10, 1 / np.log(8)
  x, q = integer_vectors(n, d, seed=3, hi=hi), integer_vectors(60, d, seed=4, hi=hi)
  ix = oracle.OracleIndex("l2").build(x, _levels(n, mult, 5), 8, 16, 60, mult)
  p = str(tmp_path / "i.idx")
  ix.save(p)
  e = _engine(tmp_path, dist_type="l2", max_m=8, max_m0=16)
  answered = 0
  for ef in (130, 200, 300, 500):
    o_ids, o_d, o_f, o_cnt = ix.search(q, k, ef, counters=True)
    for r in range(len(q)):
      e.load_index(p)
      g_ids, g_d, g_f, stats = _device_search(e, q[r:r + 1], k, ef)
      assert (g_f == o_f[r]).all() and (g_ids[0] == o_ids[r]).all() and (g_d[0] == o_d[r]).all(), (ef, r)
      assert (stats[0, 1:] == o_cnt[r, 1:4]).all()
      answered += e.last_search_repeats == 0
  assert answered > 20  # (by the first pass, equal keys and all)
