"""Small batches, which a workgroup of wavefronts per query searches (team_phase in cuhnsw_amd/csrc/device_core.h), against the oracle
-- ids, distances, found counts and hop counters -- at the batch sizes where the split over the GPU changes (a query, a
round of workgroups and the query beyond, the last size that is searched so and the first that is not), for every query
layout, sets of the smallest and largest size, and link rows whose lists need one to seven eights of lanes, or more than fit."""
import numpy as np
import pytest

from helpers import gauss_mixture, integer_vectors
from test_gpu_search import _device_search, _engine, _levels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,dist,max_m,max_m0,kind,ef", [
    (4000, 50, "dot", 12, 24, "gauss", 300),
    (4000, 100, "dot", 16, 32, "gauss", 64),       # the smallest set
    (3000, 24, "l2", 16, 32, "gauss", 1000),       # the largest, which most nodes go into
    (3000, 180, "l2", 16, 32, "scattered", 200),
    (2500, 300, "l2", 16, 32, "gauss", 150),       # rows too long for registers
    (2500, 16, "l2", 32, 64, "scattered", 300),    # link rows of 64 ids, nearly all of them new at first
    (2000, 64, "dot", 2, 4, "gauss", 100),         # of four
    (3000, 128, "l2", 16, 32, "int", 128),         # equal keys in most searches
], ids=["dot50", "small", "large", "d180", "long", "full64", "thin", "ties"])
def test_batches_that_leave_the_machine_idle_match_the_oracle(oracle, tmp_path, n, d, dist, max_m, max_m0, kind, ef):
  def draw(m, seed):
    if kind == "int":
      return integer_vectors(m, d, seed=seed, hi=30)
    if kind == "scattered":
      return np.random.default_rng(seed).standard_normal((m, d)).astype(np.float32)
    return gauss_mixture(m, d, seed=seed, normalise=dist == "dot")
  k = 10
  x, q = draw(n, 8), draw(1025, 9)
  mult = 1.0 / np.log(max(max_m, 4))
  ix = oracle.OracleIndex(dist).build(x, _levels(n, mult, 7), max_m, max_m0, 80, mult)
  p = str(tmp_path / "i.idx")
  ix.save(p)
  e = _engine(tmp_path, dist_type=dist, max_m=max_m, max_m0=max_m0)
  o_ids, o_d, o_f, o_cnt = ix.search(q, k, ef, counters=True)
  for nq in (1, 3, 255, 256, 257, 513, 769, 1024, 1025):
    print("teams", d, kind, ef, nq, flush=True)
    for first in sorted({0, 1025 - nq}):
      part = slice(first, first + nq)
      e.load_index(p)  # (what earlier batches handed over is forgotten)
      g_ids, g_d, g_f, stats = _device_search(e, q[part], k, ef)
      assert (g_f == o_f[part]).all() and (g_ids == o_ids[part]).all() and (g_d == o_d[part]).all(), nq
      assert (stats[:, 1:] == o_cnt[part, 1:4]).all(), nq


@pytest.mark.parametrize("n,d,dist,max_m,max_m0,efc,kind,extra", [
    (5200, 16, "l2", 8, 16, 60, "int", {}),                                   # equal keys everywhere
    (4500, 100, "dot", 32, 64, 130, "gauss", dict(heuristic_coef=0.25)),      # link rows of 64 ids
    (2500, 300, "l2", 3, 6, 100, "gauss", dict(save_remains=True)),           # many levels; rows too long for registers
    (4500, 180, "l2", 16, 32, 700, "scattered", {}),                          # the largest set
], ids=["ties", "full64", "levels", "large"])
def test_index_built_by_teams_is_the_one_built_without(tmp_path, n, d, dist, max_m, max_m0, efc, kind, extra):
  """Batches of a build go through every size up to a quarter of the nodes; a filter of a given size takes the wavefront alone."""
  if kind == "int":
    x = integer_vectors(n, d, seed=3, hi=6)
  elif kind == "scattered":
    x = np.random.default_rng(4).standard_normal((n, d)).astype(np.float32)
  else:
    x = gauss_mixture(n, d, seed=5, normalise=dist == "dot")
  levels = _levels(n, 1.0 / np.log(max_m), 6)
  files = []
  for entries in (0, 16384):
    options = dict(dict(heuristic_coef=0.0), dist_type=dist, max_m=max_m, max_m0=max_m0, ef_construction=efc)
    options.update(extra)
    e = _engine(tmp_path, **options)
    e.set_tunable("filter_entries", entries)
    e.set_data(x)
    e.set_random_levels(levels)
    print("built by teams", kind, entries, flush=True)
    e.build_graph()
    p = tmp_path / "b.idx"
    e.save_index(str(p))
    files.append(p.read_bytes())
  assert files[0] == files[1]
