"""Searches that expand several candidates at a time (tie_free_phase in cuhnsw_amd/csrc/device_core.h) against the
oracle -- ids, distances, found counts and hop counters -- where that can go wrong: link rows so full that a batch's new
nodes exceed one pass of 64 lanes (it is cut short), rows of a few ids, sets just above the sizes the batches start at,
sets that a search barely fills, equal keys inside a batch, and every query layout."""
import numpy as np
import pytest

from helpers import gauss_mixture, integer_vectors
from test_gpu_search import _check_parity, _engine, _levels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,dist,max_m,max_m0,kind,efs", [
    (3000, 50, "dot", 32, 64, "gauss", (129, 300)),     # up to eight full rows of 64 ids
    (3000, 16, "l2", 31, 63, "scattered", (130, 512)),  # no clusters: next to every neighbour is new
    (2000, 100, "dot", 2, 4, "gauss", (200, 320)),      # rows of four ids
    (400, 96, "l2", 16, 32, "gauss", (390, 400, 420)),  # the set holds nearly every node there is
    (3000, 128, "l2", 16, 32, "int", (150, 330)),       # equal keys in most batches
    (1500, 300, "l2", 16, 32, "scattered", (140, 600)), # rows too long for registers
], ids=["full64", "full63", "thin", "whole", "ties", "long"])
def test_batched_hops_match_the_oracle(oracle, tmp_path, n, d, dist, max_m, max_m0, kind, efs):
  def draw(m, seed):
    if kind == "int":
      return integer_vectors(m, d, seed=seed, hi=30)
    if kind == "scattered":
      return np.random.default_rng(seed).standard_normal((m, d)).astype(np.float32)
    return gauss_mixture(m, d, seed=seed, normalise=dist == "dot")
  x, q = draw(n, 5), draw(80, 6)
  mult = 1.0 / np.log(max(max_m, 4))
  ix = oracle.OracleIndex(dist).build(x, _levels(n, mult, 7), max_m, max_m0, 80, mult)
  p = str(tmp_path / "i.idx")
  ix.save(p)
  e = _engine(tmp_path, dist_type=dist, max_m=max_m, max_m0=max_m0)
  e.load_index(p)
  for ef in efs:
    print("batched hops", n, d, kind, ef, flush=True)
    _check_parity(oracle, ix, e, q, 10, ef)
