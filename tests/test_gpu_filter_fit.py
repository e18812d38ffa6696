"""The size of the visited filter is a matter of the search alone, not of what was searched before it: the evaluations that a batch
counts (which say what the filter forgot) are those of an engine that has made no other search."""
import numpy as np
import pytest

from helpers import gauss_mixture
from test_gpu_search import _device_search, _engine, _levels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("before,then", [
    ((600, 1000), (10, 1000)),    # the same filter to begin with; only the second answer leaves it room to be halved in
    ((600, 600), (600, 700)),     # answers that are longer than either filter is to begin with
    ((200, 300), (200, 256)),
], ids=["answers", "filters", "five"])
def test_a_batch_counts_the_same_evaluations_whatever_was_searched_before(tmp_path, before, then):
  n, d, nq = 40000, 24, 1500
  x, q = gauss_mixture(n, d, seed=3), gauss_mixture(nq, d, seed=4)
  p, counts, answers = str(tmp_path / "f.idx"), [], []
  for searches in ((then,), (before, then)):
    e = _engine(tmp_path, dist_type="l2", max_m=16, max_m0=32, ef_construction=60, heuristic_coef=0.0)
    if not counts:
      e.set_data(x)
      e.set_random_levels(_levels(n, 1 / np.log(16), 5))
      e.build_graph()
      e.save_index(p)
    else:
      e.load_index(p)
    e.set_tunable("fast_path", 2)
    for k, ef in searches:
      ids, _, _, stats = _device_search(e, q, k, ef)
    counts.append(stats[:, 0])
    answers.append(ids)
    print("searched", searches, int(counts[-1].sum()), flush=True)
  assert (answers[0] == answers[1]).all()
  assert (counts[0] == counts[1]).all()
