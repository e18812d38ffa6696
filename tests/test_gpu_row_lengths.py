"""Row lengths around the ends of the distance passes' chunks and fetch rounds: the chunks past a row's end are fetched
(chunk 0 in their place) and must not count, whatever lies there.  Every search path against the oracle on the file of a
build on the GPU, which runs the same passes; distances are compared bit for bit (one order of summation on both sides)."""
import numpy as np
import pytest

from helpers import gauss_mixture
from test_gpu_search import _check_parity, _engine, _levels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True], ids=["fp32", "fp16"])
@pytest.mark.parametrize("dist", ["dot", "l2"])
@pytest.mark.parametrize("d", [1, 4, 61, 64, 65, 127, 128, 129, 256, 257, 513, 960])
def test_row_lengths(oracle, tmp_path, dist, d, half):
  n, mult = 700, 1 / np.log(8)
  x = gauss_mixture(n, d, seed=d, normalise=False) + np.float32(3.0)  # (nothing near zero: a chunk too many shows)
  q = gauss_mixture(24, d, seed=d + 1, normalise=False)
  e = _engine(tmp_path, dist_type=dist, max_m=8, max_m0=24, ef_construction=60)
  e.set_tunable("fp16_storage", 1 if half else 0)
  e.set_data(x)
  e.set_random_levels(_levels(n, mult, 5))
  e.build_graph()
  p = str(tmp_path / "r.idx")
  e.save_index(p)
  ix = oracle.OracleIndex(dist).load(p)
  assert ix.validate() == 0
  for k, ef in ((10, 100), (5, 300)):
    _check_parity(oracle, ix, e, q, k, ef, dup_bound=None)
