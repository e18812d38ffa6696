"""A batch's descents, four queries to a wavefront, at the batch sizes where its grid changes (256 CUs: one round of four
wavefronts on a SIMD, of five, two rounds of five, and one query more than each): ids, found counts and the counters of the
descents against the oracle."""
import numpy as np
import pytest

from helpers import gauss_mixture
from test_gpu_search import _device_search, _engine, _levels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,dist", [(24, "dot"), (100, "dot"), (24, "l2"), (100, "l2")])
def test_descents_of_large_batches_match_the_oracle(oracle, tmp_path, d, dist):
  n, k, ef, mult = 3000, 3, 16, 1 / np.log(4)   # (levels enough for several steps of every descent)
  x, q = gauss_mixture(n, d, seed=5, normalise=dist == "dot"), gauss_mixture(40964, d, seed=6, normalise=dist == "dot")
  ix = oracle.OracleIndex(dist).build(x, _levels(n, mult, 7), 4, 8, 40, mult)
  p = str(tmp_path / "d.idx")
  ix.save(p)
  e = _engine(tmp_path, dist_type=dist, max_m=4, max_m0=8)
  e.load_index(p)
  o_ids, o_d, o_f, o_cnt = ix.search(q, k, ef, counters=True)
  for nq in (16384, 16385, 20480, 20481, 40960, 40961, 40964):
    print("descents", d, dist, nq, flush=True)
    g_ids, g_d, g_f, stats = _device_search(e, q[:nq], k, ef)
    assert (g_ids == o_ids[:nq]).all() and (g_f == o_f[:nq]).all() and (g_d == o_d[:nq]).all(), nq
    assert (stats[:, 2:] == o_cnt[:nq, 2:4]).all(), nq
