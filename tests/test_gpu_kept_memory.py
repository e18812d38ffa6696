"""What an engine keeps allocated between calls, and that it can be had back."""
import struct

import numpy as np
import pytest

from cuhnsw_amd import capi
from helpers import gauss_mixture

pytestmark = pytest.mark.gpu


def _free():
  import torch
  torch.cuda.synchronize()
  return torch.cuda.mem_get_info()[0]


def _index(e, x):
  e.set_data(x)
  e.set_random_levels(np.zeros(x.shape[0], np.int32))
  e.build_graph()


def test_workspace_is_given_back(tmp_path):
  n, d = 300_000, 24
  x = gauss_mixture(n, d, seed=91)
  p = str(tmp_path / "a.idx")
  e = capi.Engine()
  e.set_tunable("trails", 0)               # (their buffers belong to the searches)
  _index(e, x)                             # kept: a build's work space of this size is 100 MB and more
  kept = _free()
  e.set_tunable("keep_workspace", 0)
  assert _free() - kept > 100 << 20
  bare = _free()
  _index(e, x)
  e.save_index(p)
  assert abs(_free() - bare) < 8 << 20
  # a load that is refused once the whole file is on the GPU
  raw = bytearray(open(p, "rb").read())
  record = 4 * 24 + 4 + 4 * d + 8
  struct.pack_into("<I", raw, 96 + (n - 1) * record, 25)
  open(p, "wb").write(bytes(raw))
  with pytest.raises(RuntimeError, match="link count"):
    e.load_index(p)
  assert abs(_free() - bare) < 8 << 20
  e.set_tunable("keep_workspace", 1)
  _index(e, x)
  assert bare - _free() > 100 << 20
  e.close()
  assert _free() > bare



def test_engines_together_keep_a_bounded_amount():
  """Uploading rows that are padded on their way takes 32 MB of pinned blocks and as much on the device: the engines of
  a process keep 256 MB of the former together, and those beyond that keep neither."""
  x = gauss_mixture(2000, 50, seed=92)
  before = _free()
  engines = []
  for _ in range(14):
    e = capi.Engine()
    e.set_tunable("trails", 0)
    e.set_data(x)
    engines.append(e)
  assert before - _free() < 330 << 20      # (fourteen times 32 MB would be 448)
  for e in engines[::5] + engines[-1:]:    # whether they keep the blocks or not
    _index(e, x)
    ids, _, _ = e.search_knn(x[:3], 1, 50)
    assert list(ids[:, 0]) == [0, 1, 2]
  for e in engines:
    e.close()
  assert before - _free() < 64 << 20
