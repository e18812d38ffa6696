"""Index files packed, checked and unpacked on the GPU: byte for byte what the CPU oracle writes."""
import os
import struct

import numpy as np
import pytest

from cuhnsw_amd import capi
from helpers import gauss_mixture

pytestmark = pytest.mark.gpu


def oracle_file(oracle, path, n, d, max_m, max_m0, marked=()):
  levels = (-np.log(np.random.default_rng(n).uniform(size=n)) * 0.5).astype(np.int32)
  ix = oracle.OracleIndex("dot").build(gauss_mixture(n, d, seed=d), levels, max_m, max_m0, 20, 0.5)
  ix.save(path)
  record = 4 * max_m0 + 4 + 4 * d + 8
  raw = bytearray(open(path, "rb").read())
  for i in marked:
    raw[96 + i * record + 2] |= 1    # hnswlib's delete mark
  open(path, "wb").write(bytes(raw))
  return bytes(raw), record


@pytest.mark.parametrize("n,d,max_m,max_m0,marked", [
    (1, 1, 2, 3, ()), (3, 64, 2, 64, (2,)), (257, 7, 4, 65, ()), (6001, 50, 12, 24, (0, 31, 32, 6000)),
    (9001, 101, 20, 70, ()),         # three blocks and a rest on the way up and down
])
def test_load_and_save_keep_every_byte(oracle, tmp_path, n, d, max_m, max_m0, marked):
  p, q = str(tmp_path / "a.idx"), str(tmp_path / "b.idx")
  raw, record = oracle_file(oracle, p, n, d, max_m, max_m0, marked)
  e = capi.Engine()
  e.load_index(p)
  assert (e.num_data, e.num_dims, e.num_deleted) == (n, d, len(marked))
  open(q, "wb").write(b"x" * (len(raw) + 12345))   # a longer file that is there already
  e.save_index(q)
  assert open(q, "rb").read() == raw
  # a file with a bad last record (count, then id) is refused and the index that was resident stays
  for at, word, what in ((0, max_m0 + 1, "link count"), (4, n, "out of range")):
    bad = bytearray(raw)
    struct.pack_into("<I", bad, 96 + (n - 1) * record, 1)
    struct.pack_into("<I", bad, 96 + (n - 1) * record + at, word)
    open(p, "wb").write(bytes(bad))
    with pytest.raises(RuntimeError, match=what):
      e.load_index(p)
  e.save_index(q)
  assert open(q, "rb").read() == raw


@pytest.mark.parametrize("d", [3, 32, 50, 129])
@pytest.mark.parametrize("half", [0, 1])
def test_rows_go_up_padded_and_come_back(tmp_path, d, half):
  n = 20011                        # several blocks of rows at d = 129
  x = gauss_mixture(n, d, seed=d)
  e = capi.Engine()
  e.set_tunable("fp16_storage", half)
  e.set_data(x)
  e.set_random_levels(np.zeros(n, np.int32))
  e.set_tunable("build_batch", n)
  e.build_graph()
  p = str(tmp_path / "a.idx")
  e.save_index(p)
  record = 4 * 24 + 4 + 4 * d + 8
  body = np.frombuffer(open(p, "rb").read()[96:96 + n * record], np.uint8).reshape(n, record)
  rows = np.ascontiguousarray(body[:, 100:100 + 4 * d]).view(np.float32)
  np.testing.assert_array_equal(rows, x.astype(np.float16).astype(np.float32) if half else x)
  assert os.path.getsize(p) == 96 + n * record + 4 * n
