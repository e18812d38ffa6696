"""Python front end of the MI355X-native engine: class CuHNSW with the constructor options,
methods, argument meanings and return values of the reference's cuhnsw.pyhnsw.CuHNSW
(cuhnsw/pyhnsw.py:22-88 in js1010/cuhnsw).  Importing this module needs the native extension
(ImportError otherwise); there is no CPU fallback.

Behaviour kept from the reference on purpose, because callers rely on it:
  * `level_mult` unset -> 1 / ln(max_m) (cuhnsw/pyhnsw.py:26; the README says max_m0, the code wins);
  * dist_type aliases ip -> dot, cosine -> dot, euclidean -> l2.  The alias is resolved before
    anything looks at the name, so "cosine" does NOT switch `nrz` on (cuhnsw/pyhnsw.py:31-33 has
    a branch for that which can never fire); callers who want normalised rows pass nrz=True, as
    the reference's example does (examples/example1.py:38-44);
  * with `nrz` the rows are divided by their L2 norm in the array's own dtype; queries are never
    normalised (cuhnsw/pyhnsw.py:50-59, 79-88);
  * levels come from numpy's legacy global generator seeded with `seed`:
    int32(-ln(max(u, 1e-10)) * level_mult) (cuhnsw/pyhnsw.py:65-71) — `datasets.random_levels`;
  * search_knn raises ef_search to topk and returns (nns int32 [nq, topk], distances float32
    [nq, topk], found_cnt int32 [nq]); entries beyond found_cnt[i] are -1 / inf here
    (uninitialised in the reference);
  * the options reach the engine as a JSON file whose path is passed to `init`
    (cuhnsw/pyhnsw.py:34-46), so a failure to read them is an AssertionError as before.
"""
import contextlib
import json
import os
import tempfile

import numpy as np

from cuhnsw_amd import aux, datasets

try:
  from cuhnsw_amd.cuhnsw_bind import CuHNSWBind, copy_bytes
except ImportError as exc:  # pragma: no cover
  raise ImportError(
      "cuhnsw_amd: the native extension is missing (%s); build it with "
      "`python -m cuhnsw_amd.build`" % exc) from exc

_ALIASES = {"ip": "dot", "cosine": "dot", "euclidean": "l2"}
_KNOWN_DISTANCES = ("dot", "l2") + tuple(_ALIASES)
_MAX_BLOCK_DIM = 1024  # the reference's CUDA limit (32 warps of 32); validated, not used by the HIP kernels


def _resolve(raw):
  """Option table with defaults filled, the alias applied and the level multiplier set."""
  opt = aux.get_opt_as_proto(raw or {})
  if not opt.level_mult:
    opt.level_mult = 1.0 / np.log(opt.max_m)
  assert opt.dist_type in _KNOWN_DISTANCES, opt.dist_type
  opt.dist_type = _ALIASES.get(opt.dist_type, opt.dist_type)
  assert 0 < opt.block_dim <= _MAX_BLOCK_DIM and opt.block_dim % 32 == 0, \
      "invalid block dim (%d, warp size: 32)" % opt.block_dim
  return opt


@contextlib.contextmanager
def _option_file(opt):
  """The option table as the JSON file `init` reads; removed again whatever happens."""
  fd, path = tempfile.mkstemp(prefix="cuhnsw_opt_", suffix=".json")
  try:
    with os.fdopen(fd, "w") as f:
      json.dump(aux.proto_to_dict(opt), f, indent=2)
    yield path
  finally:
    os.remove(path)


def _copy_of(data):
  """data.copy(), on several threads where that pays."""
  if type(data) is not np.ndarray or data.nbytes < 8 << 20 or not data.flags.c_contiguous or data.dtype.hasobject:
    return data.copy()
  rows = np.empty(data.shape, data.dtype)
  copy_bytes(rows, data)
  return rows


class CuHNSW:
  """HNSW index built and searched on the GPU."""

  def __init__(self, opt=None):
    self.opt = _resolve(opt)
    self.logger = aux.get_logger("cuhnsw", self.opt.py_log_level)
    self.data = None
    self.obj = CuHNSWBind()
    with _option_file(self.opt) as path:
      self.logger.debug("options: %s", aux.proto_to_dict(self.opt))
      assert self.obj.init(path.encode("utf8")), "failed to load %s" % path

  # -- data ------------------------------------------------------------------------------------
  def set_data(self, data):
    rows = _copy_of(data)
    if self.opt.nrz:
      if self.opt.dist_type == "l2":
        self.logger.warning("it is not common to set nrz = True and dist_type = l2")
      rows /= np.linalg.norm(rows, axis=1)[:, None]
    self.data = rows
    self.logger.info("data shape: %d x %d", *rows.shape)
    self.obj.set_data(rows)

  def set_random_levels(self):
    levels = datasets.random_levels(self.data.shape[0], self.opt.level_mult, seed=self.opt.seed)
    self.obj.set_random_levels(levels)

  # -- index -----------------------------------------------------------------------------------
  def build(self):
    self.set_random_levels()
    self.obj.build_graph()

  def save_index(self, fpath):
    self.obj.save_index(fpath.encode("utf-8"))

  def load_index(self, fpath):
    self.obj.load_index(fpath.encode("utf-8"))

  # -- search ----------------------------------------------------------------------------------
  def search_knn(self, qdata, topk, ef_search):
    queries = np.ascontiguousarray(qdata, dtype=np.float32)
    rows = 1 if queries.ndim == 1 else queries.shape[0]
    out = (np.empty((rows, topk), np.int32), np.empty((rows, topk), np.float32), np.empty(rows, np.int32))
    self.obj.search_knn(queries, topk, max(topk, ef_search), *out)
    return out
