"""The work that users of this engine wait for, as cases that can be timed: indexing a data set (vectors in,
index file out), bringing a stored index into service, and answering query batches of every size, through the
public entry points (`CuHNSW` for host arrays, `capi.Engine.search_knn_device` for buffers that are on the GPU).

Data follow the laws of the benchmark configurations (cuhnsw_amd/datasets.py): Gaussian mixtures, normalised
("angular", dot product), rounded to small integers ("sift", squared L2, equal distances everywhere) or clipped to
[0, 1] ("gist", squared L2); they are drawn on the GPU, so that making them is quick.
"""
import json
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from cuhnsw_amd import CuHNSW, capi, datasets

_ANGULAR = dict(law="angular", max_m=12, max_m0=24, efc=110, coef=0.0, half=False)
_SIFT = dict(law="sift", max_m=16, max_m0=32, efc=200, coef=0.0, half=False)
_GIST = dict(law="gist", max_m=16, max_m0=32, efc=200, coef=0.0, half=False)
_DEEP = dict(law="angular", max_m=16, max_m0=32, efc=150, coef=0.0, half=False)


def listed():
  return [
      # one user's query against a small index: nothing but latency counts
      dict(_ANGULAR, name="one_query", kind="search", api="host", n=100_000, d=50, nq=1, topk=10, ef=300),
      # a handful of requests collected by a server, on integer descriptors
      dict(_SIFT, name="few_queries", kind="search", api="host", n=200_000, d=128, nq=32, topk=10, ef=128),
      # the small angular configuration, whole
      dict(_ANGULAR, name="angular_1k", kind="search", api="host", n=100_000, d=50, nq=1000, topk=10, ef=300),
      # the headline configuration: 10 000 queries that are on the GPU already
      dict(_ANGULAR, name="angular_10k", kind="search", api="device", n=1_183_514, d=50, nq=10_000, topk=10, ef=300),
      # descriptors with equal distances in most searches, from and to host arrays
      dict(_SIFT, name="sift_10k", kind="search", api="host", n=500_000, d=128, nq=10_000, topk=10, ef=128),
      # long rows: each distance is a few memory lines, a batch that leaves room on the machine
      dict(_GIST, name="gist_1k", kind="search", api="device", n=100_000, d=960, nq=1000, topk=10, ef=300),
      # one large offline batch with many results per query
      dict(_DEEP, name="deep_100k", kind="search", api="device", n=1_000_000, d=96, nq=100_000, topk=100, ef=256),
      # half-precision storage, a size that is no multiple of anything
      dict(_ANGULAR, name="half_odd", kind="search", api="host", n=345_678, d=101, nq=5003, topk=7, ef=77, half=True),
      # a small data set indexed and saved, over and over (experiments, per-tenant indexes)
      dict(_ANGULAR, name="index_20k", kind="index", n=20_000, d=50),
      # integer descriptors with the option table's default heuristic_coef
      dict(_SIFT, name="index_sift", kind="index", n=200_003, d=128, coef=0.25),
      # the headline configuration's build, from the caller's array to the file
      dict(_ANGULAR, name="index_1m", kind="index", n=1_183_514, d=50),
      # a server starts: index file read, first thousand queries answered
      dict(_DEEP, name="load_500k", kind="load", api="host", n=500_000, d=96, nq=1000, topk=10, ef=128),
  ]


def _log_int(rng, low, high):
  return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _evaluations(ef):
  """Distances of one level-0 search, about (counted on the benchmark configurations: 1 268 at ef 300, 830 at 128)."""
  return 400 + 3 * ef


def _tests(efc):
  """Distances of one insertion, about: its search, and ten pairs per candidate when its neighbours are selected."""
  return _evaluations(efc) + 10 * efc


def draw(rng):
  kind = rng.choice(["search"] * 6 + ["index"] * 2 + ["load"])
  c = dict(rng.choice([_ANGULAR, _SIFT, _GIST, _DEEP]), kind=kind)
  c["d"] = _log_int(rng, 200, 1000) if c["law"] == "gist" else _log_int(rng, 24, 200)
  c["n"] = min(_log_int(rng, 20_000, 1_183_514), 96_000_000 // c["d"])
  c["coef"] = rng.choice([0.0, 0.0, 0.25])
  c["half"] = rng.random() < 0.15
  if kind == "index":
    c["n"] = min(c["n"], 1_183_514 * _tests(110) * 50 // (_tests(c["efc"]) * c["d"]))
  else:
    c["api"] = rng.choice(["host", "device"]) if kind == "search" else "host"
    c["topk"] = _log_int(rng, 1, 100)
    c["ef"] = max(_log_int(rng, 32, 512), c["topk"])
    most = 100_000 * _evaluations(256) * 96 // (_evaluations(c["ef"]) * c["d"])
    c["nq"] = _log_int(rng, 1, min(100_000, most)) if kind == "search" else _log_int(rng, 1, 2000)
  return c


def _mixture(c, seed):
  """n + nq rows of the case's law, on the GPU: the data set and, from the same mixture, the queries."""
  g = torch.Generator(device="cuda")
  g.manual_seed(1_000_003 * int(seed) + 17)
  rows, d = c["n"] + c.get("nq", 0), c["d"]
  centres = max(20, c["n"] // 1000)
  if c["law"] == "angular":
    mid, sigma = torch.randn(centres, d, generator=g, device="cuda"), 0.5
  elif c["law"] == "sift":
    mid, sigma = 128.0 * torch.rand(centres, d, generator=g, device="cuda"), 20.0
  else:
    mid, sigma = torch.rand(centres, d, generator=g, device="cuda"), 0.05
  x = torch.empty(rows, d, device="cuda")
  for s in range(0, rows, 1 << 18):
    e = min(rows, s + (1 << 18))
    pick = torch.randint(0, centres, (e - s,), generator=g, device="cuda")
    y = mid[pick] + sigma * torch.randn(e - s, d, generator=g, device="cuda")
    if c["law"] == "angular":
      y /= y.norm(dim=1, keepdim=True)
    elif c["law"] == "sift":
      y = y.clamp_(0.0, 218.0).round_()
    else:
      y = y.clamp_(0.0, 1.0)
    x[s:e] = y
  return x[:c["n"]].cpu().numpy(), x[c["n"]:].clone()


def _options(c):
  return dict(dist_type="dot" if c["law"] == "angular" else "l2", max_m=c["max_m"], max_m0=c["max_m0"],
              ef_construction=c["efc"], heuristic_coef=c["coef"], py_log_level=1)


def _index(c):
  h = CuHNSW(_options(c))
  if c["half"]:
    h.obj.set_tunable("fp16_storage", 1)
  return h


def _engine(c, data):
  """The same index behind the C interface, for callers whose queries are on the GPU."""
  e = capi.Engine()
  o = dict(_options(c), level_mult=1.0 / np.log(c["max_m"]))
  fd, path = tempfile.mkstemp(suffix=".json")
  with os.fdopen(fd, "w") as f:
    json.dump(o, f)
  assert e.init(path) == 0
  os.remove(path)
  if c["half"]:
    e.set_tunable("fp16_storage", 1)
  e.set_data(data)
  e.set_random_levels(datasets.random_levels(c["n"], o["level_mult"]))
  e.build_graph()
  return e


class _Folder:
  """A folder for index files that goes away with its state; in memory where there is room, so that a disk's
  moods are not what is timed."""

  def __init__(self):
    shm = "/dev/shm"
    roomy = os.path.isdir(shm) and os.access(shm, os.W_OK) and shutil.disk_usage(shm).free > 8 << 30
    self.path = tempfile.mkdtemp(prefix="cuhnsw_", dir=shm if roomy else None)

  def file(self):
    return os.path.join(self.path, "index.hnsw")

  def __del__(self):
    shutil.rmtree(self.path, ignore_errors=True)


def prepare(case, seed):
  c = dict(case)
  data, queries = _mixture(c, seed)
  if c["kind"] == "index":
    return dict(case=c, data=data, index=_index(c), folder=_Folder())
  if c["kind"] == "load":
    folder = _Folder()
    made = _index(c)
    made.set_data(data)
    made.build()
    made.save_index(folder.file())
    return dict(case=c, queries=queries.cpu().numpy(), index=_index(c), folder=folder)
  if c["api"] == "device":
    nq, k = c["nq"], c["topk"]
    return dict(case=c, queries=queries, engine=_engine(c, data),
                ids=torch.empty((nq, k), dtype=torch.int32, device="cuda"),
                distances=torch.empty((nq, k), dtype=torch.float32, device="cuda"),
                found=torch.empty(nq, dtype=torch.int32, device="cuda"))
  h = _index(c)
  h.set_data(data)
  h.build()
  return dict(case=c, queries=queries.cpu().numpy(), index=h)


def run(state):
  c = state["case"]
  if c["kind"] == "index":
    h = state["index"]
    h.set_data(state["data"])
    h.build()
    h.save_index(state["folder"].file())
    return np.memmap(state["folder"].file(), dtype=np.int32, mode="r")  # (a file of whole 32-bit words)
  if c["kind"] == "load":
    h = state["index"]
    h.load_index(state["folder"].file())
    return h.search_knn(state["queries"], c["topk"], c["ef"])
  if c["api"] == "device":
    state["engine"].search_knn_device(state["queries"].data_ptr(), c["nq"], c["topk"], c["ef"], state["ids"].data_ptr(),
                                      state["distances"].data_ptr(), state["found"].data_ptr())
    return state["ids"], state["distances"], state["found"]
  return state["index"].search_knn(state["queries"], c["topk"], c["ef"])


def work(case):
  """Vectors, links and files once each; two operations per element of each distance.  A search needs the rows
  its queries evaluate: a row per evaluation, or each row of the index once where that is less."""
  c = dict(case)
  n, d = c["n"], c["d"]
  row = d * (2 if c["half"] else 4)
  whole = n * (row + 4 * c["max_m0"])
  file = n * (4 * d + 4 * c["max_m0"] + 16)
  if c["kind"] == "index":
    return dict(bytes=4 * n * d + whole + file, flops=2.0 * d * n * _tests(c["efc"]))
  nq, ef = c["nq"], c["ef"]
  gathered = min(nq * (_evaluations(ef) * row + ef * 4 * c["max_m0"]), whole)
  total = gathered + nq * (4 * d + 8 * c["topk"] + 4) + (file + whole if c["kind"] == "load" else 0)
  return dict(bytes=total, flops=2.0 * d * nq * _evaluations(ef))


def tolerance(case):  # pylint: disable=unused-argument
  """Searches return the ids an exact statement of the algorithm returns, and distances summed in a fixed order;
  an index file is the same file every time."""
  return "exact"
