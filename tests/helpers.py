"""Shared helpers of the test-suite (small synthetic data, tiny hand-built graphs)."""
import numpy as np


def gauss_mixture(n, d, centres=32, seed=0, sigma=0.5, normalise=True):
  rng = np.random.default_rng(seed)
  c = rng.standard_normal((centres, d)).astype(np.float32)
  x = c[rng.integers(0, centres, n)] + np.float32(sigma) * rng.standard_normal((n, d)).astype(np.float32)
  if normalise:
    x /= np.linalg.norm(x, axis=1, keepdims=True)
  return x.astype(np.float32)


def integer_vectors(n, d, seed=0, hi=8):
  """Small-integer coordinates: squared L2 distances are exact in fp32 in any
  summation order and collide often (ties)."""
  rng = np.random.default_rng(seed)
  return rng.integers(0, hi, (n, d)).astype(np.float32)


def ring_graph(n, max_m0, hops=(1, 2)):
  """Level-0 links of a connected ring: node i links to i±h for h in hops."""
  links0 = np.zeros((n, 1 + max_m0), dtype=np.uint32)
  for i in range(n):
    nb = []
    for h in hops:
      for s in (+1, -1):
        j = (i + s * h) % n
        if j != i and j not in nb:
          nb.append(j)
    nb = nb[:max_m0]
    links0[i, 0] = len(nb)
    links0[i, 1:1 + len(nb)] = nb
  return links0


def graph_cut_between_equals(rng, ef, width):
  """(coordinates on a line, level-0 links) of a graph on which the search for the origin from node 0 fills its set of ef
  entries and then expands a node that offers as many closer entries as there are beyond one of the set, E, and among them
  O, as far from the origin as E.  E is the set's last entry then and O the first outside it, or the other way round; only O
  leads to the last node, the nearest of all.  At most `width` links a node; squared distances are exact."""
  chain = -(-(ef - 1) // width)                  # nodes that bring the set's entries in, the next one and in the end the offers
  m = int(rng.integers(2, min(width, ef - chain) - 1))      # offers beside O, and entries beyond E (node 0 the farthest)
  lows = ef - chain - m - 1                      # entries closer than E
  places = np.sort(2 * rng.choice(np.arange(50, 50 + 3 * (lows + 2 * m + 1)), lows + 2 * m + 1, replace=False))
  closer, e, beyond = rng.permutation(places[:lows + m]), places[lows + m], places[lows + m + 1:]
  coordinates, rows = [], []

  def add(distance, side=None):
    coordinates.append(int(distance) * (side or int(rng.choice([-1, 1]))))
    rows.append([0])                             # (back to where the search began: nothing new)
    return len(rows) - 1

  add(beyond[-1])
  entries = [(v, None) for v in np.concatenate([closer[:lows], beyond[:-1]])] + [(e, 1)]
  entries = [entries[i] for i in rng.permutation(len(entries))]
  at = 0
  for step in range(chain):
    nb = [add(*v) for v in entries[:width - 1]]
    entries = entries[width - 1:]
    nb.insert(int(rng.integers(0, len(nb) + 1)), add(3 + 2 * (chain - step)))
    rows[at], at = nb, max(nb, key=lambda i: -abs(coordinates[i]))
  assert not entries and len(rows) == ef
  nb = [add(v) for v in closer[lows:]]
  o = add(e, -1)
  nb.insert(int(rng.integers(0, m)), o)          # (not the last, when the bound has come down to E)
  rows[at] = nb
  rows[o] = [0, len(rows)]
  add(1)
  return coordinates, rows


def recall(found_ids, truth_ids):
  k = truth_ids.shape[1]
  return float(np.mean([len(set(a) & set(b)) / k for a, b in zip(found_ids, truth_ids)]))
