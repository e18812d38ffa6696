"""A model of how a list of offers enters the sorted set in one go (frontier_insert_all of device_core.h), step by step as the
lanes do it: the offers put in order, each entry's count of offers before it found by halving, each offer's place from the
last entry of every count, everything moved through 64 * (NS + 1) words."""
import numpy as np
import pytest


def insert_all(ns, ef, size, held, offers):
  """(the set afterwards, or None where equal keys send the offers the other way; every index that was written or read)"""
  total, n = 64 * ns, len(offers)
  touched = []
  less = np.array([np.count_nonzero(offers < k) for k in offers])
  keys = np.where(np.arange(64) < n, -np.inf, np.inf).astype(np.float32)
  keys[less] = offers
  if np.isneginf(keys).any():
    return None, touched
  before = np.zeros(total, int)
  half = 1 << (n.bit_length() - 1)
  while half:
    touched += list(before + half - 1)
    before += np.where(keys[before + half - 1] < held, half, 0)
    half >>= 1
  assert max(touched) < 64
  room = np.zeros(total + 64, np.float64)
  counts = np.zeros(64, int)
  last_of_its_count = np.append(before[1:] != before[:-1], True)
  counts[before[last_of_its_count]] = np.flatnonzero(last_of_its_count) + 1
  place = np.maximum.accumulate(counts)[:n] + np.arange(n)
  to = np.arange(total) + before
  assert len(set(to) | set(place)) == total + n and max(to.max(), place.max()) < total + 64
  room[to] = held
  room[place] = keys[:n]
  after = room[:total]
  finite = np.isfinite(after)
  if (after[1:] == after[:-1])[finite[1:]].any():
    return None, touched
  return after.astype(np.float32), touched


@pytest.mark.parametrize("ns,ef", [(2, 65), (2, 128), (3, 150), (4, 256), (5, 300), (8, 512)])
def test_merged_lists_are_the_smallest_of_both(ns, ef):
  rng = np.random.default_rng(ns * 1000 + ef)
  for case in range(400):
    n = int(rng.integers(4, 64))
    full = case % 2 == 1
    size = ef if full else int(rng.integers(0, ef - min(n, ef) + 1))
    if not full and size + n > ef:
      continue
    draw = (lambda m: rng.integers(0, 4000, m).astype(np.float32)) if case % 3 == 0 else (lambda m: rng.normal(size=m).astype(np.float32))
    entries = np.unique(draw(4 * size + 8))[:size]
    rng.shuffle(entries)
    entries = np.sort(entries)
    size = len(entries)
    offers = draw(n) - (np.float32(9) if case % 5 == 0 else np.float32(0))
    held = np.full(64 * ns, np.inf, np.float32)
    held[:64 * ns - ef] = -np.inf
    held[64 * ns - ef:64 * ns - ef + size] = entries
    after, _ = insert_all(ns, ef, size, held, offers)
    both = np.sort(np.concatenate([entries, offers]))
    if len(set(both)) < len(both):
      # (equal keys: refused, unless all but one of them fell off the end)
      if after is None:
        continue
      both = np.sort(np.unique(both))
    assert after is not None
    want = both[:ef]
    first = 64 * ns - ef
    assert (after[first:first + len(want)] == want).all() and (after[:first] == -np.inf).all()
    assert (after[first + len(want):] == np.inf).all()
