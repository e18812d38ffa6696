"""A model of the lane arithmetic by which a list of offers enters the sorted set in one go (frontier_insert_all of
device_core.h): where each entry and each offer is written.  Entries pushed past the end are dropped by the kernel,
an offer is written wherever its place says; so every offer's place has to lie inside the 64 * NS words that are saved
and put back around it."""
import numpy as np
import pytest

LARGEST = np.float32(3.402823466e+38)


def stop(key):
  """finish_sum of device_core.h: an ordering key is never infinite."""
  return np.clip(np.float32(key), -LARGEST, LARGEST)


def insert_all(ns, ef, entries, offers):
  """(places of the offers, the set afterwards); entries: the keys in the set, ascending."""
  total = 64 * ns
  held = np.full(total, np.inf, np.float32)
  held[:total - ef] = -np.inf
  held[total - ef:total - ef + len(entries)] = entries
  place = np.array([total - np.count_nonzero(k < held) + np.count_nonzero(offers < k) for k in offers])
  after = np.full(total, np.nan, np.float32)
  for at, k in enumerate(held):
    to = at + np.count_nonzero(offers < k)
    if to < total:
      after[to] = k
  for at, k in zip(place, offers):
    if at < total:
      after[at] = k
  return place, after


@pytest.mark.parametrize("ns,ef", [(2, 128), (5, 300), (8, 512), (8, 400)])
@pytest.mark.parametrize("extreme", [[np.inf], [-np.inf], [np.inf, -np.inf]], ids=["above", "below", "both"])
def test_overflowed_distances_find_their_place(ns, ef, extreme):
  rng = np.random.default_rng(ef)
  entries = np.sort(rng.uniform(1.0, 2.0, 40).astype(np.float32))
  offers = np.concatenate([rng.uniform(0.0, 3.0, 11).astype(np.float32), stop(extreme)])
  rng.shuffle(offers)
  place, after = insert_all(ns, ef, entries, offers)
  assert place.min() >= 0 and place.max() < 64 * ns
  first = 64 * ns - ef
  together = np.sort(np.concatenate([entries, offers]))
  assert (after[first:first + together.size] == together).all()
  assert (after[first + together.size:] == np.inf).all() and (after[:first] == -np.inf).all()


def test_an_infinite_key_would_be_written_behind_the_set():
  """Why the keys stop short of it: nothing in the set compares above an infinity, the padding included."""
  place, _ = insert_all(5, 300, np.array([1.0], np.float32), np.array([0.5, np.inf], np.float32))
  assert place.max() >= 64 * 5
