"""Ordering keys that stop at the largest finite number, in the model of how a list of offers enters the sorted set in one go
(frontier_insert_all of device_core.h): the set's padding is infinite, and an offer has to find a place in front of it."""
import numpy as np
import pytest

from test_list_merge_model import in_the_set, insert_all

LARGEST = np.float32(3.402823466e+38)


def stop(key):
  """finish_sum of device_core.h: an ordering key is never infinite."""
  return np.clip(np.float32(key), -LARGEST, LARGEST)


def merged(ns, ef, entries, offers):
  """The keys of a set of these entries (ascending) with the offers."""
  after, _ = insert_all(ns, ef, len(entries), in_the_set(ns, ef, entries), np.zeros(64 * ns, int), offers, np.zeros(len(offers), int))
  return after[0]


@pytest.mark.parametrize("ns,ef", [(2, 128), (5, 300), (8, 512), (8, 400)])
@pytest.mark.parametrize("extreme", [[np.inf], [-np.inf], [np.inf, -np.inf]], ids=["above", "below", "both"])
def test_overflowed_distances_find_their_place(ns, ef, extreme):
  rng = np.random.default_rng(ef)
  entries = np.sort(rng.uniform(1.0, 2.0, 40).astype(np.float32))
  offers = np.concatenate([rng.uniform(0.0, 3.0, 11).astype(np.float32), stop(extreme)])
  rng.shuffle(offers)
  after = merged(ns, ef, entries, offers)
  first = 64 * ns - ef
  together = np.sort(np.concatenate([entries, offers]))
  assert (after[first:first + together.size] == together).all()
  assert (after[first + together.size:] == np.inf).all() and (after[:first] == -np.inf).all()


def test_an_infinite_key_would_be_written_behind_the_set():
  """Why the keys stop short of it: nothing in the set compares above an infinity, the padding included."""
  held, ids = in_the_set(5, 300, np.array([1.0], np.float32)), np.zeros(320, int)
  after, _ = insert_all(5, 300, 1, held, ids, np.array([0.5, np.inf], np.float32), np.array([7, 8]))
  first = 64 * 5 - 300
  assert (after[0][first:first + 2] == [0.5, 1.0]).all() and after[1][first] == 7 and not (after[1] == 8).any()
