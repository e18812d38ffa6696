"""A model of how a list of offers enters the sorted set in one go (frontier_insert_all of device_core.h), step by step as the
lanes do it: the offers put in order, each entry's count of offers before it found by halving, each offer's place from the
last entry of every count, everything moved through 64 * (NS + 1) words.  An offer's equal sends them the other way, also
where the set's end comes between the two; farther out the dropped ones are no candidates any more.  Into a full set equal
entries that were there before are no reason."""
import numpy as np
import pytest


def insert_all(ns, ef, size, held, ids, offers, offer_ids):
  """(keys and ids of the set afterwards, or None where equal keys send the offers the other way; every index of the
  offers' list that was read)"""
  total, n = 64 * ns, len(offers)
  touched = []
  less = np.array([np.count_nonzero(offers < k) for k in offers])
  keys = np.where(np.arange(64) < n, -np.inf, np.inf).astype(np.float32)
  keys[less] = offers
  listed = np.zeros(64, int)
  listed[less] = offer_ids
  if np.isneginf(keys).any():
    return None, touched
  before = np.zeros(total, int)
  half = 1 << (n.bit_length() - 1)
  while half:
    touched += list(before + half - 1)
    before += np.where(keys[before + half - 1] < held, half, 0)
    half >>= 1
  assert max(touched) < 64
  room, room_ids = np.full(total + 64, np.nan, np.float32), np.zeros(total + 64, int)
  counts = np.zeros(64, int)
  last_of_its_count = np.append(before[1:] != before[:-1], True)
  counts[before[last_of_its_count]] = np.flatnonzero(last_of_its_count) + 1
  place = np.maximum.accumulate(counts)[:n] + np.arange(n)
  to = np.arange(total) + before
  assert len(set(to) | set(place)) == total + n and max(to.max(), place.max()) < total + 64
  room[to], room_ids[to] = held, ids
  room[place], room_ids[place] = keys[:n], listed[:n]
  after = room[:total]
  finite = np.isfinite(after)
  last = room[total - ef + min(size + n, ef) - 1]
  if size < ef:
    refused = (after[1:] == after[:-1])[finite[1:]].any()
  else:
    refused = any(key <= last and at > 0 and room[at - 1] == key for at, key in zip(place, keys))
  if refused:
    return None, touched
  return (after, room_ids[:total]), touched


def in_the_set(ns, ef, entries):
  held = np.full(64 * ns, np.inf, np.float32)
  held[:64 * ns - ef] = -np.inf
  held[64 * ns - ef:64 * ns - ef + len(entries)] = entries
  return held


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
    held = in_the_set(ns, ef, entries)
    ids = np.full(64 * ns, -1)
    first = 64 * ns - ef
    ids[first:first + size] = np.arange(size)
    after, _ = insert_all(ns, ef, size, held, ids, offers, 1000 + np.arange(n))
    both = np.concatenate([entries, offers])
    order = np.argsort(both, kind="stable")
    inside = both[order][:ef]
    bound = inside[-1]
    within = both[both <= bound]
    if len(set(within)) < len(within) or len(set(offers)) < n:
      assert after is None, "equal keys within the bound, or of two offers"
      continue
    assert after is not None
    assert (after[0][first:first + len(inside)] == inside).all() and (after[0][:first] == -np.inf).all()
    assert (after[0][first + len(inside):] == np.inf).all()
    assert (after[1][first:first + len(inside)] == np.concatenate([np.arange(size), 1000 + np.arange(n)])[order][:ef]).all()


@pytest.mark.parametrize("at", range(7))
def test_equal_keys_on_both_sides_of_the_sets_end_are_refused(at):
  """The dropped one is as close as the bound: a candidate still, which the offer would be lost as."""
  ns, ef = 3, 150
  entries = np.arange(10, 1510, 10).astype(np.float32)
  offers = np.insert(np.arange(5, 65, 10).astype(np.float32), at, np.float32(1440))
  held = in_the_set(ns, ef, entries)
  assert insert_all(ns, ef, ef, held, np.arange(64 * ns), offers, np.arange(7))[0] is None
  held[-9] = held[-8]  # (1 430 twice, a pair that was there before: the offers below it enter all the same)
  after = insert_all(ns, ef, ef, held, np.arange(64 * ns), np.delete(offers, at), np.arange(6))[0]
  assert after is not None and np.count_nonzero(after[0] == held[-8]) == 2
  held[-9] = 1420
  offers[at] = 1450  # (pushed out together with its equal: beyond the bound, both dead)
  assert insert_all(ns, ef, ef, held, np.arange(64 * ns), offers, np.arange(7))[0] is not None
