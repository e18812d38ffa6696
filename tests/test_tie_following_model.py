"""Pins the argument behind the sorted-set search's handling of equal keys (the rules in
search_level_fast, cuhnsw_amd/csrc/device_core.h), on the CPU: a plain-Python statement of
those rules is run on small random graphs whose integer coordinates make distances tie all
the time, and whenever it does NOT give a query up, its answer — ids, distances and the number
of expansions and evaluations — must be what the oracle's literal hnswlib search
(two std::priority_queues) returns.  A rule that lets an order-dependent case through shows
up here as a mismatch within a few thousand trials.  (The rules include the one that follows the two
twins of an eviction out of two equal largest keys through instead of giving the query up.)

The same model also keeps the TRAIL the first pass leaves for the literal pass (struct Trail in device_core.h): the
entries accepted hop by hop, no records but two markers around the hops of a group of equal keys, nothing after the
twins of an eviction come up.  A second model, hnswlib's search on literal libstdc++ heaps, replays a given-up
query from that trail — recorded hops take their accepted entries from the records and evaluate nothing, the
others are made for real — and must arrive at the oracle's answer and hop count: what a hop accepts does not depend
on the order in which a followed-through group was expanded, which is what the replay on the GPU rests on."""
import numpy as np
import pytest

from helpers import graph_cut_between_equals

INF = float("inf")


def sorted_set_search(keys_of, rows, ep, k, ef, trail=None, together=None, cut_rule=True):
  """Returns None when given up, else (ids, keys, hops, evaluations, met equal keys).  trail: a dict that receives
  "rec" (the records and markers) and "hops" (the expansions they cover).  together: so many offers of one hop or more
  enter a full set in one go (frontier_insert_all), unless one of them has the key of another or of an entry; cut_rule:
  also where one of the two is the set's last entry afterwards and the other the first that was pushed out."""
  tr = {"rec": [], "on": True, "own": False, "hops": 0}

  def stop(h):                            # the trail ends: h expansions are complete
    if tr["on"]:
      tr["on"] = False
      tr["hops"] = h
    if trail is not None:
      trail["rec"], trail["hops"] = tr["rec"], tr["hops"]

  hop_node = None                         # the node the current hop expanded (None: the seed)
  S = [[keys_of(ep), ep, False]]          # sorted by key, equal keys in order of arrival
  seen = {ep}
  have_tie = in_group = False
  calm = True                             # no equal keys at work: the tie-free loop runs (none of the bookkeeping below)
  watch = []                              # ...keeping off the waiting entries that have an equal in the set (at most four)
  group_key = 0.0
  group_edge = INF                        # smallest key rejected or evicted while the group is expanded
  ek_min = INF
  ghosts = 0                              # evictions that had equal largest keys to choose from
  ghost = None                            # the entry the single such eviction pushed out
  twin_phase = False                      # its twins are being expanded: no offer may be accepted
  hops = 0
  offers = []
  while True:
    accepted = []
    passing = [o for o in offers if S[-1][0] > o[0]]
    if together is not None and calm and len(S) >= ef and len(passing) >= together:
      new = {node for _, node in passing}
      merged = sorted(S + [[key, node, False] for key, node in passing], key=lambda e: e[0])  # (an offer behind its equal)
      reach = len(merged) if cut_rule else ef
      equal = any(a[0] == b[0] <= merged[ef - 1][0] and b[1] in new for a, b in zip(merged[:reach], merged[1:reach]))
      equal = equal or len({key for key, _ in passing}) < len(passing)
      if not equal and not (watch and merged[ef - 1][0] <= max(w[0] for w in watch)):
        S = merged[:ef]
        offers = []
        sorted_set_search.entered_together += 1
        sorted_set_search.entered_beside_equal_keys += have_tie
    for key, node in offers:
      full = len(S) >= ef
      if full and not (S[-1][0] > key):
        if in_group:
          group_edge = min(group_edge, key)
        continue
      if any(e[0] == key for e in S):
        have_tie = True
        calm = False                          # the rules for equal keys apply from this very offer on
      if calm and full and watch and S[-1][0] <= max(w[0] for w in watch):
        calm = False                          # an eviction that reaches a watched entry or its equal
      twins = not calm and full and S[-1][0] == S[-2][0]   # eviction with equal largest keys to choose from
      last = list(S[-1])
      pos = len(S)
      while pos > 0 and S[pos - 1][0] > key:
        pos -= 1
      S.insert(pos, [key, node, False])
      accepted.append((key, node))
      if len(S) > ef:
        if in_group:
          group_edge = min(group_edge, S[-1][0])
          if S[-1][0] == group_key and not S[-1][2]:
            stop(hops - 1)
            return None                       # a member of the group pushed out before its turn
        S.pop()
      if twins:
        ek_min = min(ek_min, last[0])
        ghost = last
        # three equal largest keys, a second such eviction, or the whole set asked for: the plain rule
        ghosts += 2 if (S[-1][0] == S[-2][0] or k >= ef) else 1
      if twin_phase:
        stop(hops - 1)
        return None                           # which twin goes first now decides whether the other is expanded at all
    if tr["on"] and not tr["own"] and hop_node is not None:
      tr["rec"] += [("rec", hop_node, node, key, hops) for key, node in accepted]
    was_in_group = in_group
    pick = next((i for i, e in enumerate(S) if not e[2]), -1)
    d = S[pick][0] if pick >= 0 else INF
    if in_group and pick >= 0 and d < group_key:
      # a closer candidate turned up inside the group: it is expanded before the rest of the group under
      # any order; a group within the group is not followed
      if any((not e[2]) and e[0] == d for i, e in enumerate(S) if i != pick):
        stop(hops)
        return None
    elif in_group and d != group_key:
      # the group is through: with another order of its members an offer or an entry whose key
      # equals the bound reached now could have ended up on the other side of it, and with the bound
      # below the group's key a member popped late would not have been expanded at all
      if len(S) >= ef and (group_edge == S[-1][0] or S[-1][0] < group_key):
        stop(hops)
        return None
      in_group = False
    if pick < 0:
      stop(hops)
      if len(S) >= ef and S[-1][0] >= ek_min:
        # an evicted twin is still a live candidate of hnswlib
        if ghosts != 1:
          return None
        if not ghost[2]:
          ghost[2] = True                     # expanded although it is not in the set; nothing of it may be accepted
          twin_phase = True
          hops += 1
          offers = []
          for nb in rows[ghost[1]]:
            if nb not in seen:
              seen.add(nb)
              offers.append((keys_of(nb), nb))
          continue
      break
    if calm and pick >= 0 and any(w is S[pick] for w in watch):
      calm = False                            # a watched entry's turn
    if have_tie and not calm:
      if d >= ek_min:
        # the twin the set kept (its last entry: the key is the bound)
        others = any((not e[2]) and e[0] == d for i, e in enumerate(S) if i != pick)
        if ghosts == 1 and not in_group and not others:
          twin_phase = True
        else:
          stop(hops)
          return None
      if not in_group and not twin_phase:
        in_group = any((not e[2]) and e[0] == d for i, e in enumerate(S) if i != pick)
        group_key = d
        group_edge = INF
    if twin_phase:
      stop(hops)
    elif tr["on"] and in_group != was_in_group:
      tr["rec"].append(("own" if in_group else "back", hops + 1))
      tr["own"] = in_group
    hop_node = S[pick][1]
    S[pick][2] = True
    hops += 1
    offers = []
    for nb in rows[S[pick][1]]:
      if nb not in seen:
        seen.add(nb)
        offers.append((keys_of(nb), nb))
    # equal keys do no harm while none of them that still waits is expanded or pushed out (unless the whole set
    # is the answer): once the set is full the tie-free loop takes over again until the next offer meets an equal
    # key, a watched entry's turn comes or an eviction reaches one
    if not calm and k < ef and len(S) >= ef and not in_group and not twin_phase and (ghosts == 0 or S[-1][0] < ek_min):
      watch = [e for i, e in enumerate(S)
               if (not e[2]) and ((i > 0 and S[i - 1][0] == e[0]) or (i + 1 < len(S) and S[i + 1][0] == e[0]))]
      if len(watch) <= 4:
        calm = True
        sorted_set_search.calmed_down_past_a_ghost += ghosts != 0
        ghosts, ghost, ek_min = 0, None, INF  # (an eviction out of equal largest keys on record is beyond the bound: dead)
        sorted_set_search.calmed_down += 1
        sorted_set_search.calmed_down_watching += bool(watch)
  T = min(k, len(S))
  if have_tie and T < len(S) and S[T - 1][0] == S[T][0]:
    return None                               # equal keys across the cut: the result heap's choice (the trail is complete)
  best = sorted((e[0], e[1]) for e in S[:T])  # equal keys among the k best: listed by label
  sorted_set_search.answered_after_twins += bool(twin_phase)
  return [e[1] for e in best], [e[0] for e in best], hops, len(seen), have_tie


sorted_set_search.answered_after_twins = 0    # (statistics for the test below: the twin rule has to be exercised)
sorted_set_search.calmed_down = 0             # (and so has the return to the tie-free loop,
sorted_set_search.calmed_down_watching = 0    # with and without entries to watch,
sorted_set_search.calmed_down_past_a_ghost = 0  # and after an eviction out of equal largest keys)
sorted_set_search.entered_together = 0        # (and offers that entered a full set in one go,
sorted_set_search.entered_beside_equal_keys = 0  # also once equal keys have met)


def _push_heap(h, value):
  """std::push_heap after push_back, max-heap on value[0] (bits/stl_heap.h, __push_heap)."""
  h.append(value)
  hole = len(h) - 1
  while hole > 0:
    parent = (hole - 1) // 2
    if not (h[parent][0] < value[0]):
      break
    h[hole] = h[parent]
    hole = parent
  h[hole] = value


def _pop_heap(h):
  """std::pop_heap + pop_back (bits/stl_heap.h, __pop_heap / __adjust_heap); returns the former top."""
  top = h[0]
  value = h.pop()
  n = len(h)
  if n == 0:
    return top
  hole = child = 0
  while child < (n - 1) // 2:
    child = 2 * (child + 1)
    if h[child][0] < h[child - 1][0]:
      child -= 1
    h[hole] = h[child]
    hole = child
  if n % 2 == 0 and child == (n - 2) // 2:
    child = 2 * (child + 1)
    h[hole] = h[child - 1]
    hole = child - 1
  while hole > 0:                             # __push_heap(first, hole, 0, value)
    parent = (hole - 1) // 2
    if not (h[parent][0] < value[0]):
      break
    h[hole] = h[parent]
    hole = parent
  h[hole] = value
  return top


def literal_search(keys_of, rows, ep, k, ef, trail=None):
  """hnswlib's searchBaseLayerST + searchKnn on two literal priority queues (hnswalg.h).  With a trail: the
  expansions it covers take their accepted entries from its records and evaluate nothing (their neighbours only
  become visited), except inside the stretches its markers set apart, which are made for real.
  Returns (ids, keys, hops, evaluations made)."""
  rec = trail["rec"] if trail else []
  covered = trail["hops"] if trail else 0
  at = 0
  own = False
  top, cand = [], []                          # (key, id) max-heap; (-key, id) max-heap
  d0 = keys_of(ep)
  _push_heap(top, (d0, ep))
  _push_heap(cand, (-d0, ep))
  lower = d0
  visited = {ep}
  hops = evals = 0
  while cand:
    if -cand[0][0] > lower:
      break
    node = _pop_heap(cand)[1]
    hops += 1
    offers = None
    if hops <= covered:
      while at < len(rec) and rec[at][0] != "rec" and rec[at][1] == hops:
        own = rec[at][0] == "own"
        at += 1
      if not own:
        offers = []
        while at < len(rec) and rec[at][0] == "rec" and rec[at][4] == hops:
          assert rec[at][1] == node, "the trail names another node for this hop"
          offers.append((rec[at][3], rec[at][2]))
          at += 1
        visited.update(rows[node])
    if offers is None:
      offers = []
      for nb in rows[node]:
        if nb not in visited:
          visited.add(nb)
          evals += 1
          offers.append((keys_of(nb), nb))
    for key, nb in offers:
      if len(top) < ef or lower > key:
        if hops <= covered and not own:
          pass                                # (a recorded entry: it passes, as it did in the first pass)
        _push_heap(cand, (-key, nb))
        _push_heap(top, (key, nb))
        if len(top) > ef:
          _pop_heap(top)
        lower = top[0][0]
      else:
        assert not (hops <= covered and not own), "a recorded entry is turned away"
  while len(top) > k:
    _pop_heap(top)
  best = sorted(top)
  return [e[1] for e in best], [e[0] for e in best], hops, evals


@pytest.mark.parametrize("seed", list(range(4)))
def test_given_up_queries_replayed_from_the_trail_match_the_oracle(oracle, seed):
  rng = np.random.default_rng(5000 + seed)
  replayed = with_markers = covered_hops = all_hops = plain = 0
  for graph in range(60):
    n = int(rng.integers(12, 60))
    dim = int(rng.integers(1, 4))
    hi = int(rng.integers(3, 30))
    x = rng.integers(0, hi, (n, dim)).astype(np.float32)
    deg = int(rng.integers(2, 7))
    links0 = np.zeros((n, 1 + 8), np.uint32)
    rows = []
    for i in range(n):
      others = [j for j in range(n) if j != i]
      nb = list(rng.choice(others, size=min(deg, len(others)), replace=False))
      nb.append((i + 1) % n)
      nb = list(dict.fromkeys(int(v) for v in nb if v != i))[:8]
      links0[i, 0] = len(nb)
      links0[i, 1:1 + len(nb)] = nb
      rows.append(nb)
    ix = oracle.OracleIndex("l2").from_arrays(x, np.zeros(n, np.int32), links0, np.zeros(0, np.uint32),
                                              max_m=4, max_m0=8, maxlevel=0, enterpoint=0)
    q = rng.integers(0, hi, (24, dim)).astype(np.float32)
    for k, ef in ((1, 1), (2, 3), (3, 5), (4, 4), (5, 8), (2, 12)):
      ids, dists, found, cnt = ix.search(q, k, ef, convention="hnswlib", counters=True)
      for r in range(q.shape[0]):
        keys_of = lambda node, qq=q[r]: float(np.float32(((qq - x[node]) ** 2).sum()))
        f = found[r]
        if r < 2:
          # the literal model by itself is the oracle's search (this pins the Python heaps)
          l_ids, l_keys, l_hops, l_evals = literal_search(keys_of, rows, 0, k, ef)
          assert l_ids == list(ids[r, :f]) and l_keys == list(dists[r, :f]) and l_hops == cnt[r, 1]
          assert l_evals + 1 == cnt[r, 0]
          plain += 1
        trail = {}
        if sorted_set_search(keys_of, rows, 0, k, ef, trail) is not None or not trail.get("rec") or trail["hops"] == 0:
          continue
        l_ids, l_keys, l_hops, l_evals = literal_search(keys_of, rows, 0, k, ef, trail)
        assert l_ids == list(ids[r, :f]) and l_keys == list(dists[r, :f]), (seed, graph, r, k, ef)
        assert l_hops == cnt[r, 1], (seed, graph, r, k, ef)
        replayed += 1
        with_markers += any(e[0] != "rec" for e in trail["rec"])
        covered_hops += trail["hops"]
        all_hops += l_hops
  # given-up queries with a trail are common on this data, many of their trails lead through a group of equal
  # keys, and the trails cover a good part of the expansions
  assert replayed > 1000 and with_markers > 500 and plain > 500, (replayed, with_markers, plain)
  assert covered_hops * 4 > all_hops, (covered_hops, all_hops)


@pytest.mark.parametrize("seed", list(range(6)) + [141])   # 141: the case that showed the need for the rule on the group's edge
def test_rules_never_let_an_order_dependent_case_through(oracle, seed):
  rng = np.random.default_rng(1000 + seed)
  answered = given_up = answered_with_ties = 0
  for graph in range(60):
    n = int(rng.integers(12, 60))
    dim = int(rng.integers(1, 4))
    hi = int(rng.integers(3, 30))
    x = rng.integers(0, hi, (n, dim)).astype(np.float32)
    deg = int(rng.integers(2, 7))
    links0 = np.zeros((n, 1 + 8), np.uint32)
    rows = []
    for i in range(n):
      others = [j for j in range(n) if j != i]
      nb = list(rng.choice(others, size=min(deg, len(others)), replace=False))
      nb.append((i + 1) % n)                  # a ring keeps everything reachable
      nb = list(dict.fromkeys(int(v) for v in nb if v != i))[:8]
      links0[i, 0] = len(nb)
      links0[i, 1:1 + len(nb)] = nb
      rows.append(nb)
    ix = oracle.OracleIndex("l2").from_arrays(x, np.zeros(n, np.int32), links0, np.zeros(0, np.uint32),
                                              max_m=4, max_m0=8, maxlevel=0, enterpoint=0)
    q = rng.integers(0, hi, (24, dim)).astype(np.float32)
    for k, ef in ((1, 1), (2, 3), (3, 5), (4, 4), (5, 8), (2, 12)):
      ids, dists, found, cnt = ix.search(q, k, ef, convention="hnswlib", counters=True)
      for r in range(q.shape[0]):
        keys_of = lambda node, qq=q[r]: float(np.float32(((qq - x[node]) ** 2).sum()))
        for together in (None, 1, 3):
          got = sorted_set_search(keys_of, rows, 0, k, ef, together=together)
          if got is None:
            given_up += together is None
            continue
          m_ids, m_keys, hops, evals, tied = got
          if together is None:
            answered += 1
            answered_with_ties += bool(tied)
          f = found[r]
          assert f == len(m_ids)
          assert list(ids[r, :f]) == m_ids, (seed, graph, r, k, ef, together)
          assert list(dists[r, :f]) == m_keys
          assert cnt[r, 1] == hops and cnt[r, 0] == evals, (seed, graph, r, k, ef, together)
  # both outcomes are exercised, and so are searches that met equal keys and were still answered, some of them
  # by following the twins of an eviction through
  assert answered > 1000 and given_up > 100 and answered_with_ties > 300, (answered, given_up, answered_with_ties)
  assert sorted_set_search.answered_after_twins > 0
  assert sorted_set_search.calmed_down > 100 and sorted_set_search.calmed_down_watching > 100
  assert sorted_set_search.calmed_down_past_a_ghost > 20
  assert sorted_set_search.entered_together > 100 and sorted_set_search.entered_beside_equal_keys > 20


@pytest.mark.parametrize("seed", range(3))
def test_a_cut_between_two_equal_keys_is_noticed(oracle, seed):
  """Offers that push a full set's entries out up to one whose equal is among them: hnswlib expands both, and what the
  equal that was dropped leads to is in the answer.  (Without the rule for the cut nearly every such search is answered
  wrongly, and none given up.)"""
  rng = np.random.default_rng(7000 + seed)
  wrong = {True: 0, False: 0}
  for _ in range(100):
    ef = int(rng.integers(10, 30))
    coordinates, rows = graph_cut_between_equals(rng, ef, width=64)
    x = np.array(coordinates, np.float32)[:, None]
    links0 = np.zeros((len(rows), 1 + 64), np.uint32)
    for i, nb in enumerate(rows):
      links0[i, 0] = len(nb)
      links0[i, 1:1 + len(nb)] = nb
    ix = oracle.OracleIndex("l2").from_arrays(x, np.zeros(len(rows), np.int32), links0, np.zeros(0, np.uint32),
                                              max_m=32, max_m0=64, maxlevel=0, enterpoint=0)
    k = int(rng.integers(1, 8))
    ids, dists, found, cnt = ix.search(np.zeros((1, 1), np.float32), k, ef, convention="hnswlib", counters=True)
    f = found[0]
    assert ids[0, 0] == len(rows) - 1          # the nearest is where only the dropped equal leads
    for cut_rule in (True, False):
      got = sorted_set_search(lambda node: float(x[node, 0] ** 2), rows, 0, k, ef, together=3, cut_rule=cut_rule)
      if got is None:
        continue
      wrong[cut_rule] += not (got[0] == list(ids[0, :f]) and got[1] == list(dists[0, :f]) and got[2] == cnt[0, 1])
  assert wrong[True] == 0 and wrong[False] > 60, wrong
