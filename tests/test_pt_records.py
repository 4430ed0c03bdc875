"""The record ring of the chained parallel-tempering exchange, replayed on the
host with the library's own row numbers (csmc_pt_record_rows, no device).

A system publishes its record of exchange x, sweeps, and reads its partner
slot's record only before its next Metropolis sweep; nothing else orders the
systems.  For every index distance of consecutive exchanges, with one system
held back at every exchange until no other can move, each read finds the
record it waits for."""
import random

import numpy as np
import pytest

from csmc import _lib

EXCHANGES = 24


def _rows(orr, swap):
    x, row = np.zeros(EXCHANGES, dtype=np.int64), np.zeros(EXCHANGES, dtype=np.int32)
    _lib.check(_lib.lib().csmc_pt_record_rows(orr, swap, EXCHANGES, _lib.ptr(x), _lib.ptr(row)))
    # every sweep at which the schedule exchanges, in turn
    do = orr or 1
    s = [k for k in range(int(x[-1]) * swap + 1) if k % do == 0 and k % swap == 0]
    assert [k // swap for k in s] == x.tolist()
    return x.tolist(), row.tolist()


def _partner(r, x, R):
    lo = r - (r - x % 2) % 2
    if lo < 0 or lo + 1 >= R:
        return None
    return lo + 1 if r == lo else lo


def _replay(R, x, row, held, at, seed):
    """every system through all exchanges; system `held` reads exchange `at`
    only when no other system can move.  Returns the first read that can never
    end, or None."""
    rng = random.Random(seed)
    rec = {}                      # (row, slot) -> the exchange index it carries
    slot, k, published = list(range(R)), [0] * R, [False] * R
    swapped = {}                  # (exchange, pair) -> the decision
    todo = set(range(R))
    while todo:
        moved = False
        order = sorted(todo, key=lambda s: (s == held and k[s] == at and published[s], rng.random()))
        for s in order:
            if not published[s]:
                rec[row[k[s]], slot[s]] = x[k[s]]
                published[s] = True
            else:
                p = _partner(slot[s], x[k[s]], R)
                if p is not None:
                    if rec.get((row[k[s]], p)) != x[k[s]]:
                        continue
                    if swapped.setdefault((k[s], min(p, slot[s])), rng.random() < 0.5):
                        slot[s] = p
                published[s] = False
                k[s] += 1
                if k[s] == EXCHANGES:
                    todo.discard(s)
            moved = True
            break
        if not moved:
            s = min(todo, key=lambda s: k[s])
            return s, x[k[s]]
    return None


@pytest.mark.parametrize("orr,swap", [(d, 1) for d in range(0, 18)] + [(16, 2), (40, 5), (80, 10), (10, 10), (6, 4)])
def test_no_record_is_lost(orr, swap):
    x, row = _rows(orr, swap)
    for R in (2, 3, 4, 7):
        for held in range(R):
            for at in (0, 1, 2, 5, 12):
                lost = _replay(R, x, row, held, at, seed=101 * held + at)
                assert lost is None, (R, held, at, lost)
