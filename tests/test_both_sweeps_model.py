"""A CPU model of how the workgroups of a launch that holds both sweeps start and wait (csrc/fcr.hip, both_sweeps_kernel).

Row tiles and column tiles of a pair are workgroups of one launch; a column tile needs the values of row tiles.  The GPU is a few
dies of a few places; every die takes its share of a launch in order, as places get free, and knows nothing of the others.  Beside it
runs a launch whose workgroups hold their places until all of them have started (a single sweep that a graph replays).  The model
runs both under random interleavings:

  * a column tile that waits for values whoever was to compute them, which relies on row tiles having started first, can wait for a row
    tile that never starts: its die's places are held by the other launch, whose last workgroups wait for the places of column tiles,
  * a column tile that first looks whether its row tiles have begun, and takes one that has not in hand itself, never does, whatever
    the order in which workgroups start; every tile's values are stored, and a tile that was taken by another is stored twice at most
    by its own workgroup and one other.
"""
import random

import pytest


class Gpu:
    def __init__(self, dies, places, rng):
        self.free = [places] * dies
        self.queues = [[[] for _ in range(dies)]]
        self.rng = rng
        self.running = []

    def launch(self, groups):
        """groups: generators, dealt to the dies in turn; a stream of its own."""
        queue = [[] for _ in self.free]
        for i, g in enumerate(groups):
            queue[i % len(self.free)].append(g)
        self.queues.append(queue)

    def run(self, steps=20000):
        """True once everything has ended."""
        for _ in range(steps):
            choices = [("start", q, d) for q in self.queues for d, waiting in enumerate(q) if waiting and self.free[d] > 0]
            choices += [("step", i, None) for i in range(len(self.running))]
            if not choices:
                return True
            kind, a, d = self.rng.choice(choices)
            if kind == "start":
                self.running.append((a[d].pop(0), d))
                self.free[d] -= 1
            else:
                group, d = self.running[a]
                if next(group, "end") == "end":
                    self.running.pop(a)
                    self.free[d] += 1
        return False


NOT_YET, BEGUN = "not yet", "begun"


def sweep_rows(words, tile, stored):
    for _ in range(3):
        yield
    words[tile] = tile
    stored[tile] += 1


def row_place(words, tile, stored):
    if words[tile] == NOT_YET:
        words[tile] = BEGUN
    yield
    yield from sweep_rows(words, tile, stored)


def column_place(words, needs, stored, look, patience):
    while look:
        tile = next((t for t in needs if words[t] == NOT_YET), None)
        if tile is None:
            break
        if patience > 0:
            patience -= 1
            yield
            continue
        words[tile] = BEGUN          # compare and swap: in one step
        yield from sweep_rows(words, tile, stored)
    for tile in needs:
        while words[tile] in (NOT_YET, BEGUN):
            yield
        assert words[tile] == tile
        yield


def team_place(team, size):
    team.append(1)
    while len(team) < size:
        yield


def one(seed, look, columns_first=False):
    rng = random.Random(seed)
    dies, places, rows, cols = 2, 2, 6, 6
    words, stored = [NOT_YET] * rows, [0] * rows
    gpu, team = Gpu(dies, places, rng), []
    row_places = [row_place(words, t, stored) for t in range(rows)]
    col_places = [column_place(words, range(t, rows), stored, look, rng.randrange(3)) for t in range(cols)]
    gpu.launch(col_places + row_places if columns_first else row_places + col_places)
    gpu.launch([team_place(team, dies * places) for _ in range(dies * places)])
    ended = gpu.run()
    if ended:
        assert all(1 <= n <= 2 for n in stored) and words == list(range(rows))
    return ended


@pytest.mark.parametrize("columns_first", [False, True])
def test_every_wait_ends_whatever_starts_first(columns_first):
    assert all(one(seed, True, columns_first) for seed in range(300))


def test_waiting_for_rows_that_have_not_begun_can_last_for_ever():
    assert not all(one(seed, False) for seed in range(300))
