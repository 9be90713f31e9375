"""The ping-pong GEMM's order of DMAs, waits, barriers and LDS reads, walked through on the CPU.

``csrc/gemm_pingpong.h`` overlaps the tiles of a block: a tile's last k tiles
fetch the next tile's first ones, and its two groups of waves run half a phase
apart. A wave's wait covers the DMAs that it issued itself, so a unit may be
read only behind a barrier that every wave reached after waiting for its share,
and its slot may be refilled only behind a barrier that every wave reached after
reading it. Here both groups' programs are written out for sequences of full
and half tiles (at most 128 rows), with the wait counts of the header, and every
read and refill is checked against all waves.
"""

from __future__ import annotations

import itertools
import re
from pathlib import Path

import pytest

HEADER = Path(__file__).resolve().parents[1] / "pluggy_amd" / "csrc" / "gemm_pingpong.h"
UNITS = ("N0", "A0", "N1", "A1")  # in the order of the phases that refill them


def waits() -> dict[str, int]:
    found = dict(re.findall(r"constexpr int (kPp\w+) = (\d+);", HEADER.read_text()))
    assert sorted(found) == ["kPpFull", "kPpFullHalf", "kPpHalf"]
    return {k: int(v) for k, v in found.items()}


def program(second: bool, halves: list[bool], nk: int, tail: bool, w: dict[str, int], last: int):
    """One wave's events over a block's tiles: ("dma" | "read", (k tile in the stream, unit)),
    ("wait", instructions left in flight) and ("barrier", None). ``last``: the wait of a full
    tile's last phase before a half one."""
    ev = []

    def dma(half, s, *units):
        ev.extend(("dma", (s, u)) for u in units if not (half and u == "A1"))

    def read(s, *units):
        ev.extend(("read", (s, u)) for u in units)

    def wait(n):
        ev.append(("wait", n))

    def barrier():
        ev.append(("barrier", None))

    halves = halves + [True]  # past the last tile: no rows
    for s in range(2):
        dma(halves[0], s, *UNITS)
    wait(0)
    barrier()
    read(0, "N0")
    barrier()
    lean_end = nk - 3 if tail else nk - 2
    for t in range(len(halves) - 1):
        if second:
            barrier()
        for kt in range(nk):
            s, half = t * nk + kt, halves[t + (kt >= nk - 2)]  # of what this k tile's DMAs fetch
            if halves[t]:
                read(s, "A0", "N1")
                dma(half, s + 2, "N0")
                if kt > 0:
                    wait(w["kPpHalf"])
                barrier(), barrier()
                read(s + 1, "N0")
                dma(half, s + 2, "A0", "N1", "A1")
                if kt > 0:
                    wait(w["kPpHalf"])
                barrier(), barrier()
                continue
            for p, unit in enumerate((("A0", s), ("N1", s), ("A1", s), ("N0", s + 1))):
                read(unit[1], unit[0])
                dma(half, s + 2, UNITS[p])
                few = kt >= nk - 2 and half
                if 2 <= kt < lean_end:
                    wait(w["kPpFull"])
                elif kt > 1 or (p >= 2 and kt == 1):
                    wait(w["kPpFull"] if not few else last if p == 3 and kt == nk - 1 else w["kPpFullHalf"])
                barrier(), barrier()
        if not second:
            barrier()
        wait(0)  # then the epilogue, without a barrier
    return ev


def hazards(halves, nk, tail, w, last):
    landed, reads, fills = [], [], []  # per group: unit -> barriers behind the wait / the read / the refill
    counts = []
    for second in (False, True):
        at, flight, b = {}, [], 0
        rd, fl = {}, {}
        for kind, arg in program(second, halves, nk, tail, w, last):
            if kind == "barrier":
                b += 1
            elif kind == "dma":
                flight += [arg, arg]  # two instructions a unit
                fl[arg] = b
            elif kind == "read":
                rd[arg] = b
            else:
                while len(flight) > arg:
                    at[flight.pop(0)] = b  # the second instruction's wait stays
        landed.append(at), reads.append(rd), fills.append(fl), counts.append(b)
    assert counts[0] == counts[1], "both groups pass the same barriers"
    bad = []
    total = nk * len(halves)
    for rd in reads:
        for unit, b in rd.items():
            if unit[0] < total and any(unit not in at or at[unit] >= b for at in landed):
                bad.append(("read before it landed", unit))
    for fl in fills:
        for (s, u), b in fl.items():
            if any(rd[(s - 2, u)] >= b for rd in reads if (s - 2, u) in rd):
                bad.append(("refilled before it was read", (s, u)))
    return bad


@pytest.mark.parametrize("tail", [False, True])
@pytest.mark.parametrize("nk", [2, 3, 4, 5, 6, 9])
def test_every_read_and_refill_is_ordered(nk, tail):
    w = waits()
    for halves in itertools.product([False, True], repeat=4):
        assert not hazards(list(halves), nk, tail, w, w["kPpHalf"]), (halves, nk, tail)


def test_the_walk_sees_an_unordered_read():
    """A full tile's last wait as for any other phase: the half tile after it
    reads the second half of its columns before other waves' share has landed."""
    w = waits()
    assert ("read before it landed", (4, "N1")) in hazards([False, True], 4, False, w, w["kPpFullHalf"])
    assert not hazards([False, False], 4, False, w, w["kPpFullHalf"])
