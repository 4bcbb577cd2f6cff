"""Launch-shape autotuner for a batch arena: the tile, then the flux threads per cell once few
slots run.

The main launch-shape choice of the time step is the tile: threads per block of every cell,
face and wall kernel (64, 128 or 256; each slot's ranges are padded to it, so a block never
spans two meshes).  Small tiles spread a latency-bound arena over more compute units; large
tiles cut padding and block scheduling overhead once the arena fills the chip.  The tuner
builds the same arena at every candidate tile, times `trials` trial replays after `warmup`
and keeps the fastest, except that a larger tile within 1% of the fastest wins the tie: it
has fewer blocks, less padding and fewer faces evaluated by two tiles, and its batches end
sooner once few slots run (256 LF2 meshes, FP32: tiles 64 and 128 within 0.3% per full-batch
step, but 99.6 s against 97.0 s for the whole steady solve).  The choice changes only the block partition: per-slot results are
bitwise identical between runs at the same tile, and within the FP64/FP32 tolerances across
tiles (the monitor's block partial sums are the only tile-dependent reduction order).

The second choice is the few-slot launch shape (`Batch.set_launch_shape`): when few slots of a
closed batch are still running, each trial is bound by latency and more threads per cell in the
flux launches shorten it; with many running they are slower (fewer blocks per CU).  The tuner times
trials with k = 32, 16, 8 and 2 running slots at the spread that the arena chose by its size and at
every larger one that the tile admits, and takes the one that wins at and below the largest k (0:
none wins, or the arena's own spread is the largest there is).  256 LF2 meshes, FP32, tile 128, us a
trial at one / two / three threads: 2 running 66.2 / 61.4 / 57.5, 8: 69.3 / 64.5 / 72.3, 16: 82.6 /
77.4 / 114, 32: 101 / 117 / 167, so two threads from 16 slots down (the blocks of ended slots, which
the others wait behind, hold as many threads).  Results are bitwise independent of both choices at a
given tile.

Results are cached per (precision, slot count, total cells rounded to 1%, feature set) for
the life of the process.
"""
from __future__ import annotations

import time

from . import batch as B

TILES = (64, 128, 256)
TIE = 0.01  # relative step-time margin within which the larger tile is kept
_CACHE: dict = {}


def choose(timings: dict) -> int:
    """The tile to use from {tile: seconds per trial}: the largest within TIE of the fastest."""
    fastest = min(timings.values())
    return max(t for t, s in timings.items() if s <= fastest * (1 + TIE))


def _key(meshes, precision, features):
    cells = sum(int(m.n_cells) for m in meshes)
    return (precision, len(meshes), round(cells, -max(0, len(str(cells)) - 2)),
            tuple(getattr(features, k) for k in ("laminar", "sa", "small", "visc_group")))


def time_tile(meshes, params, states, precision: int, tile: int, trials: int = 50, warmup: int = 10) -> float:
    """Seconds per trial of the arena of these meshes at this tile (graph replays, synchronised)."""
    with B.Batch.of_meshes(meshes, params, states, precision=precision, tile=tile) as b:
        b.set_targets(1e30)
        b.run(warmup)
        t0 = time.perf_counter()
        b.run(trials)
        return (time.perf_counter() - t0) / trials


def pick_tile(meshes, params, states, precision: int = 32, tiles=TILES, trials: int = 50,
              warmup: int = 10) -> tuple[int, dict]:
    """(best tile, {tile: seconds per trial}) for this set of meshes."""
    feats = B.union([B.capacity(m)[1] for m in meshes])
    key = _key(meshes, precision, feats)
    if key in _CACHE:
        return _CACHE[key]
    timings = {t: time_tile(meshes, params, states, precision, t, trials, warmup) for t in tiles}
    best = choose(timings)
    _CACHE[key] = (best, timings)
    return best, timings


FEW_PROBES = (32, 16, 8, 2)
MAX_BLOCK = 512  # threads of the largest flux block


def pick_few_shape(meshes, params, states, precision: int, tile: int, probes=FEW_PROBES, seconds: float = 0.25,
                   warmup: int = 10, spreads=(2, 3)) -> tuple[int, int, dict]:
    """(few_slots, few_flux_spread, {k: {threads per cell: us per trial}}) at this tile, for
    `Batch.set_launch_shape(0, few_slots, few_flux_spread)`; (0, 0, {}) when no spread of `spreads` is
    larger than the arena's own."""
    if len(meshes) < 2:
        return 0, 0, {}
    feats = B.union([B.capacity(m)[1] for m in meshes])
    key = ("few", tuple(spreads)) + _key(meshes, precision, feats) + (tile,)
    if key in _CACHE:
        return _CACHE[key]
    n = len(meshes)
    out = {}
    with B.Batch.of_meshes(meshes, params, states, precision=precision, tile=tile) as b:
        own = b.launch_shape()[0]
        tried = [own] + [s for s in spreads if s > own and tile * s <= MAX_BLOCK]
        b.set_targets(1e30)
        b.run(warmup)
        for k in sorted({min(k, n) for k in probes}, reverse=True) if len(tried) > 1 else ():
            out[k] = {}
            for spread in tried:
                b.set_launch_shape(spread, 0, spread)
                b.set_targets([1e30] * k + [0.0] * (n - k))
                b.run(warmup)
                before = sum(s["steps"] + s["rejected"] for s in b.states()[:k])
                t0 = time.perf_counter()
                b.advance("all", budget=seconds)
                elapsed = time.perf_counter() - t0
                trials = (sum(s["steps"] + s["rejected"] for s in b.states()[:k]) - before) / k
                out[k][spread] = round(elapsed / max(trials, 1.0) * 1e6, 1)
    few, spread = choose_few_shape(out)
    _CACHE[key] = (few, spread, out)
    return few, spread, out


def pick_few_slots(meshes, params, states, precision: int, tile: int, probes=FEW_PROBES, seconds: float = 0.25,
                   warmup: int = 10) -> tuple[int, dict]:
    """(few_slots for two flux threads per cell, {k: (us per trial at the arena's own, at two)}) at this
    tile; (0, {}) when the arena runs two or more by itself."""
    few, _, out = pick_few_shape(meshes, params, states, precision, tile, probes, seconds, warmup, (2,))
    return few, {k: (t[min(t)], t[2]) for k, t in out.items()}


def choose_few_shape(probes: dict) -> tuple[int, int]:
    """(few_slots, threads per cell) from {running slots: {threads per cell: us per trial}}, the smallest
    spread of each being the arena's own: the spread that beats it up to the most slots, of two alike the
    faster with the fewest; (0, 0) when none beats it."""
    if not probes:
        return 0, 0
    fewest = probes[min(probes)]
    own = min(fewest)
    found = [(choose_few({k: (t[own], t[s]) for k, t in probes.items()}), -t, s) for s, t in fewest.items() if s != own]
    few, _, spread = max(found, default=(0, 0, 0))
    return (few, spread) if few else (0, 0)


def choose_few(probes: dict) -> int:
    """From {running slots: (us per trial at few, at more threads per cell)}: the largest k such
    that more threads win at k and at every smaller probe (0 if they lose at the smallest)."""
    few = 0
    for k in sorted(probes):
        if probes[k][1] < probes[k][0]:
            few = k
        else:
            break
    return few
