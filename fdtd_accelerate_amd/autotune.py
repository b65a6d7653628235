"""Tile-shape selection for the whole-step kernels.

``slab_planes`` returns the x planes per slab of the slab-ordered step: a table of
measured winners (``tune_slab``, file ``tuned_slab.json``) keyed by
(nx, ny, nz_pitch, npml, ce), else the whole grid as one slab.  (Re-reading a slab's
E and H from the 256 MB last-level cache was measured at only ~10% above HBM
bandwidth on MI355X, less than the per-launch cost of small slabs.)

``fused_tiles`` returns (rows_per_thread T, planes_per_chunk CX) for a grid: a table of
measured winners (filled by ``tune_fused``) keyed by (nx, ny, nz_pitch, npml), else a
rule on the rounds of work-groups over the 256 CUs; ``whole_grid_faster`` says whether a
grid is too small, or fills the sweep's z segments too little, for a sweep at all.
"""
from __future__ import annotations

import json
import math
import os

from ._lib import MAX_CE_TRI

_TABLE_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuned_tiles.json")
_table = None
N_CU = 256


def _load():
    global _table
    if _table is None:
        try:
            with open(_TABLE_PATH) as fh:
                _table = {tuple(json.loads(k)): tuple(v) for k, v in json.load(fh).items()}
        except (OSError, ValueError):
            _table = {}
    return _table


def lds_fits(T, CX, table, ntri=0, extra=0):
    """Whether the sweep's LDS (E and H row exchange 2 x 2 x T x 2 x 256 floats, the k-1
    carry (CX+1)(T+1)2 floats, the 3 x 256 CE table or ``ntri`` CE triples, ``extra``
    more floats, 1.25 KiB of source, probe and patch tables) fits the 160 KiB of one gfx950
    work-group."""
    tab = 4 * ((3 * ntri + 3) // 4) if ntri else (768 if table else 0)
    return 4 * (tab + 2 * 2 * T * 2 * 256 + (CX + 1) * (T + 1) * 2 + extra) + 1280 <= 160 * 1024


def lds_fits_pairs(T, CX, table):
    """Whether the two-step sweep's LDS (T+3 rows: H and E row exchanges of both levels,
    4 x (T+3) x 2 x 256 floats; the k-1 carries of both levels per plane of the chunk,
    (CX+3) x (T+3) x 4 floats; the CE table; ~0.7 KiB of source/probe tables) fits the
    160 KiB of one gfx950 work-group."""
    R = T + 3
    return 4 * ((768 if table else 0) + 4 * R * 512 + 4 * (-(-R // 4)) + (CX + 3) * R * 4) + 1024 <= 160 * 1024


def _halved(nx, ny):
    """T = 9 rows, CX = 64 planes halved while fewer than 1024 blocks."""
    T = min(9, max(1, ny // 8))
    nrb = -(-ny // T)
    cx = min(nx, 64)
    while cx > 8 and nrb * (-(-nx // cx)) < 1024:
        cx = -(-cx // 2)
    return T, max(1, cx)


def tile_cost(T, CX, box):
    """Planes times waves that the work-groups of a CU take one after the other: whole rounds of
    256 blocks of CX planes and one for a block's start, T+1 waves and two for the barrier."""
    rounds = -(-(-(-box[1] // T) * -(-box[0] // CX)) // N_CU)
    return rounds * (CX + 2) * (T + 3)


def heuristic(nx, ny, nzp, npml, halved=False, box=None, table=True):
    """(T, CX): owned rows per block (one halo row each, T+1 waves) and planes per chunk
    (one seed plane each).  One work-group runs per CU, so a sweep takes whole rounds of 256
    blocks: the tile with the least ``tile_cost`` for ``box``, the planes and rows that the
    sweep updates (default: of a grid with CPML on x and y), of the tiles that leave room for
    the largest CE table (``table``: the run has one).  Sweep against T = 9 and CX halved until
    1024 blocks: 256^3 135 / 143 us, 384^3 563 / 651, 512^3 1205-1230 / 1267, 350 x 420 x 500
    641 / 694; within 3% of the best of 126 tiles measured at five grids.  ``halved``: that
    older rule, which a Drude sweep (at most 7 rows, two blocks per CU) and a TFSF sweep (13
    rows, its z-face rows cost more) keep, and tiles of which the caller gives one number."""
    if halved:
        return _halved(nx, ny)
    edge = 2 * (npml + 1) if npml else 0
    bx, by = (max(1, n) for n in (box or (nx - edge, ny - edge)))
    best, cost = None, None
    for T in (13, 11, 9, 8, 7, 6, 5, 4, 3, 2, 1):
        if T > max(1, by // 2):
            continue
        for CX in range(min(bx, 64), min(bx, 8) - 1, -1):
            if not lds_fits(T, CX, True, MAX_CE_TRI if table else 0):
                continue
            c = tile_cost(T, CX, (bx, by))
            if cost is None or c < cost:
                best, cost = (T, CX), c
    return best


def heuristic_pairs(nx, ny, nzp, npml):
    """(T, CX) of the two-step sweep: T = 9 owned rows (12 waves, the kernel's launch
    bound; 9.95 ms per step at 1024^3 against 11.8 for T = 5), CX = 64 planes, halved
    while fewer than 1024 blocks."""
    T, cx = _halved(nx, ny)
    while cx > 1 and not lds_fits_pairs(T, cx, True):
        cx -= 1
    return T, max(1, cx)


def fused_pairs(nx, ny, nzp, npml):
    """Whether the fused engine advances steps in pairs by default on this grid: never
    (at 1024^3 with CPML 12 a pair takes 27.3 ms against 25.1 ms for two single steps on
    MI355X; the two-step sweep halves the bytes but is issue-bound)."""
    return False


def fused_tiles(nx, ny, nzp, npml, pairs=False, halved=False, box=None, table=True):
    if pairs:
        return heuristic_pairs(nx, ny, nzp, npml)
    t = _load().get((nx, ny, nzp, npml))
    return t if t is not None else heuristic(nx, ny, nzp, npml, halved, box, table)


def whole_grid_faster(cells, box, segments, tile, face_cells, ce_bytes, tri, drude, tfsf):
    """Whether a step as two passes over the whole grid is faster than the sweep of the ``box``
    (planes, rows, z cells) in ``segments`` z segments with its two shell passes.  Times in us:
    a cell of the sweep costs 48 B + CE at 8.2 TB/s and the tile's rounds 0.22 us per plane and
    wave of a segment (tile_cost), 4% more with a plane wave and 8% with a Drude box than these
    add to the whole-grid passes; a shell cell 72 B + CE at 2.7 TB/s.  A cell of the whole-grid
    passes (``cells``, the pitch's too) costs 72 B + CE at 5.4 TB/s, up to 8.4 where the fields
    stay in the last-level cache, and 9.4 us per million cells of the CPML faces.  Fitted to
    both forms of 511 runs of 40 to 1024 cells an axis (CE none, float and indices, CPML 0-12
    on all faces or on z with periodic x and y, plane waves and Drude boxes): the form picked
    is within 2% of the faster one in 486 of them and at most 13% off (172x117x170 without
    CPML: 45 us for 40).
    Sweep / whole, CE as indices, CPML 12: 224^3 205 / 184 us, 288^3 382 / 399, 384^3 913 /
    902, 448^3 1303 / 1398, 512^3 1733 / 1986; z CPML and periodic x, y, float CE: 300x300x250
    351 / 400, 384^3 956 / 935, 448^3 1345 / 1472; with a plane wave 384^3 1077 / 948, 512^3
    2018 / 2014, 640^3 3887 / 4013; with a Drude box 384^3 1376 / 997, 512^3 2375 / 2259, 768^3
    7134 / 7199, 1024^3 15326 / 17001."""
    if not box[0] * box[1] * box[2]:  # no interior: the shell passes would take the whole grid
        return True
    sweep = box[0] * box[1] * box[2] * (48 + (2 if tri else ce_bytes)) / 8.2e6 + 0.22 * segments * tile_cost(*tile, box)
    if tfsf:
        sweep *= 1.04
    if drude:
        sweep *= 1.08
    sweep += (cells - box[0] * box[1] * box[2]) * (72 + ce_bytes) / 2.7e6 + 8.0
    rate = 5.4 + 3.0 * math.exp(-cells / 5.5e6)
    whole = cells * (72 + ce_bytes) / (1e6 * rate) + 9.4e-6 * face_cells + 10.0
    return whole < sweep


def tune_fused(sim, candidates=((7, 64), (9, 64), (9, 96), (11, 64), (11, 128), (13, 64), (15, 96)), steps=5, save=True):
    """Time the interior sweep for each (T, CX) on ``sim`` (a YeeSim with engine='fused')
    and record the best.  Runs real steps (the simulation advances by
    len(candidates) * (steps + 1) steps)."""
    from .fused import FusedStepper
    f = sim.fields
    best = None
    results = {}
    for T, CX in candidates:
        if not lds_fits(T, CX, f.ce_mat is not None):
            continue
        st = FusedStepper(sim, rows_per_thread=T, planes_per_chunk=CX)
        st.run(1, None)
        ms = st.run(steps, None, time_kernel=True)
        results[(T, CX)] = ms
        if best is None or ms < results[best]:
            best = (T, CX)
    if best is None:
        raise ValueError(f"no candidate tile fits the 160 KiB of LDS : {tuple(candidates)}")
    key = (f.nx, f.ny, f.nz_pitch, sim.cpml.npml if sim.cpml else 0)
    _load()[key] = best
    if save:
        with open(_TABLE_PATH, "w") as fh:
            json.dump({json.dumps(list(k)): list(v) for k, v in _table.items()}, fh, indent=1)
    return best, results


_SLAB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuned_slab.json")
_slab_table = None


def _load_slab():
    global _slab_table
    if _slab_table is None:
        try:
            with open(_SLAB_PATH) as fh:
                _slab_table = {tuple(json.loads(k)): int(v) for k, v in json.load(fh).items()}
        except (OSError, ValueError):
            _slab_table = {}
    return _slab_table


def slab_heuristic(nx, ny, nzp):
    return nx


def slab_planes(nx, ny, nzp, npml, ce_on):
    t = _load_slab().get((nx, ny, nzp, npml, int(bool(ce_on))))
    return t if t is not None else slab_heuristic(nx, ny, nzp)


def tune_slab(sim, candidates=(1, 2, 3, 4, 6, 8, 12, 16, 32), steps=5, save=True):
    """Time each slab size on ``sim`` (advances the simulation) and record the best."""
    from .fused import SlabStepper
    f = sim.fields
    results = {}
    for S in candidates:
        if S > f.nx:
            continue
        st = SlabStepper(sim, slab_planes=S)
        st.run(1, None)
        results[S] = st.run(steps, None, time_kernel=True)
    if not results:
        raise ValueError(f"no candidate slab depth is at most nx = {f.nx} : {tuple(candidates)}")
    best = min(results, key=results.get)
    key = (f.nx, f.ny, f.nz_pitch, sim.cpml.npml if sim.cpml else 0, int(f.ce_on))
    _load_slab()[key] = best
    if save:
        with open(_SLAB_PATH, "w") as fh:
            json.dump({json.dumps(list(k)): v for k, v in _slab_table.items()}, fh, indent=1)
    return best, results
