"""Chooses the attention kernels for a step.

Every choice computes the same function (causal, optionally windowed, grouped-query attention
over the paged cache); they differ in speed and in which sizes they accept.  In bfloat16 with a
head size the matrix-core module takes (up to 128, values as wide as keys), requests that bring at least TILE_MIN rows go to the
tile kernel (tiles of as many rows as the compiled module says; keys in splits when the tiles are
few and their pasts long) and all other rows (decode tokens, short portions) to the row kernel, or into
the tiles' own launch where those leave compute units idle;
everything else (float32, other head sizes) goes to the plain kernel, whose bits the 32-bit
tile kernel repeats for whole tiles of rows.
"""
from __future__ import annotations

from typing import Optional

import numpy as np
import torch

from . import ops

TILE_MIN = 16       # fewer rows than this are cheaper one by one
F32_TILE_MIN = 16   # ... in 32 bits,
F32_TILE_MIN_WORK, F32_WIDE_TILE_MIN_WORK = 1 << 18, 300_000    # and steps of less than this many (row, head, map) items times the longest context,
                                # the second for tiles of 128 columns, 8 heads of 128 on two in what follows beside 14 of 64 on two.  us plain / in tiles, a prompt of
                                # 80 rows 16 / 24, 13 / 15; of 200 37 / 28, 30 / 16; 64 of 40 rows 68 / 25, 67 / 22; 64 rows behind 500 keys 36 / 46 (289,000 items), 34 / 23, 128
                                # rows 87 / 47, 73 / 23; 64 behind 400 beside 32 prompts of 16 70 / 38, 49 / 27, 16 behind 3,000 beside 16 of 16 387 / 82, 258 / 61; two of 2,000
                                # rows 2,760 / 247, 2,460 / 210.  480 steps drawn around the lines: 0.91 of the plain kernel's speed at worst in tiles beyond
                                # them, 0.59 and a tenth slower with a line at 1 << 17 for tiles of 128 columns; counting each request's own context is no better
F32_MAX_COLUMNS = 1 << 26        # (row, head) columns of whole tiles that a launch holds; larger steps stay with the plain kernel, which goes portion by portion
F32_SPLIT = ((64, 128), (128, 255), (256, 768))    # 32-bit tiles by four workgroups each: up to so many workgroups without that, longer contexts
                                # than this.  us whole / split: 44 workgroups of 64 elements and 200 keys 23 / 16, 112 and 256 keys 23 / 22, 220 and
                                # 1,000 keys 72 / 52; but 104 and 112 keys 15 / 20, 224 and 256 keys 23 / 34; of 128 elements 14 and 200 keys 43 / 28,
                                # 152 and 600 keys 110 / 97, 252 and 2,000 keys 320 / 246, but 112 and 200 keys 45 / 54, 256 and 500 keys 96 / 126
TILE_QT2_MIN_WORKGROUPS = 512   # two workgroups of the tile kernel for each of the 256 compute units
TILE_QT2_MIN_KEYS = 1536        # ... or rows that see this many keys on average, so that reading them from LDS half as often decides
TILE_SPLIT_BELOW = 384          # fewer workgroups than this: the tile kernel splits the keys
TILE_SPLIT_TARGET = 448         # ... aiming at this many workgroups,
TILE_SPLIT_MIN_KEYS = 512       # with at least this many keys to a split
TILE_SPLIT_MIN_LONGEST = 1536   # and only when the longest request has this many keys: writing and merging partial
                                # results costs about 20 us
TILE_SPLIT_FEW = 128            # at most this many workgroups: splits pay from
TILE_SPLIT_FEW_MIN_LONGEST = 1024   # this many keys on, and may be as short as
TILE_SPLIT_FEW_MIN_KEYS = 256       # this while the walk is short
TILE_MAX_SPLITS = 16
TILE_ORDER_MIN_ITEMS = 64       # launches of more workgroups than this get them in tile_order
TILE_GROUPS_MAX = 256       # at most this many workgroups of 64-row tiles, one for each compute unit: two groups of waves to a workgroup,
TILE_GROUPS_KEYS = 1024     # while no workgroup walks more keys than this
TILE_GROUPS_KEYS_BESIDE = 1536      # ... or than this with the step's other rows in the same launch (see choose_groups),
TILE_GROUPS_FEW, TILE_GROUPS_KEYS_FEW = 48, 1152      # of fewer workgroups than these no more than so many keys
ROW_CHUNK = 64      # keys per split of the row kernel: doubled while the launch keeps ROW_MIN_WAVES (ROW_MIN_WAVES_128
ROW_MIN_WAVES_128 = 1000   # for the step from 64 to 128) waves or more: a split costs a fixed start-up, so longer splits
ROW_MIN_WAVES = 1536       # pay when there are waves enough; and until a row has at most ROW_MAX_SPLITS splits.  The merge
ROW_MAX_SPLITS = 512       # launch shares a row of many splits among up to 8 waves, so one request over a long context may
                           # have hundreds (one row over 32,000 keys: 23.6 us in 250 splits against 35.8 in 125 with a
                           # merge of one wave; over 3,100 keys 11.8 us in 49 splits of 64 against 13.7 in 25 of 128).
ROW_WHOLE_MIN_PAIRS = 192   # (row, kv head) pairs from which a workgroup takes a pair's keys whole
ROW_WAVE_SLOTS = 2048       # waves the chip holds at the row kernel's two per SIMD
ROW_WHOLE_SHORT = 256       # keys (of 128 elements: twice as many of 64) up to which it does so whatever the number of pairs ...
ROW_WHOLE_SHORT_PAIRS = 96  # ... and pairs from which it does up to twice as many


DIRECT_MIN_WORK = 1 << 18       # rows x keys seen per row from which the tall tiles of head size 128 win
DIRECT_SPLIT_FEW = 64           # at most this many workgroups: splits from 2,048 keys on,
DIRECT_SPLIT_BELOW = 128        # at most this many: from 3,072 keys on; more workgroups are never split
DIRECT_SPLIT_MIN_KEYS = 512


def _choose_direct(tiled_rows, tiled_keys, n_heads: int, rows_of, total: int, longest: int, seen: float):
    """``choose_tiling`` for head size 128, where the tall tiles are the kernel that loads straight into LDS.
    Measured (28, 16 and 40 query heads, workgroups in ``tile_order``; us with tiles of 64 / of 128 rows, each with
    its best number of splits): 512 rows 20 / 24, 1,024 rows 37 / 30, 2,048 rows 77 / 58, 8,192 rows 865 / 533;
    512 rows after 512 keys 34 / 27, after 3,584 keys 96 / 69 (85 whole), 1,024 after 3,072 141 / 93 (117 in two
    splits), 128 after 3,968 41 / 34 (83 whole), 2,048 after 6,144 436 / 226.  The tall tiles win wherever there
    is work enough, and their keys want cutting only for few workgroups with long walks."""
    n_big = sum(-(-int(n) // rows_of(2)) for n in tiled_rows)
    if total * seen < DIRECT_MIN_WORK or n_big * rows_of(2) > 2 * total:
        return None
    groups = n_big * n_heads
    splits, chunk = 1, 0
    if (groups <= DIRECT_SPLIT_FEW and longest >= 2048) or (groups <= DIRECT_SPLIT_BELOW and longest >= 3072):
        want = min(max(1, (2 * TILE_SPLIT_TARGET + groups) // (2 * groups)), longest // DIRECT_SPLIT_MIN_KEYS, TILE_MAX_SPLITS)
        if want > 1:
            chunk = (-(-longest // want) + 63) // 64 * 64
            splits = -(-longest // chunk)
            if splits <= 1:
                splits, chunk = 1, 0
    return 2, splits, chunk


def choose_tiling(tiled_rows, tiled_keys, n_heads: int, rows_of, tall_direct: bool = False):
    """(tiling: 1 = tiles of 64 rows, 2 = of 128; key splits; keys per split) for a launch of the tile kernel:
    ``tiled_rows`` the row counts of the requests it covers, ``tiled_keys`` how many keys each of them holds after
    the step, ``rows_of(qt)`` a tile's rows, ``tall_direct`` whether the tall tiles are the kernel of head size 128
    (``_choose_direct`` then decides whether to take them).  What follows is measured on the other kernel, whose
    tall tiles are two query tiles per wave.

    Measured at head size 128 (28, 16 and 40 query heads; portions of 256-8,192 rows after pasts of 0-7,680 keys,
    workgroups in ``tile_order``): two query tiles per wave win when they still give two workgroups to each compute
    unit (4,096 rows: 178 us against 236) or when a tile walks many keys on average (2,048 rows after 2,048 keys:
    158 us against 218; 1,024 after 1,024: 74 against 80), as long as the rows fill the taller tiles, and lose
    on a short causal prompt (2,048 rows: 81 us against 75).  About 448 workgroups are the best number to cut the
    keys for (1,024 rows after 7,168 keys: 292 us whole, 199 in two splits, 208 in four), and a cut pays only when
    the walk it shortens is long (512 rows after 512 keys: 34 us whole, 40 in two splits)."""
    total = int(sum(tiled_rows))
    longest = int(max(tiled_keys))
    # keys a row sees, averaged over the launch's rows: a request's rows see from (keys - rows) to keys of them
    seen = sum(int(n) * (int(k) - int(n) / 2.0) for n, k in zip(tiled_rows, tiled_keys)) / max(total, 1)
    n_big = sum(-(-int(n) // rows_of(2)) for n in tiled_rows)
    qt = 1
    if tall_direct:
        direct = _choose_direct(tiled_rows, tiled_keys, n_heads, rows_of, total, longest, seen)
        if direct is not None:
            return direct
    elif n_big * n_heads >= TILE_QT2_MIN_WORKGROUPS:
        qt = 2
    elif seen >= TILE_QT2_MIN_KEYS and n_big * rows_of(2) * 2 <= total * 3:
        qt = 2
    groups = sum(-(-int(n) // rows_of(qt)) for n in tiled_rows) * n_heads
    splits, chunk = 1, 0
    if groups < TILE_SPLIT_BELOW and longest >= (TILE_SPLIT_FEW_MIN_LONGEST if groups <= TILE_SPLIT_FEW else TILE_SPLIT_MIN_LONGEST):
        want = min(max(1, (2 * TILE_SPLIT_TARGET + groups) // (2 * groups)), longest // TILE_SPLIT_MIN_KEYS, TILE_MAX_SPLITS)
        if groups <= TILE_SPLIT_FEW and longest < 2 * TILE_SPLIT_MIN_LONGEST:
            want = max(want, min(4, longest // TILE_SPLIT_FEW_MIN_KEYS))
        if want > 1:
            chunk = (-(-longest // want) + 63) // 64 * 64
            splits = -(-longest // chunk)
            if splits <= 1:
                splits, chunk = 1, 0
    return qt, splits, chunk


def choose_groups(tiled_rows, tiled_keys, n_heads: int, row_keys, pairs: int, window: Optional[int], splits: int = 1, beside_fits: bool = True):
    """(two groups of waves to a workgroup of 64-row tiles, and the step's other rows beside them in the same launch) for a step whose requests bring
    ``tiled_rows`` rows and hold ``tiled_keys`` keys, beside single rows of ``row_keys`` keys in ``pairs`` (row, kv head) pairs; by itself
    ``choose_tiling`` would cut the tiles' keys into ``splits``.

    A launch of at most a workgroup for each compute unit leaves a workgroup of four waves waiting for itself; with eight, of which each four
    take every other key tile, a tile of 128 elements costs 1.25 us instead of 1.65.  us as it
    was / in two groups: 16 heads of 128 on 2, 500 rows 17.9 / 15.0, 300 after 512 keys 26.2 / 21.1, 64 after 700 24.9 / 19.9, 2 prompts of 512 15.5 / 15.5,
    512 after 512 24.7 / 24.8, 512 after 1,500 43.6 / 43.6, 256 after 3,000 32 / 66; 14 heads of 64 on 2, 500 rows 14.0 / 11.4, 512 after 512 20.6 / 18.4,
    1,024 24.4 / 18.6, 512 after 1,500 29.7 / 32.1, 61 (a single tile) 5.7 / 6.2; 336 workgroups of 128 20.5 / 21.5.
    The other rows beside them cost little while they end no later than the tiles, against 10 to 13 us of their own launches: a row's walk takes some
    4.5 us and 11 for 1,000 keys, a tile's 5 and 19.5.  us with launches of their own / beside, 16 heads of 128 on 2: 500 rows and 23 rows of up to 299 keys
    28.7 / 15.6, 20 of up to 992 30.5 / 18.6, 512 after 1,500 and 20 of 981 58 / 44, 128 rows and 6 of 369 17.5 / 9.7, but 4 of 1,900 18.0 / 25.6; more
    workgroups than compute units, 28 heads on 4, 500 rows and 23 of 283 31.9 / 17.6; 2 prompts of 512, 16 heads, and 4 rows of 1,933 25.6 / 31.6.
    Few tiles with long walks are better cut into splits, which many workgroups share, whatever rows are beside them: us in splits and with launches of their own /
    beside, 12 workgroups of 128 and 1,193 keys 25.2 / 28.1, 16 and 1,463 27.2 / 32.9, 28 and 1,518 28.5 / 34.1, 36 and 1,413 31.5 / 33.4, but 12 and 1,142 27.2 / 26.8,
    48 and 1,317 32.0 / 31.7, 80 and 1,500 42.4 / 34.9, 196 and 1,512 44.0 / 36.1."""
    blocks = sum(-(-int(n) // 64) for n in tiled_rows) * n_heads
    walk = int(max(tiled_keys)) if window is None else min(int(max(tiled_keys)), window + 64)
    if blocks > TILE_GROUPS_MAX or walk > (TILE_GROUPS_KEYS_BESIDE if blocks >= TILE_GROUPS_FEW else TILE_GROUPS_KEYS_FEW):
        return False, False
    if pairs and beside_fits and pairs <= TILE_GROUPS_MAX:
        row_walk = int(max(row_keys)) if window is None else min(int(max(row_keys)), window)
        if row_walk * 4 <= walk * 7 + (2800 if blocks + pairs <= TILE_GROUPS_MAX else 0):
            return True, True
    return splits == 1 and 64 < walk <= TILE_GROUPS_KEYS, False


from .device import CUS_PER_XCD, N_XCD      # the launch deals workgroups to the XCDs in turn, and an XCD its share to its compute units in turn


def tile_order(first_pos, last_pos, n_heads: int, window: Optional[int], splits: int, chunk: int, period: int = CUS_PER_XCD) -> np.ndarray:
    """Which work item each workgroup of a tile launch takes: int32 [8 * n], place x * n + i being the i-th workgroup
    of XCD x (-1: none).  ``first_pos`` / ``last_pos``: the positions of every tile's first and last row.

    A work item is (head, tile, split), numbered head * tiles * splits + (tiles - 1 - tile) * splits + split, and
    walks a number of 64-key tiles that is known here.  Workgroups on one compute unit share its time, so a unit
    that is given three long walks finishes long after one with three short ones: a causal prompt of 2,048 rows
    took 100 us in the order longest first, head by head, where the walks of the unit that came first summed to
    96 key tiles and the average was 58.  Here the items stay in head order (an XCD's workgroups read few kv heads,
    which its L2 then holds), are cut into eight runs of equal walks, not equal counts, and go to the workgroups
    of a run in boustrophedon order of their length with a compute unit's turn as the period, so that the i-th,
    (2 * period - 1 - i)-th, (2 * period + i)-th ... longest meet on one unit."""
    first_pos, last_pos = np.asarray(first_pos, np.int64), np.asarray(last_pos, np.int64)
    n_tiles = first_pos.shape[0]
    lo = np.maximum(first_pos - window + 1, 0) if window else np.zeros(n_tiles, np.int64)
    if splits > 1:
        s = np.arange(splits, dtype=np.int64)[None, :]
        lo_ts = np.maximum(lo[:, None], s * chunk)
        hi_ts = np.minimum(last_pos[:, None], (s + 1) * chunk - 1)
    else:
        lo_ts, hi_ts = lo[:, None], last_pos[:, None]
    walk = np.where(hi_ts >= lo_ts // 64 * 64, hi_ts // 64 - lo_ts // 64 + 1, 0)        # [tiles, splits] key tiles walked
    cost = (walk[::-1] + 1).reshape(-1)                                                # + 1: a workgroup's start and end
    cost = np.tile(cost, n_heads)                                                      # [items] in the kernel's numbering
    n_items = cost.shape[0]
    cum = np.cumsum(cost)
    run = np.minimum((cum - cost) * N_XCD // cum[-1], N_XCD - 1)                       # the run an item's start falls into
    counts = np.bincount(run, minlength=N_XCD)
    per_xcd = int(counts.max())
    order = np.full((N_XCD, per_xcd), -1, np.int32)
    start = 0
    for x in range(N_XCD):
        n = int(counts[x])
        if n == 0:
            continue
        items = np.arange(start, start + n)
        by_len = items[np.argsort(-cost[start:start + n], kind="stable")]
        rank = np.arange(n)
        row, col = rank // period, rank % period
        width = np.minimum(period, n - row * period)
        place = row * period + np.where(row % 2 == 0, col, width - 1 - col)
        order[x, place] = by_len
        start += n
    return order.reshape(-1)


def _work_lists(ctx, ctx_kv_heads, tile_rows, n_heads, tile_splits=1, tile_chunk=0, window=None, row_waves=8, head_dim=128):
    """What the kernels need beyond the step's own arrays, computed once per step (and per number of
    kv heads, which decides how many waves a launch has)."""
    q_len, q_start, kv_len = ctx.h_q_len, ctx.h_q_start, ctx.h_kv_len
    tiled = q_len >= TILE_MIN
    tile_req, tile_q0 = [], []
    for r in np.nonzero(tiled)[0]:
        for q0 in range(0, int(q_len[r]), tile_rows):
            tile_req.append(r); tile_q0.append(q0)
    row_mask = ~tiled[ctx.h_row_req] if ctx.n_tokens else np.zeros(0, bool)
    rows = np.nonzero(row_mask)[0].astype(np.int32)
    out = {"n_tiles": len(tile_req), "n_rows": int(rows.size), "rows": None, "chunk": ROW_CHUNK, "max_splits": 1, "waves": 0,
           "tile_splits": 1, "tile_chunk": 0, "tile_row_list": None, "tile_order": None}
    lists = {}                       # everything that goes to the device, in one copy (each copy is a wait for the host)
    if tile_req:
        tile_req, tile_q0 = np.asarray(tile_req, np.int32), np.asarray(tile_q0, np.int32)
        lists["tile_req"], lists["tile_q0"] = tile_req, tile_q0
        if len(tile_req) * n_heads * tile_splits > TILE_ORDER_MIN_ITEMS:
            first = (kv_len[tile_req] - q_len[tile_req] + tile_q0).astype(np.int64)
            last = np.minimum(first + tile_rows, kv_len[tile_req]) - 1
            lists["tile_order"] = tile_order(first, last, n_heads, window, tile_splits, tile_chunk)
        # Few tiles with many keys each (portions of prompts with a long past) leave most of the chip idle
        # and each workgroup walking its keys alone: the keys are cut into splits that run side by side.
        if tile_splits > 1:
            out["tile_splits"], out["tile_chunk"] = tile_splits, tile_chunk
            lists["tile_row_list"] = np.nonzero(~row_mask)[0].astype(np.int32)
    if rows.size and rows.size != ctx.n_tokens:
        lists["rows"] = rows
    if lists:
        sizes = [(k, v.shape[0]) for k, v in lists.items()]
        packed = ctx.upload(np.concatenate([np.concatenate([v, np.zeros(-v.shape[0] % 4, np.int32)]) for v in lists.values()]))
        at = 0
        for k, n in sizes:
            out[k] = packed[at:at + n]
            at += n + -n % 4          # every list starts at a multiple of 16 bytes
    if rows.size:
        out["chunk"], out["waves"], out["max_splits"] = row_launch_shape(int(rows.size), ctx_kv_heads, ctx.kv_bound, row_waves, head_dim,
                                                                               n_heads // ctx_kv_heads)
    return out


def whole_row_keys(pairs: int, head_dim: int, heads_per_kv: int = 16) -> int:
    """Keys up to which rows are taken whole by a launch of ``pairs`` (row, kv head) pairs that would split longer ones.  A workgroup
    goes through a pair's keys once for every 16 of its query heads (32 heads on one of 128, 8 rows, us whole / in splits at 128 and 256
    keys 11.7, 16.2 / 13.8, 13.7; 64 heads on one at 64 and 128 keys 16.2, 20.5 / 19.5, 20.0)."""
    short = ROW_WHOLE_SHORT if head_dim > 64 and pairs < ROW_WHOLE_SHORT_PAIRS else 2 * ROW_WHOLE_SHORT
    return short // max(1, -(-heads_per_kv // 16))


def decode_kinds(caches):
    """What ``table_tokens`` has to know of a model's ``caches`` (LayerCaches, each with its number of query heads): the distinct (kv
    heads, head size, query heads per kv head) of those that the row kernel reads, head size 0 for attention through a latent."""
    kinds = set()
    for c, n_heads in caches:
        n_kv, page_size, d = c.k.shape[1:]
        if ops.mfma_attention_supported(c.k.dtype, d, page_size) and c.v.shape[2] == d:
            kinds.add((n_kv, d, n_heads // n_kv))
        elif ops.wide_attention_supported(c.k.dtype, n_kv, d, c.v.shape[2], page_size):
            kinds.add((1, 0, 0))
    return tuple(sorted(kinds))


def table_tokens(longest: int, n_rows: int, kinds, most: int, page_size: int) -> int:
    """Tokens that the block tables of a captured step of ``n_rows`` single tokens have room for where its requests hold at most
    ``longest``: ``most``, or fewer where a launch over one of the caches (``decode_kinds``) then has a shape that its shorter bound
    allows.  Rows that a workgroup takes whole: us a step at 130 to 255 / 256 to 511 tokens with tables of 1,024 tokens and of as few
    as that allows, 0.5B shape 1 request 873, 876 : 795, 840, 1.5B 64 requests 2,640, 2,670 : 2,285, 2,400, 7B 8 requests 3,180 : 3,030;
    fewer splits of a latent's rows, 8 requests 1,345 : 1,305.  Such a bound is a layout more that is captured once for a batch size, at
    3.5 to 12 ms, which these steps pay back within 30 to 130 tokens of all requests together; a bound that brings no other
    launch gets none (512 tokens where only 256 are taken whole: 1 % at best)."""
    bounds = [most]
    for n_kv, d, per_kv in kinds:
        if d == 0:
            bounds.append(ROW_WHOLE_SHORT)
        elif n_rows * n_kv < ROW_WHOLE_MIN_PAIRS:
            bounds.append(whole_row_keys(n_rows * n_kv, d, per_kv))
    return min(b for b in bounds if (b >= longest and b % page_size == 0) or b == most)


def row_launch_shape(n_rows: int, n_kv_heads: int, max_kv: int, max_waves: int = 8, head_dim: int = 128, heads_per_kv: int = 16):
    """(keys per split, waves per workgroup, splits) of a launch of the row kernel over ``n_rows`` rows whose requests
    hold at most ``max_kv`` keys (the bound of their block tables, not the lengths themselves: see
    StepContext.kv_bound).  ``max_waves``: what fits the kernel's LDS (``ops.row_waves_fit``).

    With (row, kv head) pairs enough to fill the chip by themselves, one workgroup takes a pair whole (keys per split
    0): its waves, as many as give the chip about one round of 2,048, share the row's keys evenly, meet in LDS and
    write the output, with no partial results in memory and no second launch.  Measured at 28 : 4 heads of 128 over
    3,100 keys, us whole / in splits with the merge launch: 48 rows 61 / 69, 64 rows 68 / 88, 96 rows 116 / 133, 128
    rows 129 / 178, 256 rows 250 / 361; 64 rows over 16,384 keys 328 / 358; 32 rows 57 / 48, so fewer pairs than 192
    keep the splits: their keys have to be spread over more compute units than there are pairs, which only a second
    launch can merge (one wave per split of ``chunk`` keys, waves per workgroup 0).

    Rows of few keys take a workgroup each too: a compute unit reads 256 keys in less time than the second launch takes.
    us whole / in splits at 64 and 300 keys: 14 : 2 heads of 64, 1 row 4.5, 6.3 / 8.1; 16 : 2 heads of 128, 8 rows 5.6,
    10.2 / 11.2, 64 rows 6.1, 11.3 / 14.4, 19.9; 16 heads on one of 128, 8 rows (four waves fit) 5.6, 11.5 / 10.7."""
    pairs = n_rows * n_kv_heads
    if pairs >= ROW_WHOLE_MIN_PAIRS or max_kv <= whole_row_keys(pairs, head_dim, heads_per_kv):
        waves = 1
        while waves * 2 <= min(max_waves, ROW_WAVE_SLOTS // pairs):
            waves *= 2
        return 0, waves, 1
    chunk = ROW_CHUNK
    while (-(-max_kv // chunk) > ROW_MAX_SPLITS
           or pairs * -(-max_kv // (2 * chunk)) >= (ROW_MIN_WAVES_128 if chunk == ROW_CHUNK else ROW_MIN_WAVES)):
        chunk *= 2
    return chunk, 0, -(-max_kv // chunk)


def _f32_tiles(ctx, n_heads: int, n_kv: int, maps: int, cols: int):
    """(tiles, rows that are not in one, whether parts go by workgroups of their own) of a step for ``ops.attention_f32``; the first None:
    the step has no tiles, the second None: no further rows."""
    tiled = ctx.h_q_len >= F32_TILE_MIN
    least = F32_WIDE_TILE_MIN_WORK if cols > 64 else F32_TILE_MIN_WORK
    if not tiled.any() or int(ctx.h_q_len[tiled].sum()) * n_heads * maps * int(ctx.h_kv_len[tiled].max()) < least:
        return None, None, False
    group = n_heads // n_kv
    if int((-(-ctx.h_q_len[tiled].astype(np.int64) * group // cols)).sum()) * n_kv * cols >= F32_MAX_COLUMNS:
        return None, None, False
    tiles = [(r, c) for r in np.nonzero(tiled)[0] for c in range(0, int(ctx.h_q_len[r]) * group, cols)]
    past = ctx.h_kv_len - ctx.h_q_len
    tiles.sort(key=lambda t: -int(past[t[0]]) - t[1] // group)                  # the longest walks first
    rows = np.nonzero(~tiled[ctx.h_row_req])[0].astype(np.int32)
    packed = ctx.upload(np.concatenate([np.asarray(tiles, np.int32).ravel(), rows]))       # (each copy is a call of its own)
    groups, longest = len(tiles) * n_kv * maps, int(ctx.h_kv_len[tiled].max())
    split = any(groups <= g and longest > n for g, n in F32_SPLIT)
    return packed[:2 * len(tiles)].view(-1, 2), packed[2 * len(tiles):] if rows.size else None, split


def plain_attention(q: torch.Tensor, cache, ctx, window: Optional[int], scale: float, keep_first: int = 0, sink: Optional[float] = None,
                    gate: Optional[torch.Tensor] = None, sinks: Optional[torch.Tensor] = None, block: Optional[int] = None,
                    differential=None) -> torch.Tensor:
    """The plain kernel, and in 32 bits, where there is a kernel for the sizes, the matrix cores for requests of at least F32_TILE_MIN
    rows in steps with work enough (the same bits by either)."""
    table = ctx.block_table(cache.group)
    T, nH, d = q.shape
    n_kv, page_size = cache.k.shape[1:3]
    dv = cache.v.shape[2]
    maps = 2 if differential is not None else 1
    cols = ops.attention_f32_cols(q.dtype, d // maps, dv, maps, page_size)
    tiles, rows, split = (ctx.derived(("attention_f32_tiles", nH, n_kv, maps, cols), lambda: _f32_tiles(ctx, nH, n_kv, maps, cols)) if cols
                          else (None, None, False))
    if tiles is None:
        return ops.attention_plain(q, cache.k, cache.v, ctx.row_req, ctx.positions, table, window, scale, keep_first, sink, gate,
                                   sinks=sinks, chunk=block, differential=differential)
    out = ops.empty((T, nH * dv), q.dtype, q)
    ops.attention_f32(q, cache.k, cache.v, out, tiles, ctx.q_start, ctx.q_len, ctx.kv_len, table, window, scale, keep_first, sink, gate,
                      sinks, block, differential, split)
    if rows is not None:
        ops.attention_plain(q, cache.k, cache.v, ctx.row_req, ctx.positions, table, window, scale, keep_first, sink, gate,
                            sinks=sinks, chunk=block, differential=differential, rows=rows, out=out)
    return out


def paged_attention(q: torch.Tensor, cache, ctx, window: Optional[int], scale: float, keep_first: int = 0,
                    sink: Optional[float] = None, gate: Optional[torch.Tensor] = None,
                    sinks: Optional[torch.Tensor] = None, block: Optional[int] = None, keep_splits: bool = False):
    """q [T, nH, d] of this step's rows against ``cache`` (a LayerCache); returns [T, nH*d], with ``keep_splits`` also ``SplitRows`` (where
    one launch has all rows in splits).  ``keep_first``: the first
    positions a windowed query sees beside its window; ``sink``: the score of a key without value in the softmax's
    denominator (None: none), ``sinks`` float32 [nH]: such a score for every head; ``gate`` float32
    [T, nH]: a factor on every head's output; ``block``: a row sees only the keys of its own block of that many positions,
    counted from the sequence's start."""
    T, nH, d = q.shape
    table = ctx.block_table(cache.group)
    keep_first = int(keep_first or 0) if window else 0
    if keep_first and ctx.derived(("attention_window_whole", window), lambda: ctx.h_q_len.max() >= TILE_MIN and ctx.h_kv_len.max() <= window):
        # prompts that the window holds whole see their first keys anyway, and without them the kernel that loads straight into LDS
        # takes them (2,048 rows of 16 heads of 128 82 us, then 51; steps of single rows are captured for later lengths, too)
        keep_first = 0
    other = keep_first > 0 or sink is not None or gate is not None or bool(block)      # (a sink score per head some kernels do take)
    extras = other or sinks is not None
    if not ops.mfma_attention_supported(q.dtype, d, cache.page_size) or cache.v.shape[2] != d:
        # values of another width than the keys, or heads wider than a wave's registers hold: one shared kv head (attention
        # through a latent) has a matrix-core kernel of its own, everything else (32-bit, odd sizes) the plain kernel
        if not other and ops.wide_attention_supported(q.dtype, cache.k.shape[1], d, cache.v.shape[2], cache.page_size):
            chunk, splits = ops.wide_launch_shape(T, nH, ctx.kv_bound)
            return ops.attention_wide(q, cache.k, cache.v, ctx.row_req, ctx.positions, table, window, scale, chunk, splits, sinks)
        return plain_attention(q, cache, ctx, window, scale, keep_first, sink, gate, sinks, block)
    n_kv = cache.k.shape[1]

    def plan():
        # Two query tiles per wave (128 rows per workgroup) read every key and value from LDS half as often.
        tiled = ctx.h_q_len >= TILE_MIN
        qt, splits, chunk = 1, 1, 0
        two = beside = False
        if tiled.any():
            # (Python's numbers: a step that is run launch by launch waits for this, and numpy's take three times as long one by one)
            rows, keys = ctx.h_q_len[tiled].tolist(), ctx.h_kv_len[tiled].tolist()
            qt, splits, chunk = choose_tiling(rows, keys, nH, lambda t: ops.attention_tile_rows(d, t),
                                              tall_direct=d == ops.DIRECT_TILE_HEAD_DIM and not keep_first and not block)
            others = [(n, k) for n, k in zip(ctx.h_q_len.tolist(), ctx.h_kv_len.tolist()) if 0 < n < TILE_MIN] if len(rows) < tiled.size else []
            two, beside = choose_groups(rows, keys, nH, [k for _, k in others], sum(n for n, _ in others) * n_kv, window, splits, not keep_first)
            if two:
                qt, splits, chunk = 1, 1, 0
        tile_rows = ops.attention_tile_rows(d, qt)
        return qt, 2 if two else 1, beside, ctx.derived(("attention_work_lists", n_kv, tile_rows, nH, splits, chunk, window, d),
                               lambda: _work_lists(ctx, n_kv, tile_rows, nH, splits, chunk, window, ops.row_waves_fit(nH, n_kv, d, ops.ROW_MAX_WAVES), d))

    # (once a step for all layers of a kind)
    qt, groups, beside, w = ctx.derived(("attention_plan", n_kv, nH, d, window, keep_first, block), plan)
    left = keep_splits and w["waves"] == 0 and w["n_rows"] == T > 0 and w["max_splits"] <= ops.SPLITS_READ_MAX and sink is None and gate is None
    out = None if left else ops.empty((T, nH * d), q.dtype, q)
    more = dict(keep_first=keep_first, sink=sink, gate=gate, sinks=sinks, block=block) if extras else {}
    if w["n_tiles"]:
        ops.attention_tiles(q, cache.k, cache.v, out, w["tile_req"], w["tile_q0"], ctx.q_start, ctx.q_len, ctx.kv_len,
                            table, window, scale, qt, w["tile_chunk"], w["tile_splits"], w["tile_row_list"], ctx.row_req,
                            ctx.positions, w["tile_order"], groups=groups, beside=w["rows"] if beside else None, **more)
    if w["n_rows"] and not beside:
        splits = ops.attention_rows(q, cache.k, cache.v, out, w["rows"], w["n_rows"], ctx.row_req, ctx.positions, table,
                                    window, scale, w["chunk"], w["max_splits"], w["waves"], ctx.n_tokens == ctx.n_requests, **more)
    return splits if left else out
