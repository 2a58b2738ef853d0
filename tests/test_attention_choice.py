"""How the tile attention kernel's launch is chosen (no GPU needed): the choices that were measured, and what every
choice must satisfy for the kernel to be right."""
import random
import types

import numpy as np
import torch

from inferflux_amd.kernels.attention import F32_TILE_MIN, TILE_MAX_SPLITS, _f32_tiles, choose_groups, choose_tiling, tile_order

ROWS_OF = lambda qt: 64 * qt          # head size 128


def test_head_size_128_gets_the_choices_that_were_fastest():
    """Tiles of 64 rows / of 128 rows (the kernel that loads straight into LDS), in us, each with its best splits."""
    cases = [  # rows of the portion, keys it sees, query heads -> (tiling, key splits)
        ([512], 512, 28, (1, 1)),        # 20 / 24
        ([1024], 1024, 28, (2, 1)),      # 37 / 30
        ([2048], 2048, 28, (2, 1)),      # 77 / 58
        ([8192], 8192, 28, (2, 1)),      # 865 / 533
        ([512], 1024, 28, (2, 1)),       # 34 / 27
        ([512], 2048, 28, (2, 1)),       # 62 / 47 (55 in four splits)
        ([512], 2048, 16, (2, 4)),       # 47 / 41 in four splits (47 whole)
        ([512], 4096, 28, (2, 4)),       # 96 / 69 (85 whole)
        ([256], 4096, 28, (2, 8)),       # 59 / 45 (84 whole)
        ([1024], 4096, 28, (2, 1)),      # 141 / 93 (117 in two splits)
        ([1024], 8192, 28, (2, 1)),      # 258 / 176 (174 in four splits)
        ([512], 8192, 28, (2, 4)),       # 151 / 99 (164 whole)
        ([128], 4096, 28, (2, 8)),       # 41 / 34 (83 whole)
        ([128], 8192, 28, (2, 16)),      # 56 / 40
        ([2048], 8192, 28, (2, 1)),      # 436 / 226
        ([2048], 4096, 16, (2, 1)),      # 131 / 93
        ([2048], 8192, 40, (2, 1)),      # 586 / 372
        ([130], 130, 28, (1, 1)),
        ([70] * 16, 70, 28, (1, 1)),     # sixteen short prompts: tall tiles would be half empty
    ]
    for rows, longest, heads, want in cases:
        qt, splits, chunk = choose_tiling(rows, [longest] * len(rows), heads, ROWS_OF, tall_direct=True)
        assert (qt, splits) == want, (rows, longest, heads, qt, splits, chunk)
    qt, splits, _ = choose_tiling([64], [4096], 28, ROWS_OF, tall_direct=True)        # a half-empty tall tile: 26 us, this 30
    assert qt == 1 and splits >= 8


def test_other_head_sizes_get_the_choices_measured_with_two_query_tiles_per_wave():
    cases = [  # rows of the portion, keys it sees, query heads -> (query tiles per wave, key splits)
        ([512], 1024, 28, (1, 1)),      # 34 us whole against 40 in two splits
        ([512], 1024, 16, (1, 4)),      # half as many workgroups: 29 us in four splits against 33
        ([512], 2048, 28, (2, 4)),
        ([256], 4096, 28, (2, 8)),
        ([1024], 4096, 28, (2, 2)),
        ([1024], 8192, 28, (2, 2)),
        ([512], 8192, 28, (2, 4)),
        ([2048], 2048, 28, (1, 1)),     # a short causal prompt: 75 us against 81 with two tiles per wave
        ([2048], 2048, 16, (1, 1)),
        ([4096], 4096, 28, (2, 1)),
        ([2048], 4096, 28, (2, 1)),     # 158 us against 218 with one tile per wave
        ([2048], 8192, 28, (2, 1)),
        ([8192], 8192, 28, (2, 1)),
        ([2048], 2048, 40, (2, 1)),
        ([130], 130, 28, (1, 1)),
        ([100] * 16, 100, 28, (1, 1)),
    ]
    for rows, longest, heads, want in cases:
        qt, splits, chunk = choose_tiling(rows, [longest] * len(rows), heads, ROWS_OF)
        assert (qt, splits) == want, (rows, longest, heads, qt, splits, chunk)


def test_a_short_portion_does_not_take_half_empty_tall_tiles():
    qt, splits, chunk = choose_tiling([64], [8256], 28, ROWS_OF)
    assert qt == 1 and splits > 8


def test_every_choice_covers_its_keys_in_splits_the_kernel_takes():
    rng = random.Random(5)
    for _ in range(3000):
        rows = [rng.randint(16, rng.choice([40, 300, 3000])) for _ in range(rng.randint(1, 6))]
        longest = max(rows) + rng.choice([0, rng.randint(0, 500), rng.randint(0, 40000)])
        heads = rng.choice([1, 2, 5, 16, 28, 40, 64])
        qt, splits, chunk = choose_tiling(rows, [r + rng.randint(0, longest - r) for r in rows[:-1]] + [longest], heads, ROWS_OF,
                                          tall_direct=rng.random() < 0.5)
        assert qt in (1, 2) and 1 <= splits <= TILE_MAX_SPLITS
        if splits > 1:
            assert chunk % 64 == 0 and splits * chunk >= longest > (splits - 1) * chunk
        else:
            assert chunk == 0


def _walks(first, last, window, splits, chunk):
    """Key tiles each (tile, split) walks, written out from the kernel's loop bounds."""
    out = []
    for f, l in zip(first, last):
        row = []
        for s in range(splits):
            lo = max(f - window + 1, 0) if window else 0
            hi = l
            if splits > 1:
                lo, hi = max(lo, s * chunk), min(hi, (s + 1) * chunk - 1)
            j0, n = lo // 64 * 64, 0
            while j0 <= hi:
                n, j0 = n + 1, j0 + 64
            row.append(n)
        out.append(row)
    return out


def test_the_order_names_every_work_item_once_and_balances_the_units():
    rng = random.Random(9)
    for trial in range(200):
        n_tiles, heads = rng.randint(1, 40), rng.choice([1, 4, 16, 28])
        rows = rng.choice([64, 128])
        start = rng.randint(0, 3000)
        first = [start + rows * t for t in range(n_tiles)]
        last = [f + rng.randint(1, rows) - 1 for f in first]
        window = rng.choice([None, None, 100, 1000])
        splits = rng.choice([1, 1, 2, 5])
        chunk = -(-(last[-1] + 1) // splits + 63) // 64 * 64 if splits > 1 else 0
        period = rng.choice([2, 3, 32])
        order = tile_order(first, last, heads, window, splits, chunk, period)
        n_items = n_tiles * heads * splits
        assert order.dtype == np.int32 and order.shape[0] % 8 == 0 and order.shape[0] // 8 <= n_items
        assert sorted(order[order >= 0].tolist()) == list(range(n_items))
        assert set(order[order < 0].tolist()) <= {-1}
    # a causal prompt of 2,048 rows in tiles of 64, 28 heads: the compute units' first three workgroups (unit = place
    # modulo 32 within an XCD) walk 50-61 key tiles together on every unit, where longest first head by head gave 3 to 96
    first = [64 * t for t in range(32)]
    last = [f + 63 for f in first]
    order = tile_order(first, last, 28, None, 1, 0).reshape(8, -1)
    walks = _walks(first, last, None, 1, 0)
    sums = []
    for x in range(8):
        unit = [0] * 32
        for i, w in enumerate(order[x][:96]):
            if w >= 0:
                unit[i % 32] += walks[31 - w % 32][0]
        sums += unit
        # an XCD's workgroups read the keys of few kv heads (7 query heads each)
        assert len({int(w) // 32 // 7 for w in order[x] if w >= 0}) <= 2
    assert min(sums) >= 48 and max(sums) <= 62, (min(sums), max(sums))


def test_library_products_are_cut_only_where_slices_fill_the_chip_and_stay_long():
    from inferflux_amd.kernels.ops import library_k_slices as f
    assert [f(M, 3584, 18944) for M in (129, 512, 1024, 2048, 4096)] == [8, 8, 4, 2, 1]     # down of the 7B shape
    assert all(f(M, 3584, 3584) == 1 and f(M, 4608, 3584) == 1 for M in (129, 512, 2048))  # o, q/k/v: K too short to cut
    assert f(512, 37888, 3584) == 1 and f(512, 152064, 3584) == 1                           # tall weights fill the chip as they are
    assert f(512, 2048, 11008) == 4 and f(512, 8192, 29568) == 4                            # down of the 3B and 72B shapes
    assert f(512, 3584, 18944 + 8) == 1                                                     # slices must be multiples of 8 k-values
    for M in (130, 777, 3000):
        for N in (64, 1000, 5120):
            for K in (2048, 4096, 10000, 65536):
                S = f(M, N, K)
                assert S in (1, 2, 4, 8) and K % S == 0 and (S == 1 or (K // S >= 2048 and (K // S) % 8 == 0))


def test_rows_of_few_keys_are_taken_whole():
    """Whatever the number of pairs: up to 256 keys of heads wider than 64 elements, up to 512 of heads of 64 and from 96 pairs on."""
    from inferflux_amd.kernels.attention import row_launch_shape
    whole = lambda *a: row_launch_shape(*a)[1] > 0
    for rows, kv_heads in ((1, 1), (1, 2), (24, 2), (95, 1)):
        assert whole(rows, kv_heads, 256, 8, 128) and not whole(rows, kv_heads, 257, 8, 128)
        assert whole(rows, kv_heads, 512, 8, 64) and not whole(rows, kv_heads, 513, 8, 64)
    for rows, kv_heads in ((96, 1), (48, 2), (191, 1)):
        for d in (64, 128):
            assert whole(rows, kv_heads, 512, 8, d) and not whole(rows, kv_heads, 513, 8, d)
    assert whole(192, 1, 513, 8, 128) and whole(96, 2, 100000, 8, 64)
    assert whole(8, 1, 256, 4, 128, 16) and whole(8, 1, 128, 4, 128, 17) and not whole(8, 1, 129, 4, 128, 32)      # 16 query heads at a time
    assert whole(8, 1, 64, 4, 128, 64) and not whole(8, 1, 65, 4, 128, 64) and whole(8, 1, 256, 8, 64, 32) and not whole(8, 1, 257, 8, 64, 32)


def test_captured_steps_have_short_tables_where_that_changes_a_launch():
    from inferflux_amd.cache.storage import LayerCache
    from inferflux_amd.kernels.attention import decode_kinds, row_launch_shape, table_tokens
    cache = lambda n_heads, n_kv, d, dv, page=16, dtype=torch.bfloat16: (LayerCache(torch.empty(1, n_kv, page, d, dtype=dtype),
                                                                                  torch.empty(1, n_kv, dv, page, dtype=dtype), 0, page), n_heads)
    few, small, latent, shared = cache(28, 4, 128, 128), cache(14, 2, 64, 64), cache(16, 1, 576, 512), cache(32, 1, 128, 128)
    assert decode_kinds([few, few, latent, small]) == ((1, 0, 0), (2, 64, 7), (4, 128, 7))
    assert decode_kinds([cache(4, 2, 64, 64, dtype=torch.float32), cache(4, 2, 80, 96)]) == ()
    bounds = lambda caches, rows, most=1024, page=16: [table_tokens(n, rows, decode_kinds(caches), most, page)
                                                        for n in (1, 128, 129, 256, 257, 512, 513, 1024, 1025)]
    assert bounds([few], 8) == [256] * 4 + [1024] * 5                     # 32 pairs
    assert bounds([few], 32) == [512] * 6 + [1024] * 3                    # 128 pairs
    assert bounds([few], 48) == [1024] * 9                                # 192 pairs: whole at any length
    assert bounds([small], 1) == [512] * 6 + [1024] * 3
    assert bounds([latent], 64) == [256] * 4 + [1024] * 5
    assert bounds([shared], 8) == [128] * 2 + [1024] * 7                  # (two groups of 16 query heads to a kv head)
    assert bounds([few, small], 1) == [256] * 4 + [512] * 2 + [1024] * 3  # layers that differ: two more
    assert bounds([], 1) == [1024] * 9                                    # (the plain kernel's launches do not depend on it)
    assert bounds([few], 1, most=32) == [32] * 9
    assert bounds([few], 1, most=64 * 512, page=512) == [64 * 512] * 9    # (a page holds more)
    for rows in (1, 2, 8, 16, 24, 32, 48, 64):                            # no layout whose launch is that of the wide one
        for heads, n_kv, d in ((1, 1, 128), (4, 2, 64), (14, 2, 128), (20, 4, 128), (64, 8, 128), (40, 1, 64)):
            for n in (1, 100, 256, 300, 512, 600):
                t = table_tokens(n, rows, decode_kinds([cache(heads, n_kv, d, d)]), 1024, 16)
                shape = lambda bound: row_launch_shape(rows, n_kv, bound, 8, d, heads // n_kv)[1] > 0
                assert t == 1024 or (n <= t and shape(t) and not shape(1024))


def test_row_launch_shape():
    """Launches with (row, kv head) pairs enough to fill the chip take a pair whole in one workgroup, with about one
    round of 2,048 waves; fewer pairs are cut into splits that reach past the longest request."""
    from inferflux_amd.kernels.attention import ROW_MAX_SPLITS, row_launch_shape
    assert row_launch_shape(64, 4, 4096) == (0, 8, 1)
    assert row_launch_shape(48, 4, 4096) == (0, 8, 1)
    assert row_launch_shape(96, 4, 4096) == (0, 4, 1)
    assert row_launch_shape(128, 4, 4096) == (0, 4, 1)
    assert row_launch_shape(256, 4, 4096) == (0, 2, 1)
    assert row_launch_shape(600, 4, 4096) == (0, 1, 1)
    assert row_launch_shape(64, 4, 4096, max_waves=4) == (0, 4, 1)      # what the kernel's LDS allows at these head counts
    assert row_launch_shape(64, 2, 4096)[1] == 0                        # 128 pairs: splits
    assert row_launch_shape(1, 4, 4096) == (64, 0, 64) and row_launch_shape(1, 4, 32768) == (128, 0, 256)   # one request: many short splits
    assert row_launch_shape(16, 4, 4096) == (128, 0, 32) and row_launch_shape(32, 4, 4096) == (256, 0, 16)
    for rows, kv_heads, bound in [(1, 4, 4096), (8, 4, 4096), (32, 4, 4096), (1, 1, 131072), (8, 8, 32768), (47, 4, 1024)]:
        chunk, waves, splits = row_launch_shape(rows, kv_heads, bound)
        assert waves == 0 and chunk % 32 == 0 and chunk >= 64
        assert splits * chunk >= bound > (splits - 1) * chunk and splits <= ROW_MAX_SPLITS


def _f32_step(rows, past):
    """What ``_f32_tiles`` reads of a step whose requests bring ``rows`` behind ``past`` keys."""
    q_len = np.asarray(rows, np.int32)
    return types.SimpleNamespace(h_q_len=q_len, h_kv_len=q_len + np.asarray(past, np.int32), h_row_req=np.repeat(np.arange(len(rows)), rows), upload=torch.from_numpy)


def test_prompts_in_32_bits_take_tiles_where_those_are_faster():
    """The steps that were measured on either side (us plain / in tiles), heads of 128 elements in tiles of 128 columns and of 64 in tiles of 64."""
    for rows, past, wide, narrow in [  # 8 heads of 128 on two, 14 of 64 on two
        ([80], [0], False, False),                               # 16 / 24, 13 / 15
        ([200], [0], True, True),                                # 37 / 28, 30 / 16
        ([40] * 64, [0] * 64, True, True),                       # 68 / 25, 67 / 22
        ([64], [500], False, True),                              # 36 / 46, 34 / 23
        ([128], [500], True, True),                              # 87 / 47, 73 / 23
        ([64] + [16] * 32, [400] + [0] * 32, True, True),        # 70 / 38, 49 / 27
        ([16] * 17, [3000] + [0] * 16, True, True),              # 387 / 82, 258 / 61
        ([2000] * 2, [0] * 2, True, True),                       # 2,760 / 247, 2,460 / 210
        ([15] * 500, [2000] * 500, False, False),                # (fewer rows a request than a tile is worth)
    ]:
        step = _f32_step(rows, past)
        assert (_f32_tiles(step, 8, 2, 1, 128)[0] is not None) == wide, (rows, past)
        assert (_f32_tiles(step, 14, 2, 1, 64)[0] is not None) == narrow, (rows, past)


def test_32_bit_tiles_hold_every_row_once_and_the_longest_walks_come_first():
    rng = random.Random(3)
    for cols, n_heads, n_kv, maps in ((64, 14, 2, 1), (128, 8, 8, 1), (64, 8, 2, 2), (64, 6, 2, 1)):
        rows, past = zip(*[(rng.choice([1, 15, 16, 17, 100, 333]), rng.choice([0, 1, 500])) for _ in range(40)])
        step, group = _f32_step(rows, past), n_heads // n_kv
        tiles, rest, split = _f32_tiles(step, n_heads, n_kv, maps, cols)
        assert sorted(map(tuple, tiles.tolist())) == [(r, c) for r, n in enumerate(rows) if n >= F32_TILE_MIN for c in range(0, n * group, cols)]
        starts = [past[r] + c // group for r, c in tiles.tolist()]
        assert starts == sorted(starts, reverse=True)
        assert rest.tolist() == [t for t, r in enumerate(step.h_row_req) if rows[r] < F32_TILE_MIN] and not split      # (more workgroups than are worth four each)
    assert _f32_tiles(_f32_step([200], [0]), 8, 2, 1, 128)[1:] == (None, True)


def test_steps_beyond_a_launch_of_32_bit_tiles_stay_with_the_plain_kernel():
    """The entry point takes fewer than 2^26 columns of whole tiles; the plain kernel takes any number of rows."""
    for rows, n_heads, n_kv, cols, takes in (([16], 64 * 16, 16, 64, True), ([1 << 20], 64, 64, 64, False), ([(1 << 20) - 64], 64, 64, 64, True),
                                             ([1 << 19, 1 << 19], 64, 1, 128, False), ([17] * 4, 1 << 20, 1 << 20, 64, False)):
        step = types.SimpleNamespace(h_q_len=np.asarray(rows, np.int32), h_kv_len=np.asarray(rows, np.int32), h_row_req=np.zeros(0, np.int64),
                                     upload=torch.from_numpy)
        tiles = _f32_tiles(step, n_heads, n_kv, 1, cols)[0]
        assert (tiles is not None) == takes, (rows, n_heads, n_kv)
        assert tiles is None or len(tiles) * n_kv * cols // 4 < 1 << 24


def test_two_groups_of_waves_and_rows_beside_the_tiles_where_both_were_measured():
    cases = [  # rows of the prompts' portions, their keys, query heads, keys of the other rows, their pairs, window, splits -> (two groups, beside)
        ([500], [500], 16, [], 0, None, 1, (True, False)),
        ([61], [64], 14, [], 0, None, 1, (False, False)),                   # a single tile has nothing for the second group
        ([61], [65], 14, [], 0, None, 1, (True, False)),
        ([500], [500], 16, [299] * 23, 46, None, 1, (True, True)),          # 28.7 us in three launches, 15.6 in one
        ([500], [500], 16, [1575] + [50] * 3, 8, None, 1, (True, True)),    # 4 x 1,575 = 7 x 500 + 2,800
        ([500], [500], 16, [1576] + [50] * 3, 8, None, 1, (True, False)),
        ([512], [2012], 16, [981] * 20, 40, None, 4, (False, False)),       # 2,012 keys: beyond the longest walk
        ([300], [1500], 16, [981] * 20, 40, None, 4, (True, True)),
        ([300], [1500], 16, [], 0, None, 4, (False, False)),                # in splits
        ([128], [128], 16, [1900] * 4, 8, None, 1, (True, False)),          # a row longer than the tiles: 18 us after them, 25.6 beside
        ([128], [128], 16, [924] * 4, 8, None, 1, (True, True)),
        ([128], [128], 16, [925] * 4, 8, None, 1, (True, False)),
        ([128], [128], 16, [1900] * 4, 8, 200, 1, (True, True)),            # ... of which a window leaves 200 keys
        ([64], [3000], 16, [150] * 4, 8, 512, 1, (True, True)),
        ([512, 512], [512, 512], 16, [896] * 4, 8, None, 1, (True, True)),  # more workgroups than compute units
        ([512, 512], [512, 512], 16, [897] * 4, 8, None, 1, (True, False)),
        ([512, 512, 1], [512, 512, 1], 16, [276] * 23, 46, None, 1, (False, False)),    # more tiles than compute units
        ([500], [500], 16, [299] * 40, 320, None, 1, (True, False)),
        ([500], [500], 16, [299] * 20, 40, None, 1, (True, True)),
    ]
    for rows, keys, heads, row_keys, pairs, window, splits, want in cases:
        assert choose_groups(rows, keys, heads, row_keys, pairs, window, splits) == want, (rows, keys, heads, row_keys, pairs, window)
        assert not choose_groups(rows, keys, heads, row_keys, pairs, window, splits, beside_fits=False)[1]


def test_few_tiles_with_long_walks_keep_their_splits_whatever_is_beside_them():
    for heads, rows, keys, want in ((16, 25, 1152, (True, True)), (16, 25, 1153, (False, False)), (28, 31, 1518, (False, False)), (12, 156, 1413, (False, False)),
                                    (12, 200, 1536, (True, True)), (16, 130, 1500, (True, True)), (16, 130, 1537, (False, False))):
        assert choose_groups([rows], [keys], heads, [11], 2, None, 3) == want, (heads, rows, keys)
    assert choose_groups([25], [3000], 16, [11], 2, 1024, 3) == (True, True)           # (a window of 1,024: 1,088 keys)
