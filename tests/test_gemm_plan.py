"""The choice of kernel for a matrix product is made on the host: its invariants are checked
here without a GPU, over a grid of sizes (the library is compiled if it is not there yet)."""
import itertools

import pytest

from herbert_rs_amd.kernels import lib

EPI_STORE, EPI_ADD, EPI_SWIGLU = 0, 1, 2
TILES = {112: (128, 32), 124: (128, 64), 184: (256, 64), 122: (128, 128), 142: (256, 128), 188: (256, 256), 123: (128, 128),
         168: (192, 256), 164: (96, 64), 186: (256, 192)}


@pytest.fixture(scope="module")
def plan():
    from herbert_rs_amd.kernels import mfma  # noqa: F401  (registers the signatures)
    fn = lib.load("gemm_mfma").hb_gemm_mfma_plan

    def ask(M, N, K, epi=EPI_STORE, normed=False, emit=False, scaled=False, workspace=1 << 24, deferred=False):
        return fn(M, N, K, epi, int(normed), int(emit), int(scaled), workspace, int(deferred))
    return ask


ROWS = [1, 2, 7, 8, 16, 17, 32, 33, 64, 65, 100, 256, 700, 1024, 2048, 5000]
WIDTHS = [64, 1024, 2048, 4096, 5120, 6144, 12288, 24576, 151936]
DEPTHS = [64, 128, 512, 2048, 2112, 4096, 12288, 25600]


def test_every_plan_is_a_kernel_that_takes_the_product(plan):
    for M, N, K in itertools.product(ROWS, WIDTHS, DEPTHS):
        for epi in (EPI_STORE, EPI_ADD, EPI_SWIGLU):
            p = plan(M, N, K, epi)
            assert p >= 0, (M, N, K, epi)
            if p == 0:
                assert M <= 16
                continue
            tile, slices = p % 1000, max(1, p // 1000)
            assert tile in TILES and (tile != 112 or M <= 32), (M, N, K, p)
            assert tile not in (168, 164) or (epi == EPI_SWIGLU and slices == 1), (M, N, K, p)
            assert tile != 164 or 32 < M <= 64, (M, N, K, p)
            steps = K // 64
            if slices > 1:
                per = -(-steps // slices)
                assert per * (slices - 1) < steps, (M, N, K, p)            # no slice of K is empty
                assert steps // slices >= 4 and slices * M * N <= 1 << 24, (M, N, K, p)
                assert slices in (2, 4, 8, 16)


def test_without_a_workspace_k_is_never_cut(plan):
    for M, N, K in itertools.product(ROWS, WIDTHS, DEPTHS):
        assert plan(M, N, K, EPI_ADD, workspace=0) < 1000


def test_k_in_steps_of_32_only_goes_to_the_kernel_built_for_it(plan):
    for M in (1, 16, 17, 64, 300):
        p = plan(M, 4096, 4096 + 32)
        assert p == (0 if M <= 16 else 123)


def test_a_norm_is_left_behind_by_the_few_row_kernel_or_by_the_kernel_that_adds_slices(plan):
    for M, N, K in itertools.product([1, 8, 16, 17, 40, 64, 128, 512], [192, 2048, 4096, 5120, 8192], [512, 4096, 25600]):
        p = plan(M, N, K, EPI_ADD, emit=True)
        if M <= 16:
            assert p == 0 or p >= 2000, (M, N, K, p)
        else:
            assert p >= 2000 or p == -1, (M, N, K, p)          # -1: nothing fits; the caller then norms by itself
            if M <= 64:
                assert p >= 2000, (M, N, K, p)
    assert plan(40, 8196, 4096, EPI_ADD, emit=True) == -1      # rows too wide for the adding kernel
    assert plan(40, 4096, 4096, EPI_ADD, emit=True, workspace=0) == -1


def test_a_handed_on_norm_is_finished_by_the_few_row_kernel_or_the_128x32_tile(plan):
    for M, N, K in itertools.product([1, 8, 16], [1024, 6144, 24576, 51200], [1024, 4096, 5120]):
        for epi in (EPI_STORE, EPI_SWIGLU):
            p = plan(M, N, K, epi, scaled=True)
            assert p == 0 or p % 1000 == 112, (M, N, K, epi, p)


def test_slices_left_to_the_next_kernel_are_2_4_or_8(plan):
    for M, N, K in itertools.product([1, 8, 16, 40, 100, 256, 700], [1024, 4096, 6144, 10240], [2048, 4096, 8192, 25600]):
        p = plan(M, N, K, deferred=True)
        assert p // 1000 in (0, 2, 4, 8), (M, N, K, p)


def test_known_choices(plan):
    """A few choices that measurements decided: decoding 8 rows of the 8B shape, its prompt of 2048."""
    assert plan(8, 4096, 4096, EPI_ADD, emit=True) == 0                # o: the few-row kernel
    assert plan(8, 24576, 4096, EPI_SWIGLU, scaled=True) == 112        # gate/up: 128 x 32 tiles, no slices
    assert plan(8, 5120, 25600, EPI_ADD, emit=True) >= 2000            # hidden 5120: 320 workgroups would not spread
    assert plan(2048, 24576, 4096, EPI_SWIGLU) == 188
    assert plan(2048, 4096, 12288, EPI_ADD) == 142
    assert plan(64, 24576, 4096, EPI_SWIGLU) == 164                    # 256 tiles of 96 columns, not 192 of 128
    assert plan(32, 24576, 4096, EPI_SWIGLU) == 112 and plan(64, 51200, 5120, EPI_SWIGLU) % 1000 in (124, 184)


def test_rows_just_past_whole_tiles_are_cut_off_as_a_product_of_their_own():
    """A product whose rows end a little past a whole number of large tiles would pay a round of
    tiles for them: it is cut in two along its rows where the estimates say so, never where the
    rows fill their tiles, and never for few rows."""
    from herbert_rs_amd.kernels import mfma  # noqa: F401
    split = lib.load("gemm_mfma").hb_gemm_mfma_split
    W = 1 << 26
    H, I = 4096, 12288
    for M in (2049, 2064, 2112):
        assert split(M, 2 * I, H, EPI_SWIGLU, W) == 2048 and split(M, H, I, EPI_ADD, W) == 2048, M
    assert split(2049, 2 * I, H, EPI_SWIGLU, 0) == 2048           # (a rest of few rows needs no room for K slices)
    for M in (1, 16, 64, 128, 1024, 2048, 2304, 4096):
        for N, K, epi in ((2 * I, H, EPI_SWIGLU), (H, I, EPI_ADD), (H, H, EPI_ADD), (6144, H, EPI_STORE)):
            assert split(M, N, K, epi, W) == 0, (M, N, K)
    for M, N, K in itertools.product([130, 257, 300, 513, 700, 1025, 1500, 3000, 5000], WIDTHS, [512, 2048, 4096, 12288]):
        for epi in (EPI_STORE, EPI_ADD, EPI_SWIGLU):
            for ws in (0, W):
                rows = split(M, N, K, epi, ws)
                assert rows == 0 or (0 < rows < M and rows % 128 == 0 and M - rows < 256), (M, N, K, epi, rows)


def test_decode_attention_ranges_by_how_evenly_the_waves_sit():
    """One range a (sequence, kv head) from 512 of them on, unless the waves would sit unevenly on
    the CUs (three on some where most have two, or a second round that is a quarter full): then
    eight shorter ranges; below, as many ranges as fill one round of 1,024 waves."""
    from herbert_rs_amd.kernels import mfma

    class Meta:
        def __init__(self, seqs, tokens):
            self.num_seqs, self.context_bucket = seqs, tokens
    split = lambda b, t=4096, nkv=8, window=0: mfma._decode_split(Meta(b, t), nkv, window)
    assert split(1) == (32, 2) and split(8) == (16, 4) and split(32) == (4, 16) and split(48) == (2, 32)
    for b in (64, 80, 96, 128, 200, 256):
        assert split(b) == (1, 64), b
    for b in (65, 72, 136, 160):
        assert split(b) == (8, 8), b
    assert split(65, 1024) == (4, 4) and split(65, 512) == (1, 8)
    assert split(65, 4096, window=100) == (1, 3)
    for b in range(1, 300, 7):
        for t in (64, 700, 4096, 32768):
            ranges, per = split(b, t)
            span = -(-t // 64)
            assert ranges >= 1 and per >= 1 and ranges * per >= span > (ranges - 1) * per, (b, t)


def test_decode_attention_merges_in_a_workgroup_only_where_ranges_stay_short():
    """The waves of a workgroup that share a (sequence, kv head), by pairs of those and bucket of the context: none where they would
    make a range several times longer, but for contexts of up to 256 tokens and, where single pages would sit two and more to a
    CU, of up to 512."""
    from herbert_rs_amd.kernels import mfma

    class Meta:
        def __init__(self, seqs, tokens):
            self.num_seqs, self.context_bucket = seqs, tokens
    waves = lambda pairs, tokens, window=0: mfma._range_waves(pairs, *mfma._decode_split(Meta(pairs, tokens), 1, window))
    for pairs in (1, 8, 64, 95):
        assert waves(pairs, 256) == 2, pairs
        for tokens in (512, 768, 1024, 1536, 2048, 4096, 32768):
            assert waves(pairs, tokens) == 1, (pairs, tokens)
    for pairs in (96, 128, 160):
        assert [waves(pairs, t) for t in (256, 512, 768, 1024, 2048, 4096)] == [2, 3, 1, 1, 1, 1], pairs
    assert [waves(192, t) for t in (256, 512, 768, 1024, 3072, 4096)] == [2, 3, 3, 3, 3, 1]
    assert [waves(256, t) for t in (256, 512, 768, 1024, 2048, 4096)] == [2, 3, 3, 3, 3, 3]
    assert [waves(257, t) for t in (256, 512, 1024, 4096)] == [1, 1, 1, 1] and waves(600, 256) == 1
    assert waves(8, 4096, window=64) == 2 and waves(8, 4096, window=400) == 1
    for pairs, tokens in itertools.product(range(1, 300, 9), (256, 512, 768, 1280, 2048, 8192)):
        splits, per = mfma._decode_split(Meta(pairs, tokens), 1, 0)
        n = waves(pairs, tokens)
        assert n == 1 or splits * per <= 8 or -(-splits * per // n) <= 2 * per, (pairs, tokens)


def test_decode_attention_takes_a_list_of_ranges_only_where_it_fits():
    """The list that deals the decode grid out over sequences of unequal lengths: for two sequences
    or more without a window, a round of waves or two items a sequence, up to the kernel's 1,024
    items; else equal shares."""
    import torch
    from herbert_rs_amd.engine.batch import StepEntry, pack, range_list
    from herbert_rs_amd.kernels import mfma

    def meta_of(contexts):
        return pack([StepEntry(i, [1], [0]) for i in range(len(contexts))], [c - 1 for c in contexts],
                    torch.device("cpu"))
    unequal = [9000] + [100] * 7
    items, listed = mfma._decode_ranges(meta_of(unequal), 8, 0)
    assert items == 128 and listed.tolist() == range_list(unequal, 128, 64).tolist()
    assert mfma._decode_ranges(meta_of(unequal), 2, 0)[0] == 512
    assert mfma._decode_ranges(meta_of(unequal), 1, 0)[0] == 1024           # the grid's z has no more
    assert mfma._decode_ranges(meta_of(unequal), 8, 70) is None             # a window
    assert mfma._decode_ranges(meta_of([9000] * 4 + [8000] * 4), 8, 0) is None      # lengths alike
    assert mfma._decode_ranges(meta_of([9000]), 8, 0) is None
    assert mfma._decode_ranges(meta_of([9000] + [100] * 64), 8, 0)[0] == 130   # two items a sequence
    assert mfma._decode_ranges(meta_of([9000] + [100] * 39), 16, 0)[0] == 80
    assert mfma._decode_ranges(meta_of([9000] + [100] * 31), 16, 0)[0] == 64
    assert mfma._decode_ranges(meta_of([9000] + [100] * 511), 8, 0)[0] == 1024
    assert mfma._decode_ranges(meta_of([9000] + [100] * 512), 8, 0) is None     # more items than the kernel takes
    half = [4000] * 40 + [200] * 40                             # holds 0.525 of 80 x 4000: level 1
    assert meta_of(half).unequal == 1 and meta_of(half[8:72]).unequal == 1
    assert mfma._decode_ranges(meta_of(half), 8, 0) is None     # more than a round of waves: from level 2 on
    assert mfma._decode_ranges(meta_of(half[8:72]), 8, 0)[0] == 128
    prompt = pack([StepEntry(0, [1, 2, 3], [2]), StepEntry(1, [4], [0])], [9000, 10], torch.device("cpu"))
    assert prompt.unequal and mfma._decode_ranges(prompt, 8, 0) is None     # not one token a sequence


def test_a_plan_names_the_height_of_its_tiles(plan):
    """What is launched is the plan's own tile, heights between 128 and 256 rows among them: every plan of more than 64 rows has the
    height of its number, 186 one of three, each of which some product takes; and the q/k/v product that writes the cache."""
    rows_of = lib.load("gemm_mfma").hb_gemm_mfma_plan_rows
    taken = set()
    for M, N, K in itertools.product([64, 65, 200, 700, 1500, 2048, 2600, 3072, 5000, 9404], WIDTHS, [512, 2048, 4096, 12288]):
        for epi in (EPI_STORE, EPI_ADD, EPI_SWIGLU):
            rows, tile = rows_of(M, N, K, epi, 1 << 24), plan(M, N, K, epi) % 1000
            if M <= 64:
                assert rows == 0
            elif tile == 186:
                assert rows in (160, 192, 224), (M, N, K, epi)
                taken.add(rows)
            else:
                assert rows == TILES[tile][1], (M, N, K, epi)
    assert taken == {160, 192, 224}
    assert rows_of(300, 4096, 4096 + 32, EPI_STORE, 1 << 24) == 0          # K in steps of 32: a kernel of its own
    qkv = lib.load("gemm_mfma").hb_gemm_qkv_tile
    assert qkv(2048, 6144, 4096) == 187 and qkv(8192, 6144, 4096) == 188
    assert {qkv(m, n, 2048) for m in range(1500, 9500, 100) for n in (4096, 6144)} == {185, 186, 187, 188}


def test_products_of_65_to_256_rows_keep_the_tiles_of_256_columns(plan):
    """One workgroup a CU on tiles of 256 x 64 does the 8B shape's products of around 100 rows sooner than two on tiles of 128 x 64
    (128 rows: gate/up 47 against 51 us, down 34 against 35); with other shares of K they are even, and o's few columns go the other way."""
    for M in (100, 128):
        assert plan(M, 24576, 4096, EPI_SWIGLU) == 184 and plan(M, 4096, 12288, EPI_ADD) == 8184, M
        assert plan(M, 6144, 4096) == 4184 and plan(M, 4096, 4096, EPI_ADD) == 4124, M
    assert plan(200, 12288, 2048, EPI_SWIGLU) == 184 and plan(256, 12288, 2048, EPI_SWIGLU) == 184      # 25 and 26 us; on 124 26 and 30
    assert plan(128, 6144, 4096, deferred=True) % 1000 == 184


def test_a_cut_along_the_rows_is_done_sooner_by_the_estimates():
    """Products whose rows end a little past whole tiles are cut exactly where the two parts' estimates come to less than the whole's."""
    import ctypes
    from herbert_rs_amd.kernels import mfma  # noqa: F401
    native = lib.load("gemm_mfma")
    cost = native.hb_gemm_mfma_plan_cost
    cost.restype = ctypes.c_double
    W, cuts = 1 << 24, 0
    for M, (N, K, epi) in itertools.product([130, 257, 520, 1025, 1300, 2060, 2600, 3075, 4100],
                                            [(24576, 4096, EPI_SWIGLU), (4096, 12288, EPI_ADD), (2048, 2048, EPI_ADD), (6144, 4096, EPI_STORE)]):
        of = lambda m: cost(m, N, K, epi, 0, 0, 0, W, 0)
        parts = {a: of(a) + of(M - a) for a in (M // 128 * 128, M // 256 * 256) if 0 < a < M}
        rows, best = native.hb_gemm_mfma_split(M, N, K, epi, W), min(parts.values())
        assert parts[rows] == best < of(M) if rows else best >= 0.99 * of(M) * (1 - 1e-9), (M, N, K, epi)
        cuts += rows > 0
    assert 3 < cuts < 30


def test_long_projections_past_whole_tiles_write_the_cache_themselves():
    """Rows a little past whole tiles of 256, with a last round of those that is nearly empty: the fused q/k/v product has tiles of
    other heights too and is done sooner than a plain product cut along the rows (8,200 rows of 4096 columns 143 against 179 us)."""
    from herbert_rs_amd.kernels import mfma
    for M, N in ((2600, 6144), (3100, 6144), (8200, 6144), (4120, 4096), (8200, 4096), (3100, 10240), (2048, 6144), (2300, 6144)):
        assert mfma.qkv_tile_shape(M, N) == 0, (M, N)
    assert mfma.qkv_tile_shape(128, 6144) is None and mfma.qkv_tile_shape(2048, 4096) == 1


def test_slices_that_fill_the_chip_with_tiles_alone_on_a_cu_cost_more(plan):
    """Where tiles of 256 columns in eight slices would take nearly every CU, fewer slices or tiles of two a CU are ahead (450 rows of
    2048 x 6144 28.5 to 33 us in eight slices, 26 to 29 in four); with CUs left over the tiles of 256 columns stay."""
    for M, N, K in ((450, 2048, 6144), (500, 2048, 6144), (300, 2560, 9728), (350, 2560, 9728), (384, 4096, 12288)):
        assert not 8140 < plan(M, N, K, EPI_ADD) < 8190, (M, N, K)
    assert plan(200, 2560, 9728, EPI_ADD) == 8142
