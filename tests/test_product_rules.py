"""The rules that choose between the prefill products, at sizes that were timed and at their edges."""
from spite_amd.parts.linear import whole_group_apart


def test_whole_group_apart():
    assert whole_group_apart(2048, 16, 5120, 8192) == 3          # tiles of 128 rows alone would miss their round
    assert whole_group_apart(1547, 16, 5120, 8192) == 1
    for tokens in (1, 65, 600, 1024, 1200):                      # one round together, or the weights' stream is the time
        assert whole_group_apart(tokens, 16, 5120, 8192) == 0
    assert whole_group_apart(2048, 128, 5120, 8192) == 0


def test_whole_group_apart_where_it_was_timed_beside_tiles_of_several_heights():
    for tokens, groups, N, K in ((1522, 8, 5120, 8192), (1629, 8, 5120, 8192), (1743, 8, 5120, 8192), (1685, 16, 5120, 8192), (1865, 32, 3072, 8192)):
        assert whole_group_apart(tokens, groups, N, K) == 1, (tokens, groups, N, K)
    for tokens, groups, N, K in ((850, 4, 2048, 3072), (2048, 8, 2048, 8192), (1200, 4, 3072, 8192), (1000, 8, 5120, 8192), (2600, 16, 5120, 8192)):
        assert whole_group_apart(tokens, groups, N, K) == 0, (tokens, groups, N, K)


def test_lds_suits():
    from spite_amd.csrc.hipops import latent_splits, lds_suits, lds_suits_groups, tiled_k_runs
    faster = {(1547, 5120, 5120): True, (1786, 5120, 8192): True, (1531, 2048, 2048): True, (1024, 7168, 5120): True,
              (512, 5120, 8192): False, (330, 7168, 5120): False, (300, 2048, 2048): False, (100, 512, 1024): False}
    for (M, N, K), yes in faster.items():
        assert lds_suits(M, N, K, False, tiled_k_runs(M, N, K)) is yes, (M, N, K)
    assert lds_suits(300, 16384, 5120, True, 1)
    assert lds_suits_groups(223.0, 5120) and not lds_suits_groups(128.0, 5120) and not lds_suits_groups(383.0, 1024)
    # shares of two blocks of keys, no more workgroups than compute units, shares within 4,096 keys
    assert [latent_splits(2, k) for k in (32, 256, 1024, 4096)] == [1, 8, 16, 32]
    assert latent_splits(16, 4096) == 16 and latent_splits(500, 4096) == 1 and latent_splits(500, 100000) == 25


def test_router_plan_is_one_launch_for_a_token_a_wave():
    """Its one workgroup has eight waves; a token more would wait for another's choice (16 tokens: 17.8 against 12.9 us)."""
    from spite_amd.csrc.hipops import lib
    one = lib().spite_router_plan_is_one_launch
    assert all(one(T, top) for T in (1, 5, 8) for top in (1, 8, 64))
    assert not any(one(T, top) for T in (0, 9, 64, 512) for top in (1, 8)) and not one(4, 65)


def test_latent_splits_beyond_a_window_and_for_many_items():
    """Sizes at which both sides were timed: long contexts for few items, and more items than half the compute units."""
    from spite_amd.csrc.hipops import latent_splits
    at = lambda n, *row: [latent_splits(n, k, *row) for k in (4096, 8192, 16384, 32768)]
    assert at(1) == [32, 64, 128, 256] and at(2) == [32, 64, 128, 128] and at(4) == [32, 64, 64, 64] and at(8) == [32] * 4
    assert latent_splits(1, 131072) == 256 and latent_splits(6, 16384) == 42
    for n in (100, 150, 200, 255):                       # narrow rows: several workgroups a unit
        assert latent_splits(n, 2048, 192, 128) == -(-256 // n) and latent_splits(n, 2048) == 256 // n


def test_latent_splits_of_many_items_with_long_contexts():
    """Sizes that were timed with every count of splits: one round of the compute units stays one, what overflows it is dealt so that
    the rounds come out even, and records cost their way to memory; never more than a split for every 4,096 keys."""
    from spite_amd.csrc.hipops import latent_splits
    assert [latent_splits(n, 4827, rows=40 * 700) for n in (157, 219, 250)] == [1, 1, 1]            # (2 before: 13 % more)
    assert latent_splits(469, 5627, rows=60000) == 1 and latent_splits(94, 16384, rows=12000) == 2
    assert [latent_splits(n, 16384, rows=40 * n) for n in (110, 130, 200, 256, 300, 500, 640)] == [2, 3, 1, 1, 4, 1, 2]
    assert latent_splits(640, 32768, rows=81920) == 2
    for n in range(1, 700, 3):
        for longest in (64, 4096, 4128, 9000, 32768, 50000):
            assert 1 <= latent_splits(n, longest) <= 256
            assert latent_splits(n, longest) <= max(256 // n, -(-longest // 4096)) or n < 2


def test_decode_attention_splits():
    """Where the rule's lines lie, at sizes that were timed with every count of splits."""
    from spite_amd.csrc.hipops import attn_decode_splits
    at = lambda heads, *blocks: [attn_decode_splits(heads, 32 * b) for b in blocks]
    assert at(8, 1, 12, 13, 32, 64, 128, 256, 500, 1000, 4000) == [1, 1, 8, 8, 8, 16, 32, 64, 64, 64]
    assert at(2, 320, 500, 1024, 2000) == [64, 64, 128, 248]            # shares of eight blocks, not of four
    assert at(64, 8, 12, 31, 32, 1000) == [1, 2, 4, 8, 8] and at(128, 16, 31, 500) == [2, 4, 4]
    assert at(256, 9, 32, 33) == [1, 1, 2] and at(512, 500) == [1] and at(5000, 5000) == [1]
    for heads in (1, 3, 40, 100, 300):
        for blocks in range(1, 2100, 7):
            n = attn_decode_splits(heads, 32 * blocks)
            assert 1 <= n <= 256 and n <= -(-512 // heads) and (n < 8 or n % 8 == 0)


def test_groups_of_many_tiles_stay_with_the_tiled_product():
    """The line between the two products over groups, at sizes that were timed on both sides of it."""
    from spite_amd.csrc.hipops import lds_suits_groups
    from spite_amd.parts.linear import _group_tiles
    def suits(T, E, top, whole, N, K, glu):
        return lds_suits_groups(T * top / E, K, *_group_tiles(T * (top + whole), E + whole, T, T * top / E, N, glu))
    assert _group_tiles(2 * 2048, 17, 2048, 128.0, 8192, True) == (32 * 32, 24 * 64)       # 16 experts and a shared one
    assert _group_tiles(700, 7, 700, None, 512, False) == (7, 14)
    assert suits(692, 8, 4, 0, 1024, 4096, True) and suits(533, 4, 2, 0, 2048, 5120, False)
    for slower in ((1416, 8, 1, 1, 5120, 8192, False), (4608, 4, 1, 1, 2048, 3072, False), (694, 4, 2, 1, 3072, 2048, True),
                   (3199, 8, 1, 1, 5120, 8192, False), (1786, 16, 2, 2, 4096, 5120, True), (6992, 128, 4, 1, 1024, 2048, True)):
        assert not suits(*slower), slower


def test_whole_group_stays_where_apart_was_slower():
    """Rounds that the groups alone would miss by a tile, and sizes at which the two take the same time."""
    for tokens, groups, N, K in ((2889, 8, 5120, 4096), (2510, 16, 5120, 4096), (2520, 16, 5120, 8192), (5548, 16, 5120, 4096),
                                 (4291, 16, 5120, 8192), (3252, 2, 5120, 4096), (5255, 8, 2560, 1024), (4096, 32, 5120, 4096),
                                 (2500, 8, 5120, 8192), (6000, 8, 2560, 1024)):
        assert whole_group_apart(tokens, groups, N, K) == 0, (tokens, groups, N, K)
    for tokens, groups, N, K in ((1454, 16, 5120, 8192), (1806, 8, 5120, 8192), (3107, 16, 3072, 8192), (2553, 8, 4096, 14336)):
        assert whole_group_apart(tokens, groups, N, K) == 1, (tokens, groups, N, K)


def test_variants_of_the_weight_stream():
    """Tables between 2^27 and 2^28 elements, on either side of the lines that were timed."""
    from spite_amd.csrc.hipops import lib
    plain = lambda rows, N, K, glu=0: lib().spite_gemm_skinny_variant(rows, N, K, 0, 0, glu, rows)
    assert [plain(r, 32768, 5120) for r in (1, 2, 3, 16, 17, 24, 25, 32)] == [5, 5, 8, 8, 2, 2, 10, 10]
    assert [plain(1, N, K) for N, K in ((16384, 8192), (14736, 10432), (15168, 9536), (16384, 5120), (65536, 4096))] == [5, 8, 8, 8, 4]
    assert [plain(32, N, K) for N, K in ((36864, 5120), (40960, 4096), (24576, 6144), (18432, 14336), (30720, 8192), (28672, 5120))] == [2, 2, 2, 2, 10, 10]
    assert plain(25, 18688, 13760, 1) == 2 and plain(25, 202048, 5120, 0) == 10 and plain(20, 202048, 5120) == 10
    # as it was: few rows, experts' groups, 33 to 64 rows
    assert [plain(1, N, K) for N, K in ((2048, 2048), (5120, 5120), (202048, 5120))] == [6, 8, 4] and plain(16, 202048, 5120) == 7
    group = lambda rows, N, K, glu, live: lib().spite_gemm_skinny_variant(rows * 2, N, K, 17, live, glu, rows)
    assert group(8, 8192, 5120, 1, 9) == 5 and group(8, 5120, 8192, 0, 9) == 6 and group(40, 8192, 5120, 1, 17) == 2 and group(40, 5120, 8192, 0, 17) == 10
    assert plain(40, 5120, 5120) == 9 and plain(60, 5120, 5120) == 10 and plain(60, 3072, 2048) == 2


def test_short_sums_of_many_rounds_stay_with_the_tiled_product():
    """Products that both were timed at and that were 3 to 10 % slower with both operands in LDS."""
    from spite_amd.csrc.hipops import lds_suits, tiled_k_runs
    for M, N, K, glu in ((7902, 18304, 448, True), (3601, 8320, 896, False), (7489, 22032, 448, False), (6362, 23024, 128, True),
                         (6907, 28704, 320, True), (7136, 20448, 256, False), (1822, 28224, 2048, True), (2933, 4256, 1536, True),
                         (5743, 10352, 768, False), (1871, 28704, 768, False)):
        assert not lds_suits(M, N, K, glu, 1 if glu else tiled_k_runs(M, N, K)), (M, N, K, glu)
