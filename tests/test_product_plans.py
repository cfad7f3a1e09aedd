"""The plans of the few-row matrix products are host arithmetic: which kernel, how many blocks
along k.  A plan may depend on the matrix and on the class of the row count (up to 16, 32, 64,
128 rows) only, so that a row's sums come in the same order for every batch of its class; the
consumers of partial sums take at most 8 parts."""
import importlib

import pytest
import torch

K = importlib.import_module("daisi-llogos_amd.ops.kernels")

SHAPES = [(24576, 4096), (37888, 3584), (51200, 5120), (59136, 8192),                     # other models' gate/up
          (6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336), (128256, 4096),      # Llama-3.1-8B
          (7168, 5120), (5120, 5120), (34816, 5120), (5120, 17408), (151936, 5120),      # Qwen3-14B
          (10240, 8192), (8192, 8192), (57344, 8192), (8192, 28672),                     # Llama-3.1-70B
          (3072, 2048), (16384, 2048), (2048, 8192), (331, 80), (96, 1000), (17, 8)]


@pytest.mark.parametrize("N,K_", SHAPES)
def test_a_plan_depends_on_the_class_of_the_row_count_only(N, K_):
    for lo, hi in ((1, 4), (5, 8), (9, 16), (17, 32), (33, 64)):
        plans = {K.skinny_plan(M, N, K_) for M in range(lo, hi + 1)}
        if hi <= 16:
            # up to 16 rows the kernel may change with the row count (activations held in
            # registers for the fewest rows), but not within 1..4, 5..8 and 9..16
            assert len(plans) == 1, (N, K_, lo, hi, plans)
        else:
            assert len(plans) == 1 and next(iter(plans))[0] in ("lds", "strips"), (N, K_, lo, hi, plans)
    assert len({K.lds_splits(M, N, K_) for M in range(65, 129)}) == 1


@pytest.mark.parametrize("N,K_", SHAPES)
def test_plans_are_within_what_the_kernels_and_their_consumers_take(N, K_):
    for M in (1, 4, 8, 16, 32, 64, 128):
        parts = K.lds_splits(M, N, K_)
        assert 1 <= parts <= 8
        assert parts == 1 or -(-K_ // 256) >= 2 * parts - 1        # every block along k has work
        if M <= 64:
            kernel, splits, third = K.skinny_plan(M, N, K_)
            assert kernel in ("stationary", "regs", "lds", "strips") and 1 <= splits <= 8 and third >= 1
            if kernel == "strips":
                blocks = -(-(-(-N // 16)) // third) * splits
                assert 16 < M and 5 <= third <= 9 and K_ % 64 == 0 and 0.75 * 512 <= blocks <= 512
            if kernel == "stationary":
                assert M <= 16 and K_ <= 8192 and 2 <= third <= 16
    assert 2 <= K.stationary_strips(N, K_) <= 16


def test_known_choices():
    """The choices measured to be best at the Llama-3.1-8B layer sizes (they are what the
    scoring was fitted to; a change of the scoring that moves them should be a decision)."""
    assert K.skinny_plan(8, 28672, 4096)[0] == "stationary"
    assert K.skinny_plan(8, 4096, 14336) == ("lds", 8, 1)
    assert K.skinny_plan(8, 4096, 4096) == ("lds", 8, 1)
    assert K.skinny_plan(64, 28672, 4096) == ("lds", 1, 1)
    assert K.skinny_plan(64, 6144, 4096) == ("lds", 4, 1)
    assert K.lds_splits(128, 4096, 14336) == 8
    # tall matrices whose blocks of 5 to 9 strips are all resident at once: operands straight into LDS
    assert K.skinny_plan(32, 34816, 5120) == ("strips", 2, 9) and K.skinny_plan(64, 34816, 5120) == ("strips", 2, 9)
    assert K.skinny_plan(64, 57344, 8192) == ("strips", 1, 7)
    assert K.skinny_plan(16, 57344, 8192)[0] == "stationary" and K.skinny_plan(64, 128256, 4096)[0] == "lds"
    assert K.skinny_plan(64, 24576, 4096) == ("strips", 2, 6) and K.skinny_plan(32, 37888, 3584) == ("strips", 1, 5)
    assert K.skinny_plan(64, 51200, 5120) == ("strips", 1, 7) and K.skinny_plan(64, 59136, 8192) == ("strips", 1, 8)
    # ... and not where the LDS few-row product's own blocks fill one round well, or the matrix is small
    assert K.skinny_plan(64, 28672, 4096)[0] == "lds" and K.skinny_plan(32, 28672, 4096)[0] == "lds"
    assert K.skinny_plan(64, 16384, 3072)[0] == "lds" and K.skinny_plan(64, 19456, 2560)[0] == "lds"


def test_sets_of_waves_of_the_prompt_attention():
    """Two sets of waves a block where one prompt's last tile would set the time, one where the
    work of all tiles does (the measured cases at 32 heads)."""
    for lens, want in (([512], 2), ([1536], 2), ([2048], 2), ([2560], 1), ([4096], 1), ([16384], 1),
                       ([1024] * 2, 2), ([512] * 4, 1), ([256] * 4, 2), ([512] * 8, 1)):
        assert K.prefill_halves(lens, None, 32) == want, lens
    # a continued prompt counts the pages before it
    assert K.prefill_halves([128], [4000], 32) == 2 and K.prefill_halves([128] * 64, [4000] * 64, 32) == 1


def test_where_the_tiled_product_serves_prompts(monkeypatch):
    """By default the tiled product takes the gate/up product with its SwiGLU epilogue at 1,024 to 2,048 rows and
    k up to 5,120, and plain products only for matrices much longer than high at 129 to 1,024 rows, in parts of
    k that hold at least two stages of 64."""
    assert K.PROMPT_PRODUCT == "auto"
    assert K.tiles_serve_gated(1024, 4096) and K.tiles_serve_gated(2048, 5120) and not K.tiles_serve_gated(1023, 4096)
    assert not K.tiles_serve_gated(2049, 4096) and not K.tiles_serve_gated(2048, 8192)
    down = (4096, 14336)
    assert K.tiles_plan(64, *down) is None and K.tiles_plan(128, *down) is None          # the few-row products' rows
    assert K.tiles_plan(129, *down) == (4, 2) and K.tiles_plan(256, *down) == (4, 2)
    assert K.tiles_plan(300, *down) == (4, 0) and K.tiles_plan(1024, *down) == (2, 0)
    assert K.tiles_plan(1025, *down) is None
    assert K.tiles_plan(300, 4096, 4096) is None and K.tiles_plan(300, 6144, 4096) is None   # o, qkv: the library's
    assert K.tiles_plan(300, 64, 320) == (2, 0)                                          # 5 stages of 64: not 4 parts
    assert K.tiles_plan(300, 64, 200) is None                                            # k no multiple of 64
    monkeypatch.setattr(K, "PROMPT_PRODUCT", "library")
    assert K.tiles_plan(300, *down) is None and not K.tiles_serve_gated(4096)
    monkeypatch.setattr(K, "PROMPT_PRODUCT", "tiles")
    assert K.tiles_plan(300, 4096, 4096) == (1, 0) and K.tiles_serve_gated(65)


def test_gated_products_of_long_prompts_are_the_library_s():
    """Beyond 2,048 rows, whatever k is: sizes at which the library with a SwiGLU pass was measured 2 to 13 % ahead."""
    for M, N, K_ in ((2500, 24576, 4608), (4096, 24576, 4608), (2304, 8192, 4608), (3072, 8192, 4608), (3329, 27648, 5120),
                     (3843, 32768, 5120), (4048, 65536, 4352), (2049, 16384, 5120), (5120, 8192, 5120)):
        assert not K.tiles_serve_gated(M, K_), (M, N, K_)
    assert K.tiles_serve_gated(2048, 4608) and K.tiles_serve_gated(1024, 5120)


def test_long_products_of_prompts_are_tiled_where_that_was_measured_ahead():
    """k of 16,384 and more with more than 1,024 rows: sizes measured on either side of every line of the plan.  The library's
    product was 3 to 19 % ahead at the first ones, the tiled one level or ahead at the others."""
    plan = lambda M, N, K_: K.long_tiles_plan(M, N, K_, n_cus=256)
    for M, N, K_ in ((6145, 4096, 21504), (6400, 4096, 21504), (2432, 10240, 18432), (2379, 10240, 21504),      # 400 tiles
                     (10000, 4096, 21504), (10000, 5120, 17408), (6592, 6144, 18432), (5952, 7168, 18432),      # three rounds
                     (6145, 8192, 28672), (6656, 8192, 28672),                                                  # and four
                     (7232, 2048, 16384), (4672, 3072, 16384), (5820, 2560, 16384), (1692, 8448, 16384),        # 228 to 231 tiles
                     (1306, 8448, 16384), (2560, 4096, 21504), (4096, 4096, 21504), (6144, 4096, 21504), (8192, 4096, 21504),
                     (1832, 6400, 18944), (1133, 10240, 26624), (1899, 12800, 16896), (1916, 12800, 28608),     # tiles not filled
                     (1723, 512, 32256), (1100, 4096, 16384), (2432, 3072, 16384), (4032, 2048, 16384),
                     (1024, 4096, 21504), (2048, 4096, 16320)):
        assert plan(M, N, K_) is None, (M, N, K_)
    for M, N, K_ in ((1025, 4096, 21504), (2048, 4096, 21504), (1400, 5120, 17408), (1792, 2048, 32256), (1896, 1024, 40960), (2900, 2560, 30720)):
        assert plan(M, N, K_) == (2, 0), (M, N, K_)
    for M, N, K_ in ((3400, 4096, 21504), (3400, 4096, 16384), (1700, 8192, 28672), (2500, 5120, 17408), (2005, 6400, 16896),
                     (6401, 4096, 21504), (7000, 4096, 24576), (7424, 4096, 21504), (5376, 5120, 17408), (3300, 8192, 28672),
                     (5003, 5120, 17408), (6400, 4096, 16384), (5000, 5120, 25600), (2442, 10240, 26624)):
        assert plan(M, N, K_) == (1, 0), (M, N, K_)
    # half of the units: the same shares of them
    assert K.long_tiles_plan(3400, 2048, 21504, n_cus=128) == (1, 0) and K.long_tiles_plan(3400, 4096, 21504, n_cus=128) == (1, 0)
    assert K.long_tiles_plan(1100, 2048, 21504, n_cus=128) == (2, 0) and K.long_tiles_plan(2048, 4096, 21504, n_cus=128) is None


def test_tiles_of_the_experts_product():
    """Tall tiles only where they were measured level or ahead for even and uneven segments; tiles of 64 rows below 96 rows an
    expert, of 128 from there on."""
    few = [(2, 16, 7168, 4096), (64, 16, 4096, 7168), (128, 14, 7168, 4096), (160, 16, 7168, 2048), (100, 8, 4096, 4096), (256, 16, 1024, 2048),
           (200, 16, 7168, 2048), (384, 128, 1536, 2048), (256, 128, 2048, 768)]
    for P, E, N, K_ in few:
        assert K.moe_form(P, E, N, K_, 256) == 0, (P, E, N, K_)
    for P, E, N, K_ in ((48, 8, 8192, 4096), (80, 16, 4096, 4096), (160, 32, 2048, 2048)):        # k a power of two
        assert K.moe_form(P, E, N, K_, 256) == 0 and K.moe_form(11 * E, E, N, K_, 256) == 1, (P, E, N, K_)
    for P, E, N, K_ in ((96, 16, 4096, 7168), (48, 8, 8192, 5120), (128, 16, 4096, 3584), (200, 14, 7168, 4096), (128, 8, 4096, 4096), (257, 16, 1024, 2048),
                        (384, 128, 2048, 768), (520, 128, 1536, 2048), (196, 16, 14336, 4096)):
        assert K.moe_form(P, E, N, K_, 256) == 1, (P, E, N, K_)
    for P, E, N, K_ in ((64 * 16, 16, 1024, 2048), (73 * 14, 14, 7168, 4096), (95 * 16, 16, 4096, 7168), (32 * 8, 8, 28672, 4096)):
        assert K.moe_form(P, E, N, K_) == 1, (P, E, N, K_)
    for P, E, N, K_ in ((96 * 16, 16, 4096, 7168), (141 * 16, 16, 7168, 4096), (144 * 16, 16, 3584, 2048), (256 * 16, 16, 4096, 7168),
                        (292 * 14, 14, 7168, 4096), (512 * 8, 8, 4096, 4096), (1024 * 16, 16, 1024, 2048), (1024 * 16, 16, 7168, 2048),
                        (1024 * 16, 16, 4096, 3584), (336 * 64, 64, 4096, 4096), (1024 * 16, 16, 4096, 5120)):
        assert K.moe_form(P, E, N, K_) == 2, (P, E, N, K_)
    for P, E, N, K_ in ((1024 * 16, 16, 7168, 4096), (1500 * 16, 16, 4096, 7168), (1024 * 8, 8, 14336, 4096), (512 * 8, 8, 28672, 4096),
                        (3000 * 8, 8, 4096, 4096)):
        assert K.moe_form(P, E, N, K_) == 3, (P, E, N, K_)


def test_where_the_product_that_adds_itself_to_the_stream_serves():
    """The one-pass product whose blocks own 16 or 32 rows of w and all of k serves up to 16 rows where its
    blocks fill the compute units evenly (256 of them here): one strip a block up to 256 strips (1B, 3B, 8B), two
    above (14B, 70B); the 14B down projection (160 blocks, 89 M weights) only up to 4 rows; never more than 16
    rows or a k that is no multiple of 8; tiny matrices always."""
    plan = lambda M, N, K_: K.residual_plan(M, N, K_, n_cus=256)
    for M in (1, 8, 16):
        assert plan(M, 4096, 4096) == (8, 1) and plan(M, 4096, 14336) == (8, 1)         # 8B
        assert plan(M, 2048, 2048) == (8, 1) and plan(M, 2048, 8192) == (8, 1)          # 1B
        assert plan(M, 3072, 3072) == (8, 1) and plan(M, 3072, 8192) == (8, 1)          # 3B
        assert plan(M, 8192, 8192) == (8, 2) and plan(M, 8192, 28672) == (8, 2)         # 70B
        assert plan(M, 5120, 5120) == (8, 2)                                             # 14B o
        assert plan(M, 5120, 17408) == ((8, 2) if M <= 4 else (0, 0))                    # 14B down
        assert plan(M, 1024, 8192) == (0, 0)                                             # 64 blocks on 256 units
        assert plan(M, 120, 384) == (4, 1) and plan(M, 64, 176) == (4, 1)               # tiny: only the kernel count matters
        assert plan(M, 4096, 4100) == (0, 0)
    assert plan(17, 4096, 4096) == (0, 0) and plan(0, 4096, 4096) == (0, 0)
    assert K.residual_plan(8, 4096, 4096, n_cus=64) == (8, 2)                            # fewer units: two strips a block


def test_where_that_product_takes_half_a_strip_a_block():
    """Half a strip of 16 rows of w a block where whole strips would leave half of the units without one and k is no short one."""
    form = lambda N, K_: K.residual_form(N, K_, *K.residual_plan(8, N, K_, n_cus=256), n_cus=256)
    assert form(2048, 8192) == (8, 0) and form(2048, 2048) == (16, 0) and form(1024, 4096) == (16, 0) and form(2041, 4104) == (8, 0)
    assert form(2064, 8192) == (8, 1) and form(4096, 14336) == (8, 1) and form(8192, 8192) == (8, 2)
    assert form(64, 176) == (4, 1) and form(1024, 8192) == (0, 0)


def test_short_sums_keep_whole_strips():
    """A wave with two steps of k or fewer adds no more exactly by halves, and no faster."""
    form = lambda N, K_: K.residual_form(N, K_, *K.residual_plan(8, N, K_, n_cus=256), n_cus=256)
    assert {form(N, K_) for N in (64, 1024, 2048) for K_ in (1024, 1032, 1152, 1280, 1400)} == {(8, 1)}
    assert form(2048, 1408) == (16, 0) and form(64, 1408) == (16, 0)


def test_which_recurrence_serves_short_prompts_of_heads_of_64():
    """Steps measured on either side of the line: at the first ones the kernel with a block a head was ahead (by 8 to 60 %), at the
    others the one with a wave a head; and a prompt just above the line is cut into segments of two whole chunks of eight."""
    for batch, heads, longest in ((1, 64, 2), (1, 64, 16), (1, 8, 40), (1, 128, 64), (1, 64, 80), (8, 32, 20), (8, 32, 5), (6, 40, 2), (4, 32, 64)):
        assert not K.wave_scan_serves(batch, heads, longest, n_cus=256), (batch, heads, longest)
    for batch, heads, longest in ((1, 64, None), (64, 64, None), (8, 40, 20), (8, 64, 5), (6, 64, 2), (40, 8, 2), (1, 64, 127), (1, 8, 100), (1, 64, 2048)):
        assert K.wave_scan_serves(batch, heads, longest, n_cus=256), (batch, heads, longest)
    assert K.wave_scan_segments(1, 64, 100, n_cus=256) == 7 and K.wave_scan_segments(1, 8, 127, n_cus=256) == 8
    assert K.wave_scan_segments(8, 64, 20, n_cus=256) == 1 and K.wave_scan_segments(1, 64, 8000, n_cus=256) == 32


def test_rows_of_logits_beyond_a_grids_height_are_left_to_the_general_sampler():
    """The sampler for a small top-k has a row of its grid a row of logits, of which a grid has 65,535."""
    assert K.sample_few_serves(65535, 100, 40) and not K.sample_few_serves(65536, 100, 40)
    assert K.sample_few_serves(1, 128256, 256) and not K.sample_few_serves(1, 128256, 257) and not K.sample_few_serves(0, 100, 40)


def test_parts_are_chosen_for_the_height_that_the_launch_takes():
    """Parts were once chosen for tiles of 64, 128 or 192 tokens and launched in tiles of another height.  By the costs of the launch no number of parts is
    cheaper than the one chosen, and each part holds four stages or more."""
    for N in (2048, 3072, 4096, 5120, 7168, 8192):
        for K_ in (2048, 2112, 4096, 14336, 21504):
            for M in (65, 100, 128, 129, 192, 193, 209, 256, 257, 334, 512, 700, 1024):
                parts = K.wide_tiles_plan(M, N, K_, n_cus=256)
                assert 1 <= parts <= 8 and (parts == 1 or K_ // 64 // parts >= 4)
                cost = lambda p: K._lib().llogos_gemm_tiles_cost(M, N, K_, p, 256) + p * (M * N * 0.8e-6 + 0.4)
                assert all(cost(parts) <= cost(p) for p in range(1, 9)), (M, N, K_)
    assert K.prompt_parts(200, 4096, 14336) == K.wide_tiles_plan(200, 4096, 14336) > 1


def test_wide_tiles_have_parts_that_the_kernel_takes(monkeypatch):
    """More than 64 rows of matrices of 512 rows and columns on, each part of four stages or more."""
    for N in (512, 1536, 2048, 6144, 10240, 28672):
        for K_ in (512, 576, 4096, 14336, 21504):
            for M in (65, 129, 334, 1024, 1025, 2048, 5003, 16384):
                parts = K.wide_tiles_plan(M, N, K_, n_cus=256)
                assert 1 <= parts <= 8 and (parts == 1 or K_ // 64 // parts >= 4)
    assert K.wide_tiles_plan(128, 4096, 14336, n_cus=256) > 2 and K.wide_tiles_plan(5003, 28672, 4096, n_cus=256) == 1
    for M, N, K_ in ((64, 4096, 4096), (2048, 4096, 4100), (2048, 511, 4096), (2048, 514, 4096), (2048, 4096, 448)):
        assert K.wide_tiles_plan(M, N, K_, n_cus=256) == 0
    assert K.wide_tiles_serve_gated(334, 28672, 4096) and K.wide_tiles_serve_gated(5003, 34816, 5120) and K.wide_tiles_serve_gated(256, 16384, 2048)
    assert not K.wide_tiles_serve_gated(100, 28672, 4096) and not K.wide_tiles_serve_gated(255, 16384, 2048) and not K.wide_tiles_serve_gated(64, 1 << 20, 4096)
    assert not K.wide_tiles_serve_gated(2048, 28672, 4100)
    for how in ("library", "tiles"):
        monkeypatch.setattr(K, "PROMPT_PRODUCT", how)
        assert K.wide_tiles_plan(2048, 4096, 4096, n_cus=256) == 0 and not K.wide_tiles_serve_gated(2048, 28672, 4096)


def test_packed_experts_tiles():
    """Few rows up to ten an expert; then heights that the kernel has, the lowest not above what an average segment fills."""
    assert K.moe_packed_form(160, 16) == (0, 0) and K.moe_packed_form(1, 1) == (0, 0)
    for E in (1, 16, 1024):
        for n in (11, 95, 96, 599, 600, 5000):
            least, most = K.moe_packed_form(E * n, E)
            assert 1 <= least <= most == 4 and (least == 1 or 64 * least <= n + 63)


def test_heights_of_tiles_at_sizes_measured():
    """Sizes at which the other heights were measured 5 % behind the ones named here, or more: gated matrices that the fit of the costs once
    left out (tiles of 128 and 192 tokens took 1.2 to 2 times as long there), and plain ones in parts."""
    height = lambda M, N, K_, parts=1, gated=0: K._lib().llogos_gemm_tiles_height(M, N, K_, parts, 256, gated)
    for M in (65, 100, 160, 256, 512, 1000):
        assert height(M, 4096, 768, gated=1) == 64, M
    for M in (129, 200, 300):
        assert height(M, 9728, 1024, gated=1) in (64, 96), M
    for M, N, K_, parts, best in ((300, 3072, 3072, 8, (64,)), (300, 5120, 17408, 4, (128,)), (65, 4096, 14336, 8, (64,)), (400, 8192, 1024, 4, (64, 224)),
                                  (200, 8192, 28672, 4, (128,)), (2048, 3072, 2048, 4, (64,))):
        assert height(M, N, K_, parts) in best, (M, N, K_, parts)


def test_the_library_serves_what_it_served_before_and_is_ahead_at():
    """Prompts' products that the library made before the tiled one took all of them: at the first ones the library is ahead, in the stream
    and elsewhere; at the second ones in the stream alone; at the others the tiled product is, or a hand-written one served all along."""
    for M, N, K_ in ((700, 1536, 1536), (334, 2304, 768), (65, 1536, 1536), (100, 1024, 1024), (200, 4096, 1536), (65, 21504, 4096)):
        assert K.library_serves(M, N, K_, adds=True) and K.library_serves(M, N, K_), (M, N, K_)
        assert K.prompt_parts(M, N, K_) == 0 < K.wide_tiles_plan(M, N, K_)
    for M, N, K_ in ((334, 2048, 2048), (512, 2048, 2048), (2048, 2048, 2048), (16384, 2048, 2048), (4096, 1536, 1536), (512, 3072, 2048), (8192, 3072, 3072),
                     (8192, 4096, 4096), (16384, 1536, 8960), (2048, 4096, 4096), (3529, 4096, 4096), (2500, 21504, 4096), (256, 12288, 4096), (1200, 2304, 768)):
        assert K.library_serves(M, N, K_, adds=True) and not K.library_serves(M, N, K_), (M, N, K_)
        assert K.prompt_parts(M, N, K_, adds=True) == 0 < K.prompt_parts(M, N, K_)
    for M, N, K_ in ((200, 4096, 4096), (256, 2048, 2048), (65, 8192, 8192), (1000, 4096, 14336), (2048, 4096, 14336), (1200, 4096, 11008), (1500, 1024, 4096),
                     (3529, 2048, 8192), (600, 5120, 5120), (334, 4096, 4096), (700, 3072, 3072), (300, 512, 4096), (100, 768, 3072), (5003, 5120, 17408), (2048, 4096, 21504)):
        assert not K.library_serves(M, N, K_, adds=True) and not K.library_serves(M, N, K_), (M, N, K_)
    assert K.library_serves(1200, 10240, 28672, adds=True) and not K.library_serves(1200, 10240, 28672)


def test_where_packed_experts_serve():
    """Sizes measured on either side: packed experts were 3 to 150 % behind the row-major ones at the first, level or ahead at the others."""
    for n, E, K_ in ((0.125, 1024, 1024), (8, 1024, 512), (11, 1024, 512), (300, 1024, 512), (11, 128, 768), (64, 128, 768), (32, 256, 1024), (64, 32, 768),
                     (200, 64, 1024)):
        assert not K.moe_packed_serves(int(n * E), E, K_), (n, E, K_)
    for n, E, K_ in ((0.125, 16, 4096), (10, 256, 1024), (10, 128, 768), (8, 32, 768), (11, 128, 2048), (32, 256, 2048), (200, 8, 4096), (2000, 32, 768), (1000, 256, 1024)):
        assert K.moe_packed_serves(int(n * E), E, K_), (n, E, K_)
    assert K.pack_experts(torch.empty((1024, 64, 64), dtype=torch.bfloat16)) is None
