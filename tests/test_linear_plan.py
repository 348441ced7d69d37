"""Which kernel a linear call takes, asked of the library on the host (flux_linear_plan_of): nothing here
launches or needs a GPU."""
import ctypes
import random

import pytest

from triton_kernels import _native as nv
from triton_kernels.kernels.linear import _may_cut_k

NOTHING, SCALAR, ROWS, SQUARE, RECT, EIGHT_WAVES = range(6)
PTR = 1 << 20   # stands for an aligned device address; the query reads the arguments only
NO_LIMIT = 2 ** 62


def linear_args(M, N, K, **fields):
    a = nv.LinearArgs()
    a.A = a.W = a.Y = PTR
    a.M, a.N, a.K, a.lda, a.ldw, a.ldy, a.split_n = M, N, K, K, K, N, N
    for name, value in fields.items():
        setattr(a, name, value)
    return a


def qk_args(B, L, heads, mlp, K=None, **fields):
    """linear1 of a single-stream block: q, k and v heads of 128 and the mlp columns behind them."""
    f = nv.LinearQKFusion()
    f.q_out = f.k_out = f.q_scale = f.k_scale = f.pe = PTR
    f.heads, f.seq_len, f.out_len = heads, L, L
    qkv = 3 * heads * 128
    split = dict(Y2=PTR, ldy=qkv, ldy2=qkv + mlp, split_n=qkv, act=nv.ACT_GELU_TANH, act_begin=qkv) if mlp else dict(ldy=qkv, act_begin=qkv)
    a = linear_args(B * L, qkv + mlp, K or heads * 128, **{**split, **fields})
    a.qk = ctypes.pointer(f)
    return a


def plan_of(first, second=None, workspace=NO_LIMIT):
    p = nv.LinearPlan()
    rc = nv.lib().flux_linear_plan_of(nv.byref(first), nv.byref(second) if second is not None else None, workspace, nv.byref(p))
    assert rc == 0, nv.last_error()
    return p


def test_plan_names_the_route():
    assert plan_of(linear_args(0, 8, 8)).family == NOTHING
    assert plan_of(linear_args(4, 8, 8)).family == ROWS
    assert plan_of(linear_args(4, 8, 7)).family == SCALAR
    assert plan_of(linear_args(9, 8, 8)).family in (SQUARE, RECT, EIGHT_WAVES)
    assert plan_of(linear_args(64, 96, 128), linear_args(32, 96, 128)).products == 2
    assert plan_of(linear_args(64, 96, 128), linear_args(32, 104, 128)).products == 1
    bad = nv.LinearPlan()
    assert nv.lib().flux_linear_plan_of(nv.byref(linear_args(9, 8, 8, lda=4)), None, 0, nv.byref(bad)) == -2


@pytest.mark.parametrize("far", ["", "ldy", "ldy2", "both"])
def test_qk_columns_take_a_tile_whose_waves_hold_whole_heads(far):
    """The q/k epilogue exists where a wave owns 128 columns: tiles of 256 columns. Any admitted fused call
    must get one, also where a row stride is too long for 32-bit offsets inside a tile (3.73 million
    elements of 2 bytes times 288 rows)."""
    rng = random.Random(len(far))
    for _ in range(300):
        B, L, heads = rng.randint(1, 3), rng.randint(256, 4700), rng.choice([1, 2, 8, 24])
        mlp = 256 * rng.choice([0, 1, 2 * heads]) + (128 * heads) % 256   # columns in multiples of 256
        fields = {}
        if far in ("ldy", "both"):
            fields["ldy"] = 3_800_000 // 8 * 8
        if far in ("ldy2", "both") and mlp:
            fields["ldy2"] = 4_000_000
        p = plan_of(qk_args(B, L, heads, mlp, **fields))
        assert p.tile_n == 256 and p.family in (SQUARE, RECT, EIGHT_WAVES), (B, L, heads, mlp, p.family, p.tile_m, p.tile_n)


@pytest.mark.parametrize("stride", ["ldy", "ldy2", "ldresid"])
@pytest.mark.parametrize("M", [40, 320, 700, 2700])
def test_rows_too_far_apart_for_32_bit_offsets_take_the_checked_epilogue(M, stride):
    """The branch-free epilogue of the rectangular and eight-wave tiles addresses the rows of a tile by 32-bit
    byte offsets; the checked one does not."""
    fields = dict(gate=PTR, resid=PTR, rows_per_batch=M, ldresid=3072)
    if stride == "ldy2":
        fields.update(Y2=PTR, split_n=1536, ldy2=1536)
    assert not plan_of(linear_args(M, 3072, 3072, **fields)).checked
    assert plan_of(linear_args(M, 3072, 3072, **{**fields, stride: 160_000_000})).checked


@pytest.mark.parametrize("M", [9, 64, 128, 300, 512, 1024])
@pytest.mark.parametrize("N,fields", [
    (100, {}), (1001, {}), (3073, {}),                                                    # columns no multiple of 8
    (3072, dict(Y2=PTR, split_n=1000, ldy=1000, ldy2=2072)),                              # a split no tile has at a wave's edge
    (3072, dict(act=nv.ACT_GELU_TANH, act_begin=1000)), (3072, dict(Y=PTR + 2)),
    (3072, dict(act=nv.ACT_GELU_TANH, gate=PTR, resid=PTR, rows_per_batch=1 << 20, ldresid=3072)),
])
def test_calls_outside_the_branch_free_form_still_get_small_tiles(M, N, fields):
    """256-wide tiles leave almost the whole GPU idle at these sizes, and 128-wide ones walk K with too few
    loads in flight: 64 x 3072 x 3072 with 1000 columns in the first output takes 12 us on eight-wave tiles and 63 us
    on the 256-wide one, 300 x 1001 x 3072 13 us and 30 us on 128-wide ones."""
    p = plan_of(linear_args(M, N, 3072, **fields))
    assert p.family == EIGHT_WAVES and p.checked, (p.family, p.tile_m, p.tile_n)
    pair = plan_of(linear_args(M, N, 3072, **fields), linear_args(M // 3 + 9, N, 3072, **fields))
    assert pair.products == 2 and pair.family == EIGHT_WAVES and pair.checked


def test_a_nearly_empty_last_round_is_cut_off():
    """1500 x 12289 outputs are 294 tiles of 256 x 256, a second round of 38 of them: five tile rows are one round,
    and the 220 rows behind them go to 128-wide tiles. Only where one batch element's rows stay together."""
    p = plan_of(linear_args(1500, 12289, 3072))
    assert (p.family, p.tile_m, p.head_rows) == (SQUARE, 256, 1280)
    gated = dict(gate=PTR, resid=PTR, ldresid=12289)
    assert plan_of(linear_args(1500, 12289, 3072, rows_per_batch=256, **gated)).head_rows == 1280
    assert plan_of(linear_args(1500, 12289, 3072, rows_per_batch=1500, **gated)).head_rows == 0


@pytest.mark.parametrize("rows,family,tile_m", [
    (260, EIGHT_WAVES, 128), (384, EIGHT_WAVES, 128), (513, RECT, 224), (640, RECT, 224), (960, RECT, 224), (1153, RECT, 224), (1344, RECT, 224),
    (1600, RECT, 224), (1760, RECT, 224), (1920, RECT, 224), (2049, SQUARE, 256), (2112, SQUARE, 256), (2560, RECT, 224), (3329, RECT, 224),
    (4096, SQUARE, 256), (4608, SQUARE, 256)])
def test_qk_projection_takes_the_tile_that_is_fastest_for_it(rows, family, tile_m):
    """The tile measured fastest for the single block's fused projection at each row count. Eight-wave tiles are the
    best for the plain product up to 2100 rows, but their only shape with whole heads per wave is slow: 1920 rows 257
    us against 215 on 224 x 256 tiles, 2049 rows 290 against 237 on 256 x 256."""
    p = plan_of(qk_args(1, rows, 24, 12288))
    assert (p.family, p.tile_m, p.tile_n) == (family, tile_m, 256)


@pytest.mark.parametrize("M,N,K,tile", [
    (9, 12288, 3072, (64, 64)), (64, 12288, 3072, (64, 64)), (48, 21504, 3072, (64, 96)), (81, 21504, 3072, (96, 96)), (28, 18432, 3072, (64, 96)),
    (335, 9216, 3072, (160, 128))])
def test_tiles_of_like_price(M, N, K, tile):
    """Few rows of wide products wait for the weights whatever the tile: those took the first shape of the table that
    was fast enough (64 x 12288 x 3072 25 us, 48 x 21504 39) and take the one that does least beside (20 and 27)."""
    p = plan_of(linear_args(M, N, K))
    assert (p.family, p.tile_m, p.tile_n, p.splits) == (EIGHT_WAVES, *tile, 1)


def test_no_workspace_is_needed_where_the_question_is_not_asked():
    rng, cut = random.Random(5), 0
    for _ in range(6000):
        M, N = (round(2 ** rng.uniform(*r)) for r in ((0, 14), (3, 15)))
        K = rng.choice([64, 1024, 2048, 3072, 3136, 4096, 4608, 6144, 9216, 12288, 15360])
        a = linear_args(M, N, K)
        need = nv.lib().flux_linear_workspace_bytes(nv.byref(a))
        assert need == 0 or _may_cut_k(M, N, K), (M, N, K, need)
        cut += need > 0
        other = round(2 ** rng.uniform(0, 12))
        pair = nv.LinearPairArgs()
        pair.product[0], pair.product[1] = a, linear_args(other, N, K)
        need = nv.lib().flux_linear_pair_workspace_bytes(nv.byref(pair))
        assert need == 0 or _may_cut_k(M + other, N, K), (M, other, N, K, need)
    assert cut > 100


def test_k_is_cut_only_for_a_gain_above_what_it_costs_the_host():
    assert plan_of(linear_args(64, 3072, 3072)).splits == 1      # 2 us of the GPU for 6 us of the host
    assert plan_of(linear_args(320, 3072, 15360)).splits > 1     # 30 us
    assert plan_of(linear_args(320, 3072, 15360), workspace=0).splits == 1


@pytest.mark.parametrize("ldw", [3_728_264, 3_728_272, 4_000_000, 4_194_296])
def test_weight_rows_of_a_tile_stay_within_31_bit_offsets(ldw):
    """A tile reaches its weight rows with byte offsets below 2^31, where the offset that stands for "out of range" begins:
    288 rows of them up to 3728269 values apart, 256 up to 4194303."""
    rng, widest = random.Random(ldw), 0
    shapes = [(57344, 288, 1032), (1580, 8312, 1032)]
    shapes += [(round(2 ** rng.uniform(8, 14)), 8 * round(2 ** rng.uniform(4, 11)), 8 * rng.randint(128, 600)) for _ in range(3000)]
    for M, N, K in shapes:
        p = plan_of(linear_args(M, N, K, ldw=ldw))
        assert p.tile_n * ldw * 2 < 2 ** 31, (M, N, K, p.tile_m, p.tile_n)
        widest = max(widest, p.tile_n)
    assert widest == (288 if ldw == 3_728_264 else 256)


def test_calls_beside_another_stream_keep_their_eight_wave_tiles():
    """A call that shares the GPU takes square tiles where a rectangle of up to 192 columns would be the best. The wider ones
    stand in for eight-wave tiles as well as for square ones (6100 x 9216 x 3072: 272 us on eight-wave tiles, 292 on square), so
    they are no reason to leave those."""
    assert (lambda p: (p.family, p.tile_m, p.tile_n))(plan_of(linear_args(6100, 9216, 3072))) == (RECT, 256, 224)
    p = plan_of(linear_args(6100, 9216, 3072, flags=nv.LINEAR_SHARED_GPU))
    assert p.family == EIGHT_WAVES
    p = plan_of(linear_args(4608, 12288, 3072, flags=nv.LINEAR_SHARED_GPU))
    assert (p.family, p.tile_m, p.tile_n) == (SQUARE, 256, 256)
    rng = random.Random(3)
    for _ in range(2000):
        M, N, K = round(2 ** rng.uniform(8, 14)), 8 * round(2 ** rng.uniform(7, 11.5)), 64 * rng.randint(16, 240)
        assert plan_of(linear_args(M, N, K, flags=nv.LINEAR_SHARED_GPU)).family != RECT


@pytest.mark.parametrize("rows,N,K,tile", [
    # what HBM feeds a CU counts: one row of tiles, two products of few rows
    ((64,), 3072, 15360, (64, 64, 4)), ((96,), 3072, 15360, (64, 96, 4)), ((90,), 12288, 4096, (64, 96, 1)), ((256, 64), 3072, 12288, (128, 192, 5)), ((570, 20), 3072, 12288, (192, 192, 4)),
    # and does not: another tile was up to a third slower
    ((97,), 3072, 15360, (64, 96, 4)), ((180,), 3072, 15360, (96, 96, 4)), ((129,), 12288, 4096, (96, 96, 1)), ((97,), 8192, 8192, (64, 64, 1)),
    ((168, 488), 9216, 3072, (256, 128, 1)), ((65, 35), 16384, 4096, (160, 128, 1)), ((258, 498), 6144, 6144, (192, 128, 1)), ((150, 10), 4096, 16384, (64, 64, 1)),
    ((713, 279), 16384, 4096, (192, 128, 1))])
def test_tiles_of_few_rows_and_weights_from_hbm(rows, N, K, tile):
    """The faster one of the tiles that the prices alone and the bound by HBM come to, weights from HBM."""
    p = plan_of(*(linear_args(M, N, K) for M in rows))
    assert (p.products, p.tile_m, p.tile_n, p.splits) == (len(rows), *tile)


@pytest.mark.parametrize("rows,pays", [(256, 0), (320, 0), (384, 1), (448, 0), (512, 0), (640, 1), (704, 1), (896, 0), (1024, 0), (1280, 1), (1700, 1), (4608, 1), (13008, 1)])
def test_qk_epilogue_where_it_pays(rows, pays):
    """Two rounds of the epilogue's tiles at most: on the side that was measured faster; beyond: always."""
    assert nv.lib().flux_linear_qk_pays(rows, 21504, 3072, 24) == pays


def test_qk_epilogue_rule_takes_any_size():
    for sizes in ((0, 21504, 3072, 24), (320, 0, 3072, 24), (320, 21504, 0, 24), (320, 21504, 3072, 0), (320, 512, 3072, 3), (1 << 40, 21504, 3072, 24), (320, 21504, 3072, 1 << 60), (-1, -1, -1, -1)):
        assert nv.lib().flux_linear_qk_pays(*sizes) == 1
    for rows in (1, 255, 2047, 1 << 30):
        for n, k, heads in ((256, 8, 1), (768, 64, 2), (9216, 3072, 24), (21504, 1 << 20, 24)):
            assert nv.lib().flux_linear_qk_pays(rows, n, k, heads) in (0, 1)
