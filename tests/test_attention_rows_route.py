"""Which row products run in an attention's launch, asked of the library on the host (flux_attention_rows_together): nothing here
launches or needs a GPU."""
import ctypes
import random

from triton_kernels import _native as nv
from triton_kernels.kernels.attention import _may_cut_keys, takes_rows
from test_linear_plan import PTR, linear_args


def together(B, H, L, D, M, products, K, N=96, workspace=None):
    a, rows, yes = nv.AttnArgs(), nv.LinearPairArgs(), ctypes.c_int32(-1)
    for t in (a.q, a.k, a.v):
        t.ptr, t.sb, t.sh, t.sl = PTR, H * L * D, L * D, D
    a.o, a.o_sb, a.o_sh, a.o_sl = PTR, H * L * D, L * D, D
    a.B, a.H, a.L, a.D, a.sm_scale = B, H, L, D, 0.1
    for i in range(products):
        rows.product[i] = linear_args(M, N, K, in_act=nv.ACT_SILU)
    if workspace is None:
        workspace = nv.lib().flux_attention_workspace_bytes(B, H, L, D)
    assert nv.lib().flux_attention_rows_together(nv.byref(a), nv.byref(rows), workspace, nv.byref(yes)) == 0, nv.last_error()
    return yes.value == 1


def test_at_most_256_workgroups_whatever_their_length():
    """Up to 128 rows the 32-row kernel takes any number of workgroups; products beside more than 256 of them waited for the last."""
    for L in (65, 100, 128):
        assert together(1, 256, L, 128, 1, 2, 3072) and together(8, 32, L, 128, 2, 2, 3072)
        assert not together(1, 257, L, 128, 1, 2, 3072) and not together(40, 24, L, 128, 1, 2, 3072)
    assert together(1, 24, 1280, 128, 1, 2, 3072) and not together(1, 24, 1281, 128, 1, 2, 3072)
    assert not together(1, 24, 64, 128, 1, 2, 3072) and not together(1, 24, 640, 64, 1, 2, 3072)


def test_products_of_four_rows_and_24576_values():
    assert together(1, 24, 640, 128, 4, 1, 6144) and not together(1, 24, 640, 128, 4, 1, 6152)
    assert together(1, 24, 640, 128, 2, 2, 12288) and not together(1, 24, 640, 128, 3, 2, 512)
    assert not together(1, 2, 2048, 128, 1, 2, 3072) and together(1, 2, 2048, 128, 1, 2, 3072, workspace=0)   # keys in parts


def test_the_blocks_rule_names_calls_that_share_the_launch():
    """takes_rows() is asked before there are any arguments. Where it says yes the library takes the products along; where it says no
    and the library would, keys might have been cut or the rows of both products are more than the budget of one."""
    rng, yes = random.Random(4), 0
    for _ in range(5000):
        B, H, L, D = rng.randint(1, 3), rng.choice([1, 2, 4, 8, 24, 32, 48, 96]), round(2 ** rng.uniform(0, 12.3)), rng.choice([64, 128, 128])
        K = rng.choice([H * D, 8 * rng.randint(1, 2000)])
        rule, library = takes_rows(B * H, L, D, 2 * B, K), together(B, H, L, D, B, 2, K)
        assert library or not rule, (B, H, L, D, K)
        assert rule or not library or _may_cut_keys(B * H, L) or 2 * B * K * 2 > 48 * 1024, (B, H, L, D, K)
        yes += rule
    assert yes > 500
