"""The launches of the decode attention, on the CPU (host/fake_hip.cpp records
them and refuses grids that the runtime would)."""
import pytest

from . import fake_hip


def launches(n_head, n_kv, hd, n, n_ctx=None, k_offset=0):
    """[kernel, grid x, grid y] of a call, or the error it returns."""
    return fake_hip.run(f"""
        try:
            dev.attn_decode_dev(X, X + {k_offset}, X, {n_head}, {n_kv}, {hd}, {n_ctx or n}, {n} - 1, 0.1, X)
            result = launched()
        except sa.SihipError as e:
            result = str(e)
    """)


@pytest.mark.parametrize("n_head,n_kv,n", [
    (4096, 4096, 1 << 18),  # 2^24 blocks of 64 positions: 2^32 work items
    (4096, 4096, 1 << 20),
    (32, 1, 1 << 27),
    (8, 8, 1 << 27),
    (2, 1, 1 << 29),        # the most positions
    (1, 1, 1 << 16),
])
def test_any_number_of_blocks_has_a_grid(n_head, n_kv, n):
    got = launches(n_head, n_kv, 8, n)
    assert isinstance(got, list) and len(got) == 3, got
    (_, sx, sy), (_, ex, ey), _ = got
    scores, exps = n // 64 * n_kv * -(-n_head // n_kv // 4), n // 1024 * n_head
    assert scores <= sx * sy < scores + sx and exps <= ex * ey < exps + ex


def test_refuses_more_positions_than_it_indexes():
    assert "positions" in launches(1, 1, 8, (1 << 29) + 1)


@pytest.mark.parametrize("hd,n_ctx,k_offset,want", [
    (128, 512, 0, "4,8,true"),
    (128, 515, 0, "4,8,false"),  # value rows at any alignment, key rows still by 16 bytes
    (128, 512, 8, "4,4,true"),
    (128, 512, 2, "4,1,true"),
    (100, 512, 0, "4,4,true"),
    (66, 515, 0, "4,1,false"),
    (256, 515, 0, "8,8,false"),
    (300, 512, 0, "16,4,true"),
])
def test_keys_and_values_load_by_their_own_alignment(hd, n_ctx, k_offset, want):
    got = launches(8, 8, hd, 300, n_ctx, k_offset)
    assert [k for k, *_ in got] == [f"attn_fused_kernel<{want}>"]
    got = launches(8, 8, hd, 1300, n_ctx + 1024, k_offset)
    keys, values = want.rsplit(",", 1)
    assert [k for k, *_ in got] == [f"attn_scores_kernel<{keys}>", "attn_exp_kernel", f"attn_pv_kernel<{values}>"]


@pytest.mark.parametrize("n_head,hd,workgroups", [
    (32, 128, 256), (33, 128, 132), (64, 128, 256), (128, 128, 256), (96, 96, 192), (32, 256, 256),
    (40, 200, 200),   # 13 blocks in fives
    (300, 64, 300),   # never less than one a head
    (1, 1, 1),
])
def test_the_single_launch_fits_the_cus(n_head, hd, workgroups):
    """A workgroup takes as many 16-row blocks of values as leave one per CU."""
    got = launches(n_head, n_head, hd, 100)
    assert len(got) == 1 and got[0][1] == workgroups


@pytest.mark.parametrize("n_head,hd,kernel", [
    (32, 128, "attn_fused_kernel<4,8,true>"), (33, 128, "attn_fused_blocks_kernel<4,8,true>"),
    (16, 256, "attn_fused_kernel<8,8,true>"), (16, 512, "attn_fused_blocks_kernel<16,8,true>"),
    (300, 16, "attn_fused_kernel<4,8,true>"),  # one block of value rows a head
])
def test_one_block_of_values_has_a_kernel_of_its_own(n_head, hd, kernel):
    got = launches(n_head, n_head, hd, 100, 512)
    assert [k for k, *_ in got] == [kernel]


@pytest.mark.parametrize("n_head,n_kv,hd,n_ctx,one,three", [
    (32, 8, 128, 2048, 1200, 1201),
    (16, 8, 192, 2048, 1024, 1025),
    (16, 16, 256, 2048, 800, 801),
    (32, 8, 288, 2048, 1200, 1201),  # 576 value workgroups: two rounds of the CUs
    (32, 8, 66, 2048, 1024, 1025),
    (32, 8, 128, 2047, 1000, 1001),
    (64, 8, 128, 2047, 600, 601),
])
def test_one_launch_or_three(n_head, n_kv, hd, n_ctx, one, three):
    assert len(launches(n_head, n_kv, hd, one, n_ctx)) == 1
    assert len(launches(n_head, n_kv, hd, three, n_ctx)) == 3
