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
