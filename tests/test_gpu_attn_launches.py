"""The one-launch and three-launch forms of the decode attention at the edges
of their blocks (16 value rows, 64 scored positions, 128 per scoring pass,
512 positions per value chunk, 1024 per exponential block), each
bit-identical to the oracle."""
import numpy as np
import pytest

from .test_gpu_attn import bits, check, run_attn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_head,n_kv,hd,n_ctx,n", [
    (4, 2, 128, 1040, 1024),   # the last length of the single launch; whole chunks
    (4, 2, 128, 1040, 1025),   # a tail of one position in a chunk of its own
    (4, 1, 64, 1032, 513),     # a chunk of one position
    (6, 2, 24, 520, 520),      # rows end at the allocation's end; hd below a block of 32
    (3, 3, 40, 136, 129),      # a second scoring pass of one position, a head tail of 8
    (5, 1, 120, 2600, 2559),   # five heads on one KV head, a head tail of 24, 31 tail positions
    (2, 2, 72, 1535, 1533),    # odd n_ctx: narrow value loads
    (2, 1, 192, 2056, 2049),   # keys wider than four 32-steps, a third exponential block
])
@pytest.mark.parametrize("fuse", [0, 3], ids=["three_launches", "one_launch"])
def test_block_edges(dev, oracle, option, n_head, n_kv, hd, n_ctx, n, fuse):
    """ATTN_FUSE k: one launch up to 512 k positions, else three."""
    option("ATTN_FUSE", fuse)
    rng = np.random.default_rng(hd * 4099 + n)
    q = rng.standard_normal(n_head * hd).astype(np.float32)
    k = (rng.standard_normal(n_kv * n_ctx * hd) * 2).astype(np.float16).view(np.uint16)
    v = rng.standard_normal(n_kv * hd * n_ctx).astype(np.float16).view(np.uint16)
    kq = float(np.float32(1.0 / np.sqrt(np.float32(hd))))
    want = oracle.attn_decode(q, k, v, n_head, n_kv, hd, n_ctx, n - 1, kq)
    args = (dev, q, k, v, n_head, n_kv, hd, n_ctx, n - 1, kq)
    check(run_attn(*args), want, n, f"hd={hd} n={n} fuse={fuse}")
    assert np.array_equal(bits(run_attn(*args, caller_buffers=False)[0]), bits(want[0]))


def _case(rng, n_head, n_kv, hd, n_ctx):
    q = rng.standard_normal(n_head * hd).astype(np.float32)
    k = (rng.standard_normal(n_kv * n_ctx * hd) * 2).astype(np.float16).view(np.uint16)
    v = rng.standard_normal(n_kv * hd * n_ctx).astype(np.float16).view(np.uint16)
    return q, k, v, float(np.float32(1.0 / np.sqrt(np.float32(hd))))


@pytest.mark.parametrize("hd,n_ctx,n,k_shift,v_shift", [
    (64, 1031, 1029, 0, 0),   # rows one element off the granules, a third chunk of 5
    (40, 1540, 1536, 0, 0),   # rows four elements off; whole chunks; a half block of rows
    (24, 520, 513, 0, 1),     # every row one off; one position in the last chunk
    (16, 2051, 2047, 0, 7),   # shift 7 and a tail of 31 at the end of a chunk
    (100, 600, 600, 0, 0),    # keys by 8 bytes, a tail of 4
    (128, 300, 300, 4, 0),    # keys 8 bytes off
    (36, 300, 293, 4, 3),
    (33, 200, 200, 0, 0),     # keys by elements, a tail of one
    (31, 130, 129, 0, 0),     # no whole 32-step
    (64, 200, 190, 1, 0),
    (222, 150, 150, 0, 0),    # eight 32-steps held, keys by elements, a tail of 30
    (260, 300, 290, 0, 0),
    (510, 140, 139, 0, 0),    # sixteen held
])
@pytest.mark.parametrize("fuse", [0, 3], ids=["three_launches", "one_launch"])
def test_any_alignment(dev, oracle, option, hd, n_ctx, n, k_shift, v_shift, fuse):
    """Key and value rows at element offsets that the wide loads do not take
    (k_shift, v_shift: elements past an aligned start), bit-identical."""
    option("ATTN_FUSE", fuse)
    nh, nkv = 6, 2
    q, k, v, kq = _case(np.random.default_rng(hd * 31 + n), nh, nkv, hd, n_ctx)
    want = oracle.attn_decode(q, k, v, nh, nkv, hd, n_ctx, n - 1, kq)[0]
    pad = np.full(8, 0x7e00, np.uint16)  # NaN beside the caches
    bufs = [dev.to_device(a) for a in (q, np.concatenate([pad[:k_shift], k, pad]),
                                       np.concatenate([pad[:v_shift], v, pad]), np.full(nh * hd, np.nan, np.float32))]
    try:
        dev.attn_decode_dev(bufs[0].ptr, bufs[1].ptr + 2 * k_shift, bufs[2].ptr + 2 * v_shift, nh, nkv, hd, n_ctx,
                            n - 1, kq, bufs[3].ptr)
        dev.synchronize()
        assert np.array_equal(bits(bufs[3].to_host(np.float32, nh * hd)), bits(want))
    finally:
        for b in bufs:
            b.free()


@pytest.mark.parametrize("n_head,n_kv,hd,n_ctx,n", [
    (64, 8, 128, 264, 257),    # two blocks of value rows per workgroup
    (96, 4, 96, 200, 190),     # three of six
    (128, 128, 128, 64, 40),   # four
    (40, 8, 200, 72, 70),      # five of thirteen: the last workgroup has three
    (300, 100, 24, 48, 47),    # all of a head; half a block of rows
    (64, 8, 128, 131, 131),    # value rows by elements
    (20, 4, 512, 100, 99),     # sixteen 32-steps, three of 32 blocks
])
def test_row_blocks_of_the_single_launch(dev, oracle, n_head, n_kv, hd, n_ctx, n):
    q, k, v, kq = _case(np.random.default_rng(n_head + hd), n_head, n_kv, hd, n_ctx)
    want = oracle.attn_decode(q, k, v, n_head, n_kv, hd, n_ctx, n - 1, kq)
    check(run_attn(dev, q, k, v, n_head, n_kv, hd, n_ctx, n - 1, kq), want, n, f"{n_head} heads hd={hd}")


def test_more_blocks_than_one_grid_row(dev):
    """1025 heads of 2^18 positions: 4 198 400 score blocks, past the 2^22 of
    a grid row. Equal scores give probabilities of 2^-18 exactly, so each
    head's output is its (constant) value."""
    nh, n = 1025, 1 << 18
    one = np.float16(1).view(np.uint16)
    c = np.arange(1, nh + 1).astype(np.float16)
    bufs = [dev.to_device(a) for a in (np.ones(nh, np.float32), np.full(nh * n, one, np.uint16),
                                       np.repeat(c.view(np.uint16), n), np.full(nh, np.nan, np.float32))]
    try:
        q, k, v, out = (b.ptr for b in bufs)
        dev.attn_decode_dev(q, k, v, nh, nh, 1, n, n - 1, 1.0, out)
        dev.synchronize()
        assert np.array_equal(bufs[3].to_host(np.float32, nh), c.astype(np.float32))
    finally:
        for b in bufs:
            b.free()
