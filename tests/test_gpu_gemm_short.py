"""The K-quant GEMMs of short prompts (gemmsk.h: waves of a workgroup split the
super-blocks) and longer ones (gemmx.h: activation records and weights ahead
in a ring) at the edges of their tiles, each against the oracle to the path's
bar (the reference's dot, 1e-5 of the absolute terms)."""
import numpy as np
import pytest

import siphon_amd as sa
from siphon_amd import synth

from .test_gpu_gemm import _rows
from .test_gpu_gemm_multi import _run
from .test_gpu_parity import assert_close
from .test_gpu_slices import _HipGraph, bits

pytestmark = pytest.mark.gpu

KQ = [sa.Q2_K, sa.Q3_K, sa.Q4_K, sa.Q5_K, sa.Q6_K]

# gemmx.h: m tiles -> steps of a round (ring slots times super-blocks of weights
# in registers)
ROUND = {2: 6, 3: 6, 4: 3, 5: 3, 6: 2, 8: 2}


def ring_cases(u):
    """(steps, K-slice length or 0) at the edges of a round of u steps: fewer
    steps than the ring holds, one short of a round (the longest partial one), a
    round, one and u + 1 more; slices of a round and one with a ragged last one,
    and of two."""
    return [(1, 0), (2, 0), (u - 1, 0), (u, 0), (u + 1, 0), (2 * u + 1, 0), (2 * u + 1, u + 1), (5, 2)]


def _check(dev, oracle, mats, n_in, M, what, seed=0):
    rng = np.random.default_rng(M * 131 + n_in + seed)
    Ws = [synth.make_weights(wt, n_out, n_in, rng) for wt, n_out in mats]
    ws = [dev.upload(wt, n_out, n_in, W) for (wt, n_out), W in zip(mats, Ws)]
    try:
        X = _rows(rng, M, n_in)
        for Y, (wt, n_out), W in zip(_run(dev, ws, X), mats, Ws):
            ref, L1 = oracle.gemm(wt, W, n_out, n_in, X)
            assert_close(Y.reshape(-1), ref.reshape(-1).astype(np.float64), L1.reshape(-1),
                         f"{what} {sa.NAMES[wt]} {n_out}x{n_in} M={M}")
    finally:
        for w in ws:
            w.free()


@pytest.mark.parametrize("wt", KQ, ids=[sa.NAMES[t] for t in KQ])
@pytest.mark.parametrize("waves", [4, 8])
def test_short_prompts(dev, oracle, option, wt, waves):
    """GEMMS_WAVES 4: 32 weight rows and four waves per workgroup, 8: 16 and
    eight. One super-block (most waves idle), three, and nine; rows past
    n_out in the last block, one, two and three m tiles, a second m block."""
    option("GEMMSK_MAX_M", 1000)
    option("GEMMS_WAVES", waves)
    for n_out, n_in, M in ((33, 256, 9), (16, 768, 17), (200, 2304, 48), (64, 1024, 49)):
        print(f"short {sa.NAMES[wt]} {n_out}x{n_in} M={M} waves={waves}", flush=True)
        _check(dev, oracle, [(wt, n_out)], n_in, M, f"waves={waves}")


@pytest.mark.parametrize("wt", KQ, ids=[sa.NAMES[t] for t in KQ])
def test_longer_prompts(dev, oracle, option, wt):
    """The plans of small products (32-row m blocks) with fewer, as many and more
    super-blocks than slots, K slices (few rows, long rows), and a row block past
    n_out in the last n block."""
    option("GEMMSK_MAX_M", 0)
    option("GEMMX_MIN_M", 9)
    for n_out, n_in, M in ((33, 256, 17), (200, 512, 40), (130, 768, 64), (128, 8192, 33),
                           (96, 1792, 80), (160, 2304, 96), (300, 1280, 129)):
        print(f"longer {sa.NAMES[wt]} {n_out}x{n_in} M={M}", flush=True)
        _check(dev, oracle, [(wt, n_out)], n_in, M, "ring")


@pytest.mark.parametrize("wt", KQ, ids=[sa.NAMES[t] for t in KQ])
@pytest.mark.parametrize("mt", list(ROUND))
def test_ring(dev, oracle, option, wt, mt):
    """Every m tile count at the edges of its rounds; two m blocks, the second of
    five rows, two n blocks, the second of 12. test_gemm_dispatch.py checks that
    these cases run the instance and the slices they name."""
    option("GEMMSK_MAX_M", 0)
    option("GEMMX_MIN_M", 9)
    option("RING_MT", mt)
    for steps, sbk in ring_cases(ROUND[mt]):
        option("RING_SBK", sbk)
        print(f"ring {sa.NAMES[wt]} mt={mt} steps={steps} sbk={sbk}", flush=True)
        _check(dev, oracle, [(wt, 140)], 256 * steps, 16 * mt + 5, f"mt={mt} sbk={sbk}", steps)


@pytest.mark.parametrize("short", [1000, 0], ids=["short", "longer"])
def test_groups(dev, oracle, option, short):
    """A pair of formats with an instance, and three formats (a launch each)."""
    option("GEMMSK_MAX_M", short)
    option("GEMMX_MIN_M", 9)
    _check(dev, oracle, [(sa.Q4_K, 300), (sa.Q4_K, 64), (sa.Q6_K, 100)], 1024, 37, "pair")
    _check(dev, oracle, [(sa.Q5_K, 130), (sa.Q3_K, 64), (sa.Q6_K, 40)], 1024, 70, "three")


def test_capture_takes_the_copy_that_exists(dev, oracle, option):
    """Under capture a missing weight copy cannot be built: a weight that an
    M = 40 call has prepared runs M = 600 on that copy, and one that only the
    older kernels have prepared runs M = 40 on theirs; each replay gives the
    bits of the first."""
    rng = np.random.default_rng(5)
    n_out, n_in, M = 160, 1024, 600
    W = synth.make_weights(sa.Q4_K, n_out, n_in, rng)
    X = _rows(rng, M, n_in)
    for older, then in ((False, 600), (True, 40)):
        w, other = (dev.upload(sa.Q4_K, n_out, n_in, W) for _ in range(2))
        hg = _HipGraph()
        xd = dev.to_device(X)
        yd = dev.to_device(np.zeros(M * n_out, np.float32))
        try:
            for v in (0, -1):
                if older == (v == 0):
                    option("GEMMSK_MAX_M", v)
                    option("GEMMX_MIN_M", v)
                    dev.gemm_dev(w, xd.ptr, 40, yd.ptr, hg.stream.value)
            option("GEMMSK_MAX_M", -1)
            option("GEMMX_MIN_M", -1)
            dev.gemm_dev(other, xd.ptr, M, yd.ptr, hg.stream.value)  # grows the workspaces
            dev.synchronize()
            hg.begin()
            dev.gemm_dev(w, xd.ptr, then, yd.ptr, hg.stream.value)
            hg.end()
            ref, L1 = oracle.gemm(sa.Q4_K, W, n_out, n_in, X[:then])
            got = []
            for _ in range(3):
                yd.fill(np.full(M * n_out, np.nan, np.float32))
                hg.replay()
                got.append(yd.to_host(np.float32, then * n_out))
                dev.gemm_dev(other, xd.ptr, M, yd.ptr, hg.stream.value)
                dev.synchronize()
            assert_close(got[0], ref.reshape(-1).astype(np.float64), L1.reshape(-1), f"M={then}")
            assert all(np.array_equal(bits(g), bits(got[0])) for g in got)
        finally:
            hg.close()
            xd.free()
            yd.free()
            w.free()
            other.free()


@pytest.mark.parametrize("wt,n_in", [(sa.Q5_K, 2048), (sa.F16, 1024)], ids=["Q5_K", "F16"])
def test_capture_without_room_for_slices(wt, n_in):
    """A captured call whose partial sums were never allocated runs without K
    slices: the bits of the eager unsliced call."""
    rng = np.random.default_rng(7)
    n_out, M = 140, 40
    dev = sa.Device(0)  # its workspaces hold what the calls below ask for
    hg = _HipGraph()
    bufs, w = [], None
    try:
        for name, v in (("GEMMSK_MAX_M", 0), ("GEMMX_MIN_M", 9), ("GEMMD_MIN_M", 9), ("RING_MT", 2), ("RING_SBK", 0)):
            dev.set_option(name, v)
        w = dev.upload(wt, n_out, n_in, synth.make_weights(wt, n_out, n_in, rng))
        bufs = [dev.to_device(_rows(rng, M, n_in)), *(dev.to_device(np.full(M * n_out, np.nan, np.float32)) for _ in range(2))]
        x, eager, got = (b.ptr for b in bufs)
        dev.gemm_dev(w, x, M, eager, hg.stream.value)
        dev.synchronize()
        dev.set_option("RING_SBK", 2)
        hg.begin()
        dev.gemm_dev(w, x, M, got, hg.stream.value)
        hg.end()
        want = bits(bufs[1].to_host(np.float32, M * n_out))
        for _ in range(3):
            bufs[2].fill(np.full(M * n_out, np.nan, np.float32))
            hg.replay()
            assert np.array_equal(bits(bufs[2].to_host(np.float32, M * n_out)), want)
    finally:
        hg.close()
        for b in bufs:
            b.free()
        if w:
            w.free()
        dev.close()
