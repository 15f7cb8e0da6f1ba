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
    """Rings of one and two super-blocks ahead at fewer, as many and more
    super-blocks than slots, K slices (few rows, long rows), every m tile
    count of the plan, and a row block past n_out in the last n block."""
    option("GEMMSK_MAX_M", 0)
    option("GEMMX_MIN_M", 9)
    for n_out, n_in, M in ((33, 256, 17), (200, 512, 40), (130, 768, 64), (128, 8192, 33),
                           (96, 1792, 80), (160, 2304, 96), (300, 1280, 129)):
        print(f"longer {sa.NAMES[wt]} {n_out}x{n_in} M={M}", flush=True)
        _check(dev, oracle, [(wt, n_out)], n_in, M, "ring")


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
