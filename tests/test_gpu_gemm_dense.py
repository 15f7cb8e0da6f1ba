"""The prompt GEMM of F16 and Q8_0-pair weights (gemmd.h) at the edges of its
tiles, each output against the oracle to the path's bar (the reference's dot,
1e-5 of the absolute terms), as single matrices and as groups, with and without
K slices, and captured."""
import numpy as np
import pytest

import siphon_amd as sa
from siphon_amd import synth

from .test_gpu_gemm import _rows
from .test_gpu_gemm_multi import _run
from .test_gpu_gemm_short import ring_cases
from .test_gpu_parity import assert_close
from .test_gpu_slices import _HipGraph, bits

pytestmark = pytest.mark.gpu

TYPES = [sa.F16, sa.Q4_0, sa.Q5_0, sa.Q8_0]

# gemmd.h: m tiles -> steps of a round
ROUND = {sa.F16: {2: 12, 3: 12, 4: 12, 5: 6, 6: 6}}
ROUND.update({t: {2: 12, 3: 12, 4: 4, 5: 4} for t in TYPES[1:]})
RING = [(t, mt) for t in TYPES for mt in ROUND[t]]


def _check(dev, oracle, mats, n_in, M, what):
    rng = np.random.default_rng(M * 131 + n_in + len(mats))
    Ws = [synth.make_weights(wt, n_out, n_in, rng) for wt, n_out in mats]
    ws = [dev.upload(wt, n_out, n_in, W) for (wt, n_out), W in zip(mats, Ws)]
    try:
        X = np.ascontiguousarray(_rows(rng, M, max(n_in, 256))[:, :n_in])
        for Y, (wt, n_out), W in zip(_run(dev, ws, X), mats, Ws):
            ref, L1 = oracle.gemm(wt, W, n_out, n_in, X)
            assert_close(Y.reshape(-1), ref.reshape(-1).astype(np.float64), L1.reshape(-1),
                         f"{what} {sa.NAMES[wt]} {n_out}x{n_in} M={M}")
    finally:
        for w in ws:
            w.free()


@pytest.mark.parametrize("wt", TYPES, ids=[sa.NAMES[t] for t in TYPES])
def test_single(dev, oracle, option, wt):
    """Small workgroups (gemmds_kernel) of one, two and three m tiles with fewer,
    as many and more steps than waves, rows past n_out and M; the longest rows of
    the Q8_0 pairs in tiles."""
    option("GEMMD_MIN_M", 9)
    for n_out, n_in, M in ((33, 128, 9), (200, 512, 17), (96, 2304, 33), (70, 1152, 49),
                           (300, 256, 600), (2080, 640, 129), (260, 4096, 400), (130, 1280, 700)):
        print(f"single {sa.NAMES[wt]} {n_out}x{n_in} M={M}", flush=True)
        _check(dev, oracle, [(wt, n_out)], n_in, M, "single")


@pytest.mark.parametrize("wt,mt", RING, ids=[f"{sa.NAMES[t]}-{mt}" for t, mt in RING])
def test_ring(dev, oracle, option, wt, mt):
    """Tiles of every m tile count at the edges of their rounds; two m blocks, the
    second of five rows, two n blocks, the second of 12. test_gemm_dispatch.py
    checks that these cases run the instance and the slices they name."""
    option("GEMMD_MIN_M", 9)
    option("RING_MT", mt)
    for steps, sbk in ring_cases(ROUND[wt][mt]):
        option("RING_SBK", sbk)
        print(f"ring {sa.NAMES[wt]} mt={mt} steps={steps} sbk={sbk}", flush=True)
        _check(dev, oracle, [(wt, 140)], 128 * steps, 16 * mt + 5, f"mt={mt} sbk={sbk}")


@pytest.mark.parametrize("wt", TYPES, ids=[sa.NAMES[t] for t in TYPES])
def test_groups(dev, oracle, wt):
    """Segments that end inside a block, in small workgroups and in tiles."""
    _check(dev, oracle, [(wt, 300), (wt, 64), (wt, 70)], 640, 20, "small group")
    _check(dev, oracle, [(wt, 1300), (wt, 130), (wt, 700)], 896, 300, "group")


@pytest.mark.parametrize("wt", [sa.F16, sa.Q8_0], ids=["F16", "Q8_0"])
@pytest.mark.parametrize("tiles", [False, True], ids=["rule", "tiles"])
def test_capture(dev, oracle, option, wt, tiles):
    """After an eager call of more rows, captured calls of fewer find their
    workspaces, by the rule (small workgroups and the older kernels) and in tiles;
    each replay gives the bits of the first."""
    if tiles:
        option("GEMMD_MIN_M", 9)
        option("RING_MT", 3)
    rng = np.random.default_rng(9)
    n_out, n_in, M = 520, 2048, 300
    W = synth.make_weights(wt, n_out, n_in, rng)
    w = dev.upload(wt, n_out, n_in, W)
    X = _rows(rng, M, n_in)
    xd = dev.to_device(X)
    yd = dev.to_device(np.zeros(M * n_out, np.float32))
    try:
        for m in (300, 230, 130, 24, 8):
            hg = _HipGraph()
            try:
                dev.gemm_dev(w, xd.ptr, M, yd.ptr, hg.stream.value)
                dev.synchronize()
                hg.begin()
                dev.gemm_dev(w, xd.ptr, m, yd.ptr, hg.stream.value)
                hg.end()
                ref, L1 = oracle.gemm(wt, W, n_out, n_in, X[:m])
                got = []
                for _ in range(3):
                    yd.fill(np.full(M * n_out, np.nan, np.float32))
                    hg.replay()
                    got.append(yd.to_host(np.float32, m * n_out))
                    dev.gemm_dev(w, xd.ptr, M, yd.ptr, hg.stream.value)
                    dev.synchronize()
                assert_close(got[0], ref.reshape(-1).astype(np.float64), L1.reshape(-1), f"M={m}")
                assert all(np.array_equal(bits(g), bits(got[0])) for g in got)
            finally:
                hg.close()
    finally:
        xd.free()
        yd.free()
        w.free()
