"""Host-vector matvec (sihip_gemv) through the pinned staging memory and past
its size: the bits of the device-pointer call, also back to back with changing
vectors, fewer rows than the weight has, and lengths that are no multiple of
four floats."""
import time

import numpy as np
import pytest

import siphon_amd as sa
from siphon_amd import synth

from .test_gpu_streams import _Streams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wt,n_out,n_in", [(sa.Q4_K, 257, 1024), (sa.Q8_0, 33, 32),
                                           (sa.Q6_K, 1030, 256), (sa.F16, 70000, 32),
                                           (sa.Q4_0, 5, 65568)])
def test_gemv_host_bits(dev, wt, n_out, n_in):
    rng = np.random.default_rng(n_out)
    W = synth.make_weights(wt, n_out, n_in, rng)
    w = dev.upload(wt, n_out, n_in, W)
    yd = dev.to_device(np.zeros(n_out, np.float32))
    try:
        for n in (n_out, max(1, n_out - 3), n_out):
            x = rng.standard_normal(n_in).astype(np.float32)
            xd = dev.to_device(x)
            got = dev.gemv(w, x, n) if n != n_out else dev.gemv(w, x)
            dev.gemv_dev(w, xd.ptr, yd.ptr, n_out)
            dev.synchronize()
            want = yd.to_host(np.float32, n_out)[:n]
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
            xd.free()
    finally:
        yd.free()
        w.free()


def test_gemv_host_behind_a_long_queue(dev):
    """A call that has to wait, past the time in which it polls the completion
    word (300 us): a sliced weight busy on another stream, whose launches this one
    follows. Then again at once with another vector."""
    rng = np.random.default_rng(11)
    wt, n_out, n_in = sa.Q6_K, 4096, 14336
    w = dev.upload(wt, n_out, n_in, synth.make_weights(wt, n_out, n_in, rng))
    ss = _Streams()
    xs = [rng.standard_normal(n_in).astype(np.float32) for _ in range(2)]
    xd, yd = dev.to_device(xs[0]), dev.to_device(np.zeros(n_out, np.float32))
    try:
        want = [dev.gemv(w, x) for x in xs]
        s = ss.create()
        dev.gemv_dev(w, xd.ptr, yd.ptr, n_out, s)
        dev.gemv(w, xs[1])  # the switch of streams drains the device once; events order later ones
        for _ in range(600):  # some 12 us each
            dev.gemv_dev(w, xd.ptr, yd.ptr, n_out, s)
        t0 = time.perf_counter()
        got = dev.gemv(w, xs[1])
        waited = time.perf_counter() - t0
        assert np.array_equal(got.view(np.uint32), want[1].view(np.uint32))
        assert np.array_equal(dev.gemv(w, xs[0]).view(np.uint32), want[0].view(np.uint32))
        assert waited > 300e-6, f"the queue was {waited * 1e6:.0f} us long"
        ss.sync(s)
    finally:
        ss.close()
        for b in (xd, yd):
            b.free()
        w.free()
