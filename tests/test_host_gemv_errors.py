"""sihip_gemv when one of its launches fails (host/fake_hip.cpp, on the CPU):
the call reports it, and returns with nothing in flight that uses the pinned
staging memory, which the next call fills."""
import pytest

from . import fake_hip


@pytest.mark.parametrize("wt", ["Q4_K", "Q8_0", "F32"])
def test_nothing_queued_after_a_failed_launch(wt):
    got = fake_hip.run(f"""
        w = upload(sa.{wt}, 256, 1024)
        x = np.zeros(1024, np.float32)
        fake.fake_reset(0)
        dev.gemv(w, x)
        result = []
        for k in range(1, fake.fake_launches() + 1):
            fake.fake_reset(k)
            try:
                dev.gemv(w, x)
                result.append(["no error", ""])
            except sa.SihipError:
                result.append(["error", fake.fake_order().decode()])
            fake.fake_reset(0)
            dev.gemv(w, x)  # and the next call runs
    """)
    assert len(got) == 3
    for k, (what, order) in enumerate(got, 1):
        assert what == "error", f"launch {k}"
        assert "l" not in order or order.endswith("s"), f"launch {k} failed: {order}"
