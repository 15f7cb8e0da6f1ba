"""Which GEMM a call takes, on the CPU (host/fake_hip.cpp records the
launches)."""
import pytest

from . import fake_hip


def gemms(options, types, n_out, n_in, Ms):
    """M -> the GEMM kernels of a call with one matrix per type."""
    got = fake_hip.run(f"""
        for name, value in {options!r}.items():
            dev.set_option(name, value)
        ws = [upload(getattr(sa, t), {n_out}, {n_in}) for t in {types!r}]
        for w in ws:
            w.prepare_gemm()
        result = []
        for M in {Ms!r}:
            fake.fake_reset(0)
            dev.gemm_multi_dev(ws, X, M, [X] * len(ws))
            result.append([k[0] for k in launched() if "quantize" not in k[0] and "convert" not in k[0]])
    """)
    return dict(zip(Ms, got))


@pytest.mark.parametrize("options,wt,want", [
    ({"GEMMKS_MAX_M": 16}, "Q5_K", {9: "gemmks", 16: "gemmks", 17: "gemmsk"}),
    ({"GEMMKS_MAX_M": 16}, "Q4_K", {9: "gemmsk", 16: "gemmsk"}),
    ({"GEMMKS_MAX_M": 16, "GEMMKS_Q4K": 1}, "Q4_K", {9: "gemmks", 16: "gemmks", 17: "gemmsk"}),
    ({"GEMMKS_MAX_M": 12}, "Q2_K", {12: "gemmks", 13: "gemmsk"}),
    ({"GEMM2S_MAX_M": 16}, "Q4_K", {9: "gemm2s_q4k", 16: "gemm2s_q4k", 17: "gemmsk"}),
    ({"GEMM2S_MAX_M": 16}, "Q5_K", {9: "gemmsk"}),
    ({"GEMM2_MIN_M": 40}, "Q4_K", {39: "gemmsk", 40: "gemm2_q4k", 200: "gemm2_q4k"}),
    ({"GEMM6_MIN_M": 20}, "Q6_K", {20: "gemm6_q6k", 64: "gemm6_q6k", 300: "gemm6_q6k"}),
    ({"GEMM6_MIN_M": 1, "GEMMSK_MAX_M": 40}, "Q6_K", {40: "gemmsk", 41: "gemm6_q6k"}),
    ({}, "Q6_K", {9: "gemmsk", 112: "gemmsk"}),
    ({}, "Q4_K", {9: "gemmsk", 200: "gemmsk", 384: "gemm2_q4k"}),
])
def test_options_place_their_kernels(options, wt, want):
    """An option that names one of the older K-quant GEMMs keeps the M it
    names on it; the built-in rule has the rest, and the newer GEMMs' own
    options go first."""
    got = gemms(options, [wt], 1024, 2048, list(want))
    assert {M: [k.split("_kernel")[0] for k in v] for M, v in got.items()} == {M: [k] for M, k in want.items()}


@pytest.mark.parametrize("wt,n_out,n_in,M,launches", [
    *[(wt, *c, 1) for wt in ("Q2_K", "Q3_K", "Q5_K", "Q6_K")
      for c in ((256, 2048, 600), (1024, 4096, 2000), (4096, 14336, 300))],
    # the planes of 1000 rows exceed the scratch: two pieces
    *[(wt, 4096, 14336, 1000, 2) for wt in ("Q2_K", "Q3_K", "Q5_K")],
])
def test_noalloc_after_a_short_prompt(wt, n_out, n_in, M, launches):
    """A weight whose first GEMM call was a short prompt holds the copy of that
    prompt's kernel alone; sihip_gemm_dev_noalloc takes it for a longer one
    rather than refuse a call that only lacks the other copy."""
    got = fake_hip.run(f"""
        w = upload(sa.{wt}, {n_out}, {n_in})
        dev.gemm_dev(w, X, 40, X)
        fake.fake_reset(0)
        dev.gemm_dev_noalloc(w, X, {M}, X)
        result = [k[0] for k in launched() if "quantize" not in k[0]]
    """)
    assert len(got) == launches and all(k.startswith(("gemmsk", "gemmx", "gemm6", "gemm_kq")) for k in got), got


@pytest.mark.parametrize("types,n_out,n_in,M", [
    (["Q5_K"], 4096, 14336, 2048), (["Q5_K"], 14336, 4096, 200), (["Q2_K"], 4096, 14336, 350),
    (["Q4_K"], 14336, 4096, 350), (["Q3_K"] * 2, 27648, 512, 1568), (["Q5_K"] * 2, 4096, 5120, 187),
    (["Q4_K"], 4096, 4096, 37), (["Q6_K"], 4096, 4096, 300),
])
def test_a_capture_takes_the_kernel_of_the_call_before(types, n_out, n_in, M):
    """The first call builds the copy of its own kernel alone, which two GEMMs
    share: a captured repetition launches what the call did."""
    eager, captured, noalloc = fake_hip.run(f"""
        ws = [upload(getattr(sa, t), {n_out}, {n_in}) for t in {types!r}]
        call = lambda: dev.gemm_multi_dev(ws, X, {M}, [X] * len(ws), 1)
        call()
        result = []
        for capture in (0, 1):
            fake.fake_reset(0)
            fake.fake_capture(capture)
            call()
            result.append(launched())
        fake.fake_reset(0)
        if {n_in * M} < 1 << 24:  # (the planes fit the scratch)
            dev.gemm_dev_noalloc(ws[0], X, {M}, X, 1)
        result.append(launched())
    """)
    assert eager == captured
    if len(types) == 1 and noalloc:
        assert noalloc[-1][0].split("<")[0] == eager[-1][0].split("<")[0]


@pytest.mark.parametrize("types,M", [(["Q4_K", "Q6_K"], 200), (["Q6_K", "Q6_K", "Q6_K"], 130), (["Q4_K", "Q4_K"], 200)])
def test_a_captured_group_after_calls_of_its_matrices(types, M):
    """Calls of one matrix each leave some with the newer kernels' copy alone and
    some with their plan's: a captured call of the group, whose launch would
    need one copy of all, runs each matrix on the copy it has."""
    calls, group = fake_hip.run(f"""
        ws = [upload(getattr(sa, t), 14336 if i else 1024, 4096) for i, t in enumerate({types!r})]
        result = [[]]
        for w in ws:
            dev.gemm_dev(w, X, {M}, X, 1)
            fake.fake_reset(0)
            dev.gemm_dev(w, X, {M}, X, 1)
            result[0] += launched()
        fake.fake_reset(0)
        fake.fake_capture(1)
        dev.gemm_multi_dev(ws, X, {M}, [X] * len(ws), 1)
        result.append(launched())
    """)
    assert group == calls and len({k.split("_kernel")[0] for k, *_ in calls if "_kernel" in k}) > 1


@pytest.mark.parametrize("n_out,M,waves,grid", [
    (4096, 48, 8, 256), (4128, 48, 4, 136), (5120, 9, 4, 160), (2048, 96, 8, 256), (2080, 96, 4, 144),
])
def test_short_prompts_fit_one_round(n_out, M, waves, grid):
    """Workgroups of eight waves only where each has a CU of its own."""
    got = fake_hip.run(f"""
        w = upload(sa.Q4_K, {n_out}, 1024)
        w.prepare_gemm()
        fake.fake_reset(0)
        dev.set_option("GEMMSK_MAX_M", 1000)
        dev.gemm_dev(w, X, {M}, X)
        result = launched()[-1]
    """)
    assert got[0].startswith("gemmsk_kernel") and got[0].endswith(f",{waves}>") and got[1] == grid, got


@pytest.mark.parametrize("wt,n_out,n_in,want", [
    # timed faster there by 5% and more
    ("Q6_K", 14336, 4096, {64: "gemmsk", 112: "gemm6_q6k", 256: "gemm6_q6k", 512: "gemm6_q6k"}),
    ("Q6_K", 4096, 4096, {96: "gemmsk", 300: "gemm6_q6k"}),
    ("Q4_K", 14336, 4096, {64: "gemmsk", 112: "gemm_kq", 224: "gemm_kq", 300: "gemmx"}),
    ("Q4_K", 4096, 14336, {16: "gemm2s_q4k", 32: "gemmsk", 340: "gemmx"}),
    ("Q5_K", 14336, 4096, {112: "gemm_kq", 144: "gemmsk", 300: "gemmx"}),
    ("Q2_K", 32000, 2048, {48: "gemmsk", 64: "gemm_kq"}),
    ("Q2_K", 1024, 4096, {9: "gemmsk", 300: "gemmsk"}),
    ("Q8_0", 256, 2048, {128: "gemmq", 200: "gemmq"}),
    ("Q8_0", 4096, 4096, {128: "gemmq", 144: "gemmd", 600: "gemmq"}),
    ("Q4_0", 1024, 4096, {129: "gemmq", 383: "gemmq"}),
    ("Q5_0", 4096, 4096, {160: "gemmd", 512: "gemmq"}),
    ("F16", 896, 896, {200: "gemmh_f16"}),
    ("F16", 5632, 2048, {144: "gemmd", 300: "gemmd"}),
    ("F16", 27648, 5120, {256: "gemmh_f16"}),
])
def test_single_matrices(wt, n_out, n_in, want):
    """A call of one matrix takes the kernel that is the faster for it."""
    got = gemms({}, [wt], n_out, n_in, list(want))
    assert {M: v[0].split("_kernel")[0] for M, v in got.items()} == want


def test_a_group_keeps_the_newer_kernels():
    got = gemms({}, ["Q6_K", "Q6_K"], 14336, 4096, [112, 256])
    assert {M: v[0].split("_kernel")[0] for M, v in got.items()} == {112: "gemmsk", 256: "gemmx"}
    got = gemms({}, ["Q8_0"] * 3, 256, 2048, [17, 200])
    assert all(v[0].startswith("gemmd") and len(v) == 1 for v in got.values())


def _ring_runs():
    """What test_ring of test_gpu_gemm_short.py and test_gpu_gemm_dense.py run:
    [type, m tiles, steps, slice length, options, elements per step]."""
    import siphon_amd as sa

    from . import test_gpu_gemm_dense as dense
    from . import test_gpu_gemm_short as short
    kq = {"GEMMSK_MAX_M": 0, "GEMMX_MIN_M": 9}
    for t in short.KQ:
        for mt, u in short.ROUND.items():
            yield from ((sa.NAMES[t], mt, *c, kq, 256) for c in short.ring_cases(u))
    for t, mt in dense.RING:
        yield from ((sa.NAMES[t], mt, *c, {"GEMMD_MIN_M": 9}, 128) for c in short.ring_cases(dense.ROUND[t][mt]))


def test_ring_cases_run_what_they_name():
    runs = list(_ring_runs())
    got = fake_hip.run(f"""
        result = []
        for t, mt, steps, sbk, options, size in {runs!r}:
            for name, value in [*options.items(), ("RING_MT", mt), ("RING_SBK", sbk)]:
                dev.set_option(name, value)
            w = upload(getattr(sa, t), 140, size * steps)
            w.prepare_gemm()
            fake.fake_reset(0)
            dev.gemm_dev(w, X, 16 * mt + 5, X)
            result.append([sa.TYPES[t], *launched()[-1]])
            w.free()
    """)
    for (t, mt, steps, sbk, _, size), (number, kernel, grid, _) in zip(runs, got):
        name = f"gemmx_kernel<{number},{number},{mt}>" if size == 256 else f"gemmd_kernel<{number},{mt}>"
        slices = -(-steps // sbk) if sbk else 1
        assert (kernel, grid) == (name, 8 * 2 * slices), (t, mt, steps, sbk)
