"""The order of copies, LDS reads and barriers in the compiled ring-buffered
prompt GEMMs (pipeline_asm.py states it), on the CPU: a step that broke it
would read a slot while it is written, which a GPU run shows only by chance."""
from concurrent.futures import ThreadPoolExecutor

import pytest

from . import pipeline_asm

# (instance, ring slots): a ring of two and of more, weights as deep as the
# ring and shallower, both segments of a pair, each record size class. Types:
# F16 1, Q5_0 6, Q8_0 8, Q2_K 10, Q4_K 12, Q5_K 13, Q6_K 14
INSTANCES = [
    ("gemmx_kernel<10, 10, 2>(GXArgs)", 3),
    ("gemmx_kernel<12, 14, 3>(GXArgs)", 3),
    ("gemmx_kernel<13, 13, 5>(GXArgs)", 3),
    ("gemmx_kernel<12, 12, 8>(GXArgs)", 2),
    ("gemmd_kernel<1, 2>(GDArgs)", 4),
    ("gemmd_kernel<1, 5>(GDArgs)", 3),
    ("gemmd_kernel<6, 5>(GDArgs)", 4),
    ("gemmd_kernel<8, 3>(GDArgs)", 4),
    ("gemmd_kernel<8, 4>(GDArgs)", 4),
]
# the build's flags, and two other schedules that the compiler might choose: the
# order must not rest on one
SCHEDULES = {"build": (), "topdown": ("-mllvm", "-misched-prera-direction=topdown"),
             "none": ("-mllvm", "-enable-misched=0")}
CASES = [(i, s) for s in SCHEDULES for i, _ in INSTANCES]


@pytest.fixture(scope="module")
def broken():
    """(instance, schedule) -> what its compiled code breaks."""
    ring = dict(INSTANCES)
    with ThreadPoolExecutor(4) as ex:
        code = list(ex.map(lambda c: pipeline_asm.compile_kernel(c[0], SCHEDULES[c[1]]), CASES))
    return {c: pipeline_asm.violations(k, ring[c[0]]) for c, k in zip(CASES, code)}


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[1]}-{c[0]}")
def test_no_copy_over_a_slot_being_read(broken, case):
    assert not broken[case]["reads"]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[1]}-{c[0]}")
def test_a_step_waits_for_its_record(broken, case):
    assert not broken[case]["copies"]
