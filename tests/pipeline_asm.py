"""Walks the gfx950 assembly of the ring-buffered prompt GEMMs (gemmx.h,
gemmd.h) and checks the order that their pipeline rests on, over every path
through the kernel. No GPU: the kernels are compiled to assembly only.

A step of those kernels waits for its own activation record by count, meets
the other waves at a bare s_barrier and then copies a later record into the
ring slot that the step before has read. So, by the waits written in the
source alone (the ones the compiler adds for its own registers may move or go
with its schedule):

  - at a step's barrier no copy of that step's record, or of an earlier one,
    is in flight: of the wave's copies at most those of the R - 2 later
    records are;
  - no copy is issued after a barrier that was passed with LDS reads in
    flight.

Memory operations of a wave retire in the order of issue (loads, and copies
to LDS), so vmcnt(N) leaves the youngest N in flight, copies or not.
"""
import os
import re
import subprocess
import tempfile

from siphon_amd import build

CSRC = os.path.join(build.PKG, "csrc")
_BRANCH = re.compile(r"s_(c?branch)\S*\s+(\S+)")
_VMCNT, _LGKM = re.compile(r"vmcnt\((\d+)\)"), re.compile(r"lgkmcnt\((\d+)\)")
_VMEM = ("buffer_", "global_", "flat_", "scratch_")


def compile_kernel(instance, flags=()):
    """The instructions of one kernel, given as an explicit instantiation."""
    src = ("#include <hip/hip_runtime.h>\n#include \"gemmd.h\"\n"
           f"namespace sihip {{ template __global__ void {instance}; }}\n")
    with tempfile.TemporaryDirectory() as d:
        hip, out = os.path.join(d, "k.hip"), os.path.join(d, "k.s")
        with open(hip, "w") as f:
            f.write(src)
        keep = [f for f in build.HIPCC_FLAGS if f not in ("-fPIC", "-shared")]
        res = subprocess.run([build.hipcc(), *keep, *flags, "--cuda-device-only", "-S", "-I", CSRC, hip, "-o", out],
                             capture_output=True, text=True)
        if res.returncode:
            raise RuntimeError(f"{instance}: {res.stderr[-2000:]}")
        with open(out) as f:
            found = _functions(f.read())
    name = instance.split("<")[0]
    return next(v for k, v in found.items() if f"{len(name)}{name}I" in k)


def _functions(asm):
    """mangled name -> its instructions [(text, written in the source)], with
    labels as text ending in a colon."""
    found, name, inside = {}, None, False
    for line in asm.splitlines():
        t = line.split(";")[0].strip()
        if "#ASMSTART" in line:
            inside = True
        elif "#ASMEND" in line:
            inside = False
        elif re.match(r"_Z\w+:", t):
            name = t[:-1]
            found[name] = []
        elif t.startswith(".Lfunc_end"):
            name = None
        elif name and t and (not t.startswith(".") or t.endswith(":")):
            found[name].append((t, inside))
    return found


def violations(code, ring):
    """What breaks each rule on some path, for a ring of that many slots:
    {"copies": texts, "reads": texts}. Before the first barrier a wave issues
    the copies of ring - 1 records."""
    first = next(i for i, (t, w) in enumerate(code) if t == "s_barrier")
    later_copies = sum(t.endswith(" lds") for t, _ in code[:first]) // (ring - 1) * (ring - 2)
    label = {t[:-1]: i for i, (t, _) in enumerate(code) if t.endswith(":")}
    bad, seen, todo = {"copies": set(), "reads": set()}, set(), [(0, "", False, False)]
    while todo:
        pc, queue, reads, stale = todo.pop()
        while True:
            t, written = code[pc]
            if t.endswith(":"):
                if (pc, queue, reads, stale) in seen:
                    break
                seen.add((pc, queue, reads, stale))
            elif t.startswith("s_waitcnt"):
                if written:
                    m = _VMCNT.search(t)
                    if m:
                        n = int(m.group(1))
                        queue = queue[len(queue) - n:] if n < len(queue) else queue
                        if n == 0:
                            break  # past the pipeline
                    m = _LGKM.search(t)
                    reads = reads and not (m and m.group(1) == "0")
            elif t.startswith("s_barrier"):
                if queue.count("D") > later_copies:
                    bad["copies"].add(f"line {pc}: {queue.count('D')} copies in flight at a barrier, {later_copies} allowed")
                stale = stale or reads
                reads = False
            elif t.startswith(_VMEM):
                if t.endswith(" lds"):
                    if stale:
                        bad["reads"].add(f"line {pc}: a copy after a barrier passed with LDS reads in flight")
                    queue += "D"
                else:
                    queue += "L"
                queue = queue[-64:]
            elif t.startswith("ds_read"):
                reads = True
            elif t.startswith("s_endpgm"):
                break
            else:
                m = _BRANCH.match(t)
                if m:
                    to = (label[m.group(2)], queue, reads, stale)
                    if m.group(1) == "branch":
                        pc, queue, reads, stale = to
                        continue
                    todo.append(to)
            pc += 1
    return bad
