"""Runs the library against a HIP runtime without a device (host/fake_hip.cpp):
which kernels a call would launch, what it refuses, and what it does when a
launch fails, on the CPU.

run(code) executes Python in a process of its own (the real runtime is not
loaded there) and returns its `result`, a JSON value. The code sees `sa`,
`np`, `dev` (a siphon_amd.Device of 256 CUs), `fake` (the runtime's controls),
`X` (an address to pass as device memory), `upload(type, n_out, n_in)` and
`launched()`, the launches since the last fake.fake_reset as [kernel, grid]
with the kernel's template arguments as numbers.
"""
import json
import os
import re
import subprocess
import sys
import textwrap

TESTS = os.path.dirname(os.path.abspath(__file__))
SRC, SO = (os.path.join(TESTS, "host", "fake_hip." + e) for e in ("cpp", "so"))


def _build():
    if not os.path.exists(SO) or os.path.getmtime(SO) < os.path.getmtime(SRC):
        tmp = f"{SO}.{os.getpid()}"
        subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", "-Wno-unused-result", "-o", tmp, SRC], check=True)
        os.replace(tmp, SO)


def run(code, lib=None):
    _build()
    res = subprocess.run([sys.executable, "-m", "tests.fake_hip", *([lib] if lib else [])],
                         input=textwrap.dedent(code), text=True, capture_output=True,
                         cwd=os.path.dirname(TESTS))
    assert res.returncode == 0, res.stderr[-4000:]
    return json.loads(res.stdout.splitlines()[-1])


def kernel(text):
    """"sihip::gemmx_kernel<12u, 14u, 5>(...)" -> "gemmx_kernel<12,14,5>"."""
    m = re.match(r"(?:void )?sihip::(\w+)(<[^>]*>)?", text)
    return m.group(1) + re.sub(r"(?<=\d)u| ", "", m.group(2) or "")


def _main():
    import ctypes

    import numpy as np

    fake = ctypes.CDLL(SO, mode=ctypes.RTLD_GLOBAL)
    fake.fake_kernel.restype = fake.fake_order.restype = ctypes.c_char_p
    fake.fake_grid.restype = ctypes.c_uint
    import siphon_amd as sa

    dev = sa.Device(0, lib_path=sys.argv[1] if len(sys.argv) > 1 else None)

    def upload(wtype, n_out, n_in):
        return dev.upload(wtype, n_out, n_in, np.zeros(n_out * sa.row_bytes(wtype, n_in), np.uint8))

    def launched():
        return [[kernel(fake.fake_kernel(i).decode()), *(fake.fake_grid(i, d) for d in range(2))]
                for i in range(fake.fake_launches())]

    scope = {"sa": sa, "np": np, "dev": dev, "fake": fake, "X": 1 << 36, "upload": upload,
             "launched": launched, "result": None}
    exec(sys.stdin.read(), scope)
    print(json.dumps(scope["result"]))


if __name__ == "__main__":
    _main()
