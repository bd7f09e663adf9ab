"""The host C layer when a large block cannot be had, under AddressSanitizer,
UndefinedBehaviorSanitizer and the leak checker, on the CPU (the device layer is
the test double tests/c/gpu_double.c): every allocation of 64 KiB or more of a
forward solution with tangents and of two gradients is refused in turn
(tests/c/alloc_checks.c); the call fails with an error, or its results are
those of a call without the failure, never a gradient with entries left out."""
import os
import subprocess

from conftest import ROOT
from test_host_sanitizers import ENV, SAN


def test_refused_allocations_are_errors(tmp_path):
    cc = ["gcc", "-std=gnu99", "-Wall", "-Wextra", "-Wno-unused-parameter", "-Wno-format-truncation"] + SAN + \
        ["-I", os.path.join(ROOT, "include")]
    host, exe = str(tmp_path / "lmie_host.o"), str(tmp_path / "alloc_checks")
    subprocess.check_call(cc + ["-Dmalloc=test_malloc", "-Dcalloc=test_calloc", "-c",
                                os.path.join(ROOT, "lmie_amd/csrc/lmie_host.c"), "-o", host])
    subprocess.check_call(cc + [host] + [os.path.join(ROOT, s) for s in ("tests/c/gpu_double.c", "tests/c/alloc_checks.c")] +
                          ["-o", exe, "-lm", "-lpthread"])
    r = subprocess.run([exe], env=ENV, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "allocation checks: ok" in r.stdout, r.stdout[-3000:] + r.stderr[-3000:]
