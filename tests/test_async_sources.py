"""Sources of asynchronous copies outlive the wait on every error path.

The host library, with AddressSanitizer, runs on stand-ins for the HIP
runtime (fake_hip.c) whose copies take place at the next wait; each launch,
copy and wait of a call fails in turn (NSFPS_INJECT).  A descriptor that is
gone by the time its copy is made is a heap-use-after-free report."""

import os
import subprocess
import sys

import pytest

from conftest import ROOT

CALLS = """
import os
import numpy as np
from ns_fps_amd.capi import Lib, NsfpsError
lib = Lib()
P = np.random.RandomState(1).uniform(-1, 1, (9, 500, 3)).astype(np.float32)
rng = (-1.0, 1.0, -1.0, 1.0, -1.0, 1.0, 8, 8, 8)
out = np.zeros((9, 60), np.int32)

def plan():
    p = lib.plan_create(P[0], 500, rng)
    try:
        lib.plan_sample(p, 60, out.ctypes.data)
    finally:
        lib.plan_destroy(p)

calls = {"host": lambda: lib.fps(P[0], 60, rng),
         "batched": lambda: lib.fps_batched(P, 60),
         "batched_ranges": lambda: lib.fps_batched(P, 60, [(*rng[:6], 8, 8, 8 + b) for b in range(9)]),
         "batched_device": lambda: lib.fps_batched_device(P.ctypes.data, 9, 500, 60, out.ctypes.data),
         "device": lambda: lib.fps_device(P.ctypes.data, 500, 60, rng, out.ctypes.data),
         "noalloc": lambda: lib.fps_device_noalloc(P.ctypes.data, 500, 60, rng, out.ctypes.data),
         "plan": plan}
os.environ["NSFPS_SMALL"] = SMALL
for name, call in calls.items():
    for kind in ("launch", "copy", "sync"):
        failed = 0
        for i in range(1, 400):
            os.environ["NSFPS_INJECT"] = f"{kind}:{i}"
            said = ""
            try:
                call()
            except NsfpsError as e:
                said = str(e)
            if "injected failure" not in said:  # nothing left to fail
                break  # (without kernels, the call may still refuse what it reads back)
            failed += 1
        assert failed >= 1, (name, kind)
        print(name, kind, failed, flush=True)
print("every call done")
"""


@pytest.mark.parametrize("small", ["0", "1"])
def test_copy_sources_outlive_the_wait(tmp_path, small):
    from ns_fps_amd import sanitize
    try:
        env = sanitize.sanitized_env()
    except RuntimeError:
        pytest.skip("sanitized build missing: python -m ns_fps_amd.build sanitize")
    fake = str(tmp_path / "fake_hip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-Wall", os.path.join(ROOT, "tests", "fake_hip.c"),
                    "-o", fake], check=True)
    env["LD_PRELOAD"] += ":" + fake
    # the two runtimes share one report file: the last log_path read wins
    env["ASAN_OPTIONS"] = f"detect_leaks=0:halt_on_error=1:abort_on_error=1:log_path={tmp_path}/report"
    env["UBSAN_OPTIONS"] = f"halt_on_error=1:log_path={tmp_path}/report"
    p = subprocess.run([sys.executable, "-c", f"SMALL = {small!r}\n" + CALLS], cwd=ROOT, env=env,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    reports = "".join(f.read_text()[:3000] for f in tmp_path.glob("report*"))
    assert not reports, p.stdout + reports
    assert p.returncode == 0 and p.stdout.endswith("every call done\n"), p.stdout
