"""The largest clouds of the allocation-free entry point, as include/nsfps.h
states them: its layout alone decides, so stand-ins for the HIP runtime
(fake_hip.c) answer on the CPU.  A cloud that fits goes on to the build."""

import os
import re
import subprocess
import sys

from conftest import ROOT

PROBE = """
import numpy as np
from ns_fps_amd.capi import Lib, NsfpsError
lib = Lib()
xyz, out = np.zeros((500000, 3), np.float32), np.zeros(500000, np.int32)

def fits(n, m, blocks):
    try:
        lib.fps_device_noalloc(xyz.ctypes.data, n, m, (-1, 1, -1, 1, -1, 1, *blocks), out.ctypes.data)
    except NsfpsError as e:
        return e.status != 4  # NSFPS_EUNSUPPORTED
    return True

for few in (True, False):
    for blocks in ((32, 32, 32), (16, 16, 16), (64, 64, 16)):
        lo, hi = 20000, 499999
        while lo < hi:
            mid = (lo + hi + 1) // 2
            lo, hi = (mid, hi) if fits(mid, mid // 16 if few else mid - 1, blocks) else (lo, mid - 1)
        print(lo)
"""


def test_stated_limits(tmp_path):
    with open(os.path.join(ROOT, "include", "nsfps.h")) as f:
        text = f.read()
    text = text[text.index("for samples of a"):text.index("Same arguments, samples and guards")]
    said = [int(v.replace(",", "")) for v in re.findall(r"\d{3},\d{3}", text)]
    fake = str(tmp_path / "fake_hip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-Wall", os.path.join(ROOT, "tests", "fake_hip.c"),
                    "-o", fake], check=True)
    env = dict(os.environ, LD_PRELOAD=":".join(filter(None, [fake, os.environ.get("LD_PRELOAD")])))
    p = subprocess.run([sys.executable, "-c", PROBE], cwd=ROOT, env=env, check=True,
                       stdout=subprocess.PIPE, text=True)
    assert [int(v) for v in p.stdout.split()] == said
