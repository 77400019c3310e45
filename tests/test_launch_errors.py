"""A kernel whose LDS limit cannot be raised: every call says so and launches
nothing, and the limit is raised on each device.  No GPU: the HIP calls a
launch makes are stand-ins (hip_stub.c), preloaded in a process of its own."""
import os
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent

PROGRAM = """
import ctypes, sys
sys.path.insert(0, {root!r})
from ztensor_amd import _lib
stub, lib, p, big = ctypes.CDLL({stub!r}), _lib.load(), 1 << 20, 1 << 40
blocks, w4 = lib.zt_gemm_blkt_tokens_f32, lib.zt_gemm_w4a16t_tokens_f32
calls = {{}}
for fmt in (5, 6, 7):  # all of K in one launch, and K ranges whose sums a second launch adds
    calls["block", fmt, 1] = lambda fmt=fmt: blocks(fmt, p, p, p, p, p, 1 << 17, 512, 20, p, big, 0)
    calls["block", fmt, 2] = lambda fmt=fmt: blocks(fmt, p, p, p, p, p, 1 << 17, 2048, 20, p, big, 0)
calls["w4a16", 0, 1] = lambda: w4(p, p, p, p, 1 << 19, 1024, 20, 128, p, big, 0)
calls["w4a16", 0, 2] = lambda: w4(p, p, p, p, 1 << 14, 1 << 15, 20, 128, p, big, 0)
calls["few", 0, 1] = lambda: lib.zt_gemm_wide_f32(0, p, 0, 0, p, 128, p, 1, p, 8192, 1024, 4, p, big, 0)
calls["wide", 1, 2] = lambda: lib.zt_gemm_wide_f32(1, p, 0, 0, 0, 0, p, 0, p, 8192, 1024, 100, p, big, 0)
for (name, fmt, launches), call in calls.items():
    for attempt in range(2):
        stub.stub_set(1, 0)
        rc = call()
        print(name, fmt, launches, "attempt", attempt, "gives", rc, "after", stub.stub_launches(), flush=True)
        # (the wide GEMM packs its activations first)
        assert rc == 1 and stub.stub_launches() == (name == "wide") and stub.hipGetLastError() == 0
done = set()
for device in (0, 1, 0):
    for (name, fmt, launches), call in calls.items():
        stub.stub_set(0, device)
        rc = call()
        print(name, fmt, launches, "device", device, "gives", rc, "after", stub.stub_launches(), flush=True)
        assert rc == 0 and stub.stub_launches() == launches
        assert stub.stub_raised() == ((name, fmt, device) not in done)
        done.add((name, fmt, device))
"""


def test_an_lds_limit_that_cannot_be_raised_is_reported_every_time(tmp_path):
    stub = tmp_path / "hip_stub.so"
    subprocess.run([os.environ.get("CC", "gcc"), "-shared", "-fPIC", "-O1", "-o", str(stub), str(HERE / "hip_stub.c")],
                   check=True)
    env = dict(os.environ, LD_PRELOAD=" ".join([str(stub), os.environ.get("LD_PRELOAD", "")]).strip())
    r = subprocess.run([sys.executable, "-c", PROGRAM.format(root=str(HERE.parent), stub=str(stub))],
                       capture_output=True, text=True, env=env, timeout=120)
    assert r.returncode == 0, r.stdout[-1500:] + r.stderr[-1500:]
