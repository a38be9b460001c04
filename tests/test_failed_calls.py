"""A host call that fails part of the way leaves nothing queued, without a GPU.

The synchronous entry points put slots, tokens and symbols into pinned memory that the step's
kernels read in place, and the head and the CDF readers write pinned memory too.  A call that
returned an error with kernels still queued would let them read what the next call puts there
and advance another stream's state.  So each runtime call of each entry point is made to fail in
turn, on a stand-in for the HIP runtime (tests/fake_hip.c) that counts what may still run, the
parts of a split step on their own streams included.
"""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = r"""
import ctypes, json, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_hip_fail.argtypes = [ctypes.c_char_p, ctypes.c_long]
import numpy as np
from redukt_amd import ffi
path, profile = sys.argv[2], int(sys.argv[3])
FORWARD_FAILED, OK = int(ffi.BackendResult.FORWARD_FAILED), 0
bad, seen = [], {}
with ffi.PluginBackend(path, profile=profile) as be:
    L, V = be.lib.lib, be.vocab
    be.batch_init(200)
    u32 = lambda a: np.ascontiguousarray(a, np.uint32).ctypes.data_as(ctypes.POINTER(ctypes.c_uint32))
    out = np.empty((200, V + 1), np.uint32)
    f32 = out.ctypes.data_as(ctypes.POINTER(ctypes.c_float))
    def entries(n):
        s, t = np.arange(n, dtype=np.uint32), np.arange(n, dtype=np.uint32) % V
        ticket = ctypes.c_uint64()
        def queued():
            rc = L.redukt_backend_forward_batch_cdf_sym_submit(n, u32(s), u32(t), u32(t), V, ctypes.byref(ticket))
            return rc if rc != OK else L.redukt_backend_forward_batch_cdf_sym_wait(ticket.value, u32(out), n)
        return {"forward_batch": lambda: L.redukt_backend_forward_batch(n, u32(s), u32(t), f32, V),
                "probs": lambda: L.redukt_backend_forward_batch_probs(n, u32(s), u32(t), f32, V),
                "cdf": lambda: L.redukt_backend_forward_batch_cdf(n, u32(s), u32(t), u32(out), V + 1),
                "cdf_sym": lambda: L.redukt_backend_forward_batch_cdf_sym(n, u32(s), u32(t), u32(t), u32(out), V),
                "cdf_find": lambda: L.redukt_backend_forward_batch_cdf_find(n, u32(s), u32(t), u32(t), u32(out), V),
                "queued": queued,
                "reset": lambda: L.redukt_backend_batch_reset(u32(s), n)}
    for n in (3, 130):
        calls = entries(n)
        if n == 3:
            calls["forward"] = lambda: L.redukt_backend_forward(1, f32, V)
        for name, call in calls.items():
            for again in (0, 1):      # the first call of a shape captures its graphs, the next ones replay them
                for fn in ("hipLaunchKernel", "hipGraphLaunch", "hipGraphInstantiate", "hipEventRecord", "hipEventQuery",
                           "hipStreamWaitEvent", "hipMemcpyAsync"):
                    for k in range(400):
                        if not again:
                            be.batch_init(200)      # (drops the graphs)
                        fake.fake_hip_fail(fn.encode(), k)
                        rc = call()
                        pending = fake.fake_hip_pending()
                        if not fake.fake_hip_failed():
                            if rc != OK or pending:
                                bad.append([name, n, fn, "none failed", rc, pending])
                            break
                        seen[name + " " + fn] = seen.get(name + " " + fn, 0) + 1
                        if rc != FORWARD_FAILED or pending:
                            bad.append([name, n, fn, k, rc, pending])
                            L.redukt_backend_batch_reset(None, 0)
    fake.fake_hip_fail(b"", -1)
print(json.dumps({"bad": bad, "seen": seen}))
"""


@pytest.mark.parametrize("arch,profile", [("mamba", 6), ("mamba", 64), ("rwkv", 2)])
def test_a_failed_call_leaves_nothing_queued(tmp_path, fake_hip, arch, profile):
    from redukt_amd import rbin, rwkv, synth

    path = str(tmp_path / "m.rbin")
    if arch == "mamba":
        synth.write_synthetic_mamba(path, rbin.MambaDims(vocab=2000, d_model=64, n_layer=1), seed=1)
    else:
        rwkv.write_synthetic(path, rwkv.RwkvDims(vocab=2000, d_model=64, n_layer=1), seed=1)
    r = subprocess.run([sys.executable, "-c", CHILD, fake_hip, path, str(profile)], cwd=ROOT, capture_output=True,
                       text=True, timeout=300, env={**os.environ, "PYTHONPATH": ROOT})
    assert r.returncode == 0, r.stderr[-2000:]
    got = json.loads(r.stdout.strip().splitlines()[-1])
    for name in ("forward_batch", "probs", "cdf", "cdf_sym", "cdf_find", "queued"):
        assert got["seen"].get(name + " hipGraphLaunch") and got["seen"].get(name + " hipEventRecord"), got["seen"]
    assert not got["bad"], (len(got["bad"]), got["bad"][:10])
