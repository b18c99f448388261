"""The engine's pools of pinned host memory (descriptor uploads, read-out results)
against a stand-in for the HIP runtime (fake_hip.c); no GPU.

Each test runs in a process of its own: the stand-in has to be loaded before
the engine.
"""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SETUP = """
import ctypes as C, sys, threading, time
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
L = C.CDLL(sys.argv[2])
L.dq_last_error.restype = C.c_char_p
L.dq_result_acquire.restype = C.c_void_p
L.dq_result_acquire.argtypes = [C.c_size_t]
L.dq_readout_ws_bytes.restype = C.c_size_t
hip.fake_flags.restype = C.c_uint32
n = 8
state = C.create_string_buffer(16 << n)
states = (C.c_void_p * 1)(C.addressof(state))
wsb = L.dq_readout_ws_bytes(n, 1, 0)

def upload():  # a read-out uploads its state pointers; 0 or an error code
    ws = C.create_string_buffer(wsb + 256)
    keep.append(ws)
    at = (C.addressof(ws) + 255) // 256 * 256
    return L.dq_readout_many(2, n, states, 1, None, 0, None, None, C.c_void_p(at), C.c_size_t(wsb), None)

keep = []
"""


def run(tmp_path, body):
    fake = tmp_path / "libfake_hip.so"
    subprocess.check_call(["cc", "-O1", "-shared", "-fPIC", "-pthread", "-o", str(fake), os.path.join(ROOT, "tests", "fake_hip.c")])
    lib = os.path.join(ROOT, "dgquest_amd", "lib", "libdgq_engine.so")
    p = subprocess.run([sys.executable, "-c", SETUP + body, str(fake), lib], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr


def test_memory_shared_with_running_kernels_is_coherent(tmp_path):
    # hipHostMallocCoherent (0x40000000): a host that polls sees a word before its kernel ends, and a kernel
    # sees what the host wrote into a buffer that an earlier kernel has read
    run(tmp_path, """
assert L.dq_result_acquire(64)
assert hip.fake_allocs() == 1
assert upload() == 0, L.dq_last_error()
assert hip.fake_allocs() == 2
for i in range(2):
    assert hip.fake_flags(i) & 0x40000000, hex(hip.fake_flags(i))
    assert not hip.fake_flags(i) & 0x80000000
""")


def test_uploads_past_a_long_queue_wait_for_one_slot_only(tmp_path):
    # 64 uploads of a busy stream hold every slot; two more threads upload.  One upload read is one of them
    # served: neither waits for the device to be idle, nor for the other.
    run(tmp_path, """
done = []
for _ in range(64):
    assert upload() == 0
assert hip.fake_queued() == 64
threads = [threading.Thread(target=lambda: done.append(upload()), daemon=True) for _ in range(2)]
for t in threads:
    t.start()
time.sleep(0.2)
seen = [len(done)]
for k in range(2):
    hip.fake_run(1)
    end = time.time() + 5
    while len(done) <= k and time.time() < end:
        time.sleep(0.001)
    seen.append(len(done))
queued, syncs = hip.fake_queued(), hip.fake_syncs()
while any(t.is_alive() for t in threads):  # let them end either way
    hip.fake_run(1000)
assert seen == [0, 1, 2], seen
assert queued == 64 and syncs == 0 and done == [0, 0], (queued, syncs, done)
""")
