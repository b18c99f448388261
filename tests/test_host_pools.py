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
    p = subprocess.run([sys.executable, "-c", SETUP + body, str(fake), lib], capture_output=True, text=True, timeout=120, cwd=ROOT)
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


def test_a_buffer_whose_kernel_was_launched_is_in_use_whatever_error_is_pending(tmp_path):
    # an error that another call left says nothing about this launch: the copy will read its buffer
    run(tmp_path, """
hip.fake_source.restype = C.c_void_p
hip.fake_pending(600)
upload()
upload()
hip.fake_pending(0)
assert upload() == 0
assert hip.fake_queued() == 3
assert len({hip.fake_source(i) for i in range(3)}) == 3
""")


def test_a_one_tile_sweep_that_was_launched_keeps_its_buffer(tmp_path):
    run(tmp_path, """
import numpy as np
from dgquest_amd import circuits, quest as Q
api = Q.load(2)
r = api.dgq_create_recorder(10)
api.apply_circuit(r, circuits.layered_u3_cz(10, 2, 1))
blocks, phases, ops, _ = api.recorder_plan(r, k=4, R=3, W=1)
assert len(blocks) == 1
job = np.zeros(1, dtype=np.dtype([("state", "<u8"), ("block", "<u4"), ("pad", "<u4"), ("base_hi", "<u8")]))
big = C.create_string_buffer(16 << 10)
job["state"] = C.addressof(big)
begin = (C.c_uint32 * 2)(0, 1)
L.dq_apply_ws_bytes.restype = C.c_size_t
wsb = L.dq_apply_ws_bytes(1, len(phases), len(ops), 1)
ws = C.create_string_buffer(wsb + 256)
at = (C.addressof(ws) + 255) // 256 * 256

def sweep():
    vp = C.c_void_p
    return L.dq_apply_blocks(2, vp(blocks.ctypes.data), 1, vp(phases.ctypes.data), len(phases), vp(ops.ctypes.data), len(ops),
                             vp(job.ctypes.data), begin, 1, vp(at), C.c_size_t(wsb), None)

before = hip.fake_allocs()
assert sweep() == 0, L.dq_last_error()
assert hip.fake_allocs() == before + 1 and hip.fake_queued() == 0  # its workgroup reads the buffer, never run here
hip.fake_pending(600)
assert sweep() != 0
hip.fake_pending(0)
assert sweep() == 0
assert hip.fake_allocs() == before + 3
hip.fake_capture(1)
assert sweep() != 0 and b"captur" in L.dq_last_error(), L.dq_last_error()
""")


def test_uploads_are_refused_while_their_stream_is_captured(tmp_path):
    # a graph would read the staging buffer at every replay, long after it went to other uploads
    run(tmp_path, """
assert upload() == 0
hip.fake_run(1)
hip.fake_capture(1)
assert upload() != 0 and b"captur" in L.dq_last_error(), L.dq_last_error()
assert hip.fake_queued() == 0
hip.fake_capture(0)
assert upload() == 0
""")


def test_a_failed_read_out_gives_its_result_slot_back_when_its_kernels_are_done(tmp_path):
    # the kernels of a call that ends with an error may still store to the slot
    run(tmp_path, """
m = 14  # two launches of 256 threads each
big = C.create_string_buffer(16 << m)
L.dq_prob_ws_bytes.restype = C.c_size_t
wsb = L.dq_prob_ws_bytes(m)
ws = C.create_string_buffer(wsb)
out = (C.c_double * (m + 1))()
hip.fake_pending(600)
assert L.dq_prob_zero_all(big, m, 2, out, ws, C.c_size_t(wsb), None) != 0
assert hip.fake_stream_syncs() == 1
assert L.dq_read_amps(big, m, 2, None, C.c_uint64(0), C.c_uint64(4), out, ws, C.c_size_t(wsb), None) != 0
assert hip.fake_stream_syncs() == 2
""")
