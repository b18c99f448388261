"""Recording a long circuit lets other Python threads run and signals be handled,
as recording it gate by gate does (no GPU)."""
import signal
import threading
import time

import pytest

from dgquest_amd import quest as Q

GATES = [("rotateZ", (1,), (0.5,))] * 2_000_000  # some 0.2 s of recording


@pytest.fixture
def register():
    api = Q.load(2)
    q = api.dgq_create_recorder(4)
    yield api, q
    api.dgq_destroy_recorder(q)


def test_other_threads_run_meanwhile(register):
    api, q = register
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.001)

    t = threading.Thread(target=tick)
    t.start()
    time.sleep(0.05)
    a = time.perf_counter()
    api.apply_circuit(q, GATES)
    b = time.perf_counter()
    stop.set()
    t.join()
    inside = [x for x in ticks if a + 0.2 * (b - a) < x < a + 0.8 * (b - a)]
    assert b - a > 0.05 and len(inside) >= 3, (b - a, len(inside))


def test_a_signal_ends_it(register):
    api, q = register

    def stop(*_):
        raise KeyboardInterrupt

    old = signal.signal(signal.SIGALRM, stop)
    try:
        a = time.perf_counter()
        with pytest.raises(KeyboardInterrupt):
            signal.setitimer(signal.ITIMER_REAL, 0.02)
            api.apply_circuit(q, GATES)
            took = time.perf_counter() - a
            time.sleep(0.1)
            pytest.fail(f"recorded to the end, {took} s")
    finally:
        signal.setitimer(signal.ITIMER_REAL, 0)
        signal.signal(signal.SIGALRM, old)
    import ctypes as C

    from dgquest_amd import serve as S

    S._bind(api.lib)
    cnt = C.c_int()
    api.dgq_recorder_export(q, None, 0, C.byref(cnt), None, None, None, None)
    assert 0 < cnt.value < len(GATES)
