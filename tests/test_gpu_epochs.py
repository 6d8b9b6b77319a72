"""Look-back launches numbered by the host (eager) and on the device (captured
in a graph) share one status array: replays and eager calls in any order, and a
capture of the queue's native stream, all match the oracle."""
import ctypes as C

import numpy as np
import pytest

import compute_amd as ca
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 40007, 3 * 32768 + 1, 1 << 21])
def test_replays_between_eager_calls(queue, n):
    rng = np.random.default_rng(n)
    queue.reserve(n, 8)
    a, out, eager = (ca.DeviceArray(n, np.int32, queue) for _ in range(3))
    g = ca.Graph(queue)
    with g:
        ca.scan(queue, a, out, True, init=3)
    for rep in range(4):
        x = rng.integers(-100, 100, n).astype(np.int32)
        ca.check(ca.lib().bcmi_memcpy(queue.h, a.ptr, x.ctypes.data_as(C.c_void_p), x.nbytes, ca.H2D, 1))
        g.launch()
        for _ in range(rep):
            ca.scan(queue, a, eager, False)
        g.launch()
        queue.finish()
        assert np.array_equal(out.to_host(queue), O.scan(x, True, 3)), rep
        if rep:
            assert np.array_equal(eager.to_host(queue), O.scan(x, False)), rep


def test_capture_of_the_native_stream(queue):
    """The queue's stream captured through the HIP API (bcmi_queue_native),
    not bcmi_graph_begin: every replay still gets epochs of its own."""
    hip = C.CDLL("libamdhip64.so")
    n = 5 * 32768 + 17
    rng = np.random.default_rng(7)
    queue.reserve(n, 8)
    a, out = ca.DeviceArray(n, np.int32, queue), ca.DeviceArray(n, np.int32, queue)
    stream = C.c_void_p(ca.lib().bcmi_queue_native(queue.h))
    graph, ex = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 1) == 0  # thread-local
    ca.scan(queue, a, out, True, init=0)
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)) == 0
    try:
        for rep in range(4):
            x = rng.integers(-100, 100, n).astype(np.int32)
            ca.check(ca.lib().bcmi_memcpy(queue.h, a.ptr, x.ctypes.data_as(C.c_void_p), x.nbytes, ca.H2D, 1))
            assert hip.hipGraphLaunch(ex, stream) == 0
            queue.finish()
            assert np.array_equal(out.to_host(queue), O.scan(x, True, 0)), rep
    finally:
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(graph)
