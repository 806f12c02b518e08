"""16-bit GEMMs captured into a HIP graph: a graph that was captured before the
library's workspace grew still replays with the workspace that it recorded."""
import ctypes as C

import numpy as np
import pytest

import edgecore_amd as ec

pytestmark = pytest.mark.gpu


class _Graph:
    """What `call` enqueues on ec_stream(), captured."""

    def __init__(self, call):
        self.hip = C.CDLL("libamdhip64.so")
        self.stream = C.c_void_p(ec.lib().ec_stream())
        graph, self.exec = C.c_void_p(), C.c_void_p()
        assert self.hip.hipStreamBeginCapture(self.stream, 1) == 0  # thread-local
        rc, err = call(), ec.last_error()
        assert self.hip.hipStreamEndCapture(self.stream, C.byref(graph)) == 0
        assert rc == 0, err
        assert self.hip.hipGraphInstantiate(C.byref(self.exec), graph, None, None, C.c_size_t(0)) == 0
        assert self.hip.hipGraphDestroy(graph) == 0

    def replay(self):
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0
        assert ec.lib().ec_sync() == 0

    def close(self):
        assert self.hip.hipGraphExecDestroy(self.exec) == 0


def _call(M, K, N, seed):
    """Device operands of one fp16 GEMM and the call."""
    rng = np.random.default_rng(seed)
    A, B = rng.normal(0, 1, (M, K)).astype(np.float32), rng.normal(0, 0.02, (N, K)).astype(np.float16)
    bufs = [ec.DeviceBuffer(4 * M * N), ec.DeviceBuffer.from_array(A), ec.DeviceBuffer.from_array(B.view(np.uint16))]
    out, a, b = (x.ptr for x in bufs)
    return bufs, lambda: ec.lib().ec_gemm_fp16_fp32_dev(out, a, b, M, K, N)


@pytest.mark.parametrize("M,K,N", [(16, 64, 40), (40, 512, 200), (5, 1001, 70), (40, 101, 70)])
def test_graph_outlives_a_larger_workspace(M, K, N):
    """Whole 16-byte chunks (the parts' workspace) and ragged rows (none)."""
    L = ec.lib()
    bufs, call = _call(M, K, N, 1)
    assert call() == 0 and L.ec_sync() == 0
    want = bufs[0].to_array(np.uint32, (M, N))
    g = _Graph(call)
    others, poison = [], np.full(1 << 18, 0xFF, np.uint8)
    try:
        for i, rows in enumerate((64, 512, 2048)):
            # a larger call each time, then memory that a freed workspace would be
            big, run = _call(rows, 1024 + 512 * i, 64, 2)
            others += big
            assert run() == 0 and L.ec_sync() == 0
            first = big[0].to_array(np.uint32, (rows, 64))
            others += [ec.DeviceBuffer.from_array(poison) for _ in range(16)]
            assert L.ec_memset_dev(bufs[0].ptr, 0, 4 * M * N) == 0
            g.replay()
            assert np.array_equal(bufs[0].to_array(np.uint32, (M, N)), want)
            assert all((b.to_array(np.uint8, poison.shape) == 0xFF).all() for b in others[-16:])
            assert run() == 0 and L.ec_sync() == 0  # the larger one again, after the replay
            assert np.array_equal(big[0].to_array(np.uint32, (rows, 64)), first)
    finally:
        g.close()
        for b in bufs + others:
            b.close()


def test_no_growth_inside_a_capture():
    """A captured call that would need a larger workspace is refused, and the
    capture goes on without it."""
    M, K, N = 8192, 32768, 8  # 1.6 GB of parts
    bufs = [ec.DeviceBuffer(n) for n in (4 * M * N, 4 * M * K, 2 * N * K)]

    def call():
        return ec.lib().ec_gemm_fp16_fp32_dev(bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, M, K, N)

    small, first = _call(16, 64, 40, 4)
    assert first() == 0 and ec.lib().ec_sync() == 0
    seen = []

    def both():
        seen.append((call(), ec.last_error()))
        return first()

    g = _Graph(both)
    try:
        assert seen[0][0] < 0 and "capture" in seen[0][1]
        g.replay()
    finally:
        g.close()
        for b in bufs + small:
            b.close()


def test_release_with_retired_workspaces():
    """ec_release gives the retired workspaces back; the next call starts anew."""
    for _ in range(2):
        bufs, call = _call(32, 256, 40, 5)
        assert call() == 0 and ec.lib().ec_sync() == 0
        want = bufs[0].to_array(np.uint32, (32, 40))
        g = _Graph(call)
        big, run = _call(256, 2048, 40, 6)
        assert run() == 0 and ec.lib().ec_sync() == 0
        g.replay()
        assert np.array_equal(bufs[0].to_array(np.uint32, (32, 40)), want)
        g.close()
        for b in bufs + big:
            b.close()
        assert ec.lib().ec_release() == 0 or "models still loaded" in ec.last_error()
