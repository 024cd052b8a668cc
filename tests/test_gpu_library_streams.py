"""MatMuls whose K is split over workgroups on streams of mi_stream_create: the memory in which they hand over their sums comes
and goes with the streams."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from mindspore_amd import kernels as K
from mindspore_amd import lib

pytestmark = pytest.mark.gpu

SPACE_BYTES = 1024 + 256 * 256 * (4 * 64 + 16)  # of a stream
ROWS, COLS, DEEP = 150, 1000, 4096              # K split in parts


@pytest.fixture
def matmul():
    """(the library, a MatMul, its input, what it gives)."""
    import torch
    from tests.test_gpu_dispatch_edges import _matmul_pair
    L = lib.init()
    rng = np.random.default_rng(3)
    kern = _matmul_pair(rng, COLS, DEEP, False, False)[4](True)
    a = torch.from_numpy(rng.integers(-128, 128, (ROWS, DEEP), dtype=np.int8)).cuda()
    with torch.cuda.stream(torch.cuda.Stream()):
        want = kern.run(a)  # on one piece of K
    torch.cuda.synchronize()
    before = _splits(L)
    assert torch.equal(kern.run(a), want) and _splits(L) == before + 1
    return L, kern, a, want


def _splits(L):
    return L.mi_debug_split_launches(None, None)


def _create(L):
    stream = C.c_void_p(None)
    assert L.mi_stream_create(C.byref(stream)) == lib.MI_OK
    return stream


def _destroy(L, streams):
    for stream in streams:
        assert L.mi_stream_destroy(stream) == lib.MI_OK


def _run(L, kern, a, stream, rows=ROWS, run="mi_matmul_run"):
    import torch
    out = torch.full((rows, COLS), 55, dtype=torch.int8, device="cuda")
    torch.cuda.synchronize()
    assert getattr(L, run)(kern._h, a.data_ptr(), rows, out.data_ptr(), stream) == lib.MI_OK
    return out


@pytest.mark.parametrize("memory", ["held", "made", "none"])
def test_runs_on_a_library_stream_allocate_nothing(matmul, memory):
    """What mi_matmul_reserve promises, also at the first MatMul with a split K on a stream: with memory that the library held for
    it, with memory made with it, and where there was none, so that K is not split."""
    import torch
    L, kern, a, want = matmul
    if memory == "none":
        L.mi_debug_fail_alloc(SPACE_BYTES)
    streams = [_create(L) for _ in range(1 if memory == "held" else 8)]
    assert L.mi_matmul_reserve(kern._h, ROWS) == lib.MI_OK
    _run(L, kern, a, streams[-1], rows=1)  # (what the runtime makes for a stream's first launch)
    out = torch.empty((ROWS, COLS), dtype=torch.int8, device="cuda")
    torch.equal(out, want)  # (and torch for a comparison)
    torch.cuda.synchronize()
    before, _ = torch.cuda.mem_get_info()
    split = _splits(L)
    try:
        for _ in range(3):
            out.fill_(55)
            torch.cuda.synchronize()
            assert L.mi_matmul_run(kern._h, a.data_ptr(), ROWS, out.data_ptr(), streams[-1]) == lib.MI_OK
            assert L.mi_stream_synchronize(streams[-1]) == lib.MI_OK
            assert torch.equal(out, want)
        assert torch.cuda.mem_get_info()[0] == before and _splits(L) == split + (0 if memory == "none" else 3)
    finally:
        L.mi_debug_fail_alloc(0)
    _destroy(L, streams)


def test_the_end_of_a_stream_does_not_wait_for_others(matmul):
    import torch
    L, kern, a, want = matmul
    streams = [_create(L) for _ in range(9)]
    for stream in streams:
        out = _run(L, kern, a, stream)
        assert L.mi_stream_synchronize(stream) == lib.MI_OK and torch.equal(out, want)
    busy, others = streams[0], streams[1:]
    rng = np.random.default_rng(1)
    n = 8192
    big = K.MatmulInt8Kernel(rng.integers(-128, 128, (n, n), dtype=np.int8), None, K.QuantParam(0.02, 7), [K.QuantParam(0.004, 0)],
                             K.QuantParam(1.0, 0), True, 0)
    x = torch.zeros((n, n), dtype=torch.int8, device="cuda")
    y = torch.empty((n, n), dtype=torch.int8, device="cuda")
    torch.cuda.synchronize()
    for _ in range(1000):  # about 0.3 s
        assert L.mi_matmul_run(big._h, x.data_ptr(), n, y.data_ptr(), busy) == lib.MI_OK
    still = torch.cuda.ExternalStream(busy.value)
    assert not still.query()
    _destroy(L, others)
    assert not still.query()
    assert L.mi_stream_synchronize(busy) == lib.MI_OK
    _destroy(L, [busy])


def test_streams_end_while_another_thread_captures(matmul):
    """The capture is not disturbed, and the streams' memory is given back with the last of them."""
    import threading
    import torch
    L, kern, a, want = matmul

    def session(count, ends):
        streams = [_create(L) for _ in range(count)]
        for stream in streams:
            out = _run(L, kern, a, stream)
            assert L.mi_stream_synchronize(stream) == lib.MI_OK and torch.equal(out, want)
        ends.append(streams)

    first = []
    session(10, first)  # (what the runtime keeps for ten streams)
    _destroy(L, first[0])
    torch.cuda.synchronize()
    before, _ = torch.cuda.mem_get_info()
    ends = []
    session(10, ends)
    failed = []

    def end():
        failed.extend(s for s in ends[0] if L.mi_stream_destroy(s) != lib.MI_OK)

    out = torch.empty((ROWS, COLS), dtype=torch.int8, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="global"):
        kern.run(a, out=out)
        thread = threading.Thread(target=end)
        thread.start()
        thread.join()
        kern.run(a, out=out)
    assert not failed
    for _ in range(3):
        out.fill_(55)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    assert torch.equal(kern.run(a), want)
    assert torch.cuda.mem_get_info()[0] >= before


def test_a_stream_made_after_another_takes_over_its_memory(matmul):
    """Again and again, the work of the stream before still on its way when its end is asked for: the sums start anew."""
    import torch
    L, kern, a, want = matmul
    held = [_create(L) for _ in range(7)]
    outs = []
    for _ in range(20):
        stream = _create(L)
        for _ in range(5):
            outs.append(torch.full((ROWS, COLS), 55, dtype=torch.int8, device="cuda"))
        torch.cuda.synchronize()
        split = _splits(L)
        for out in outs[-5:]:
            assert L.mi_matmul_run(kern._h, a.data_ptr(), ROWS, out.data_ptr(), stream) == lib.MI_OK
        assert _splits(L) == split + 5
        _destroy(L, [stream])
    torch.cuda.synchronize()
    assert all(torch.equal(out, want) for out in outs)
    _destroy(L, held)


def test_the_entry_point_that_allocates_nothing_splits_on_library_streams(matmul):
    import torch
    L, kern, a, want = matmul
    stream = _create(L)
    split = _splits(L)
    out = _run(L, kern, a, stream, run="mi_matmul_run_noalloc")
    assert L.mi_stream_synchronize(stream) == lib.MI_OK
    assert torch.equal(out, want) and _splits(L) == split + 1
    _destroy(L, [stream])


@pytest.mark.parametrize("run", ["mi_matmul_run", "mi_matmul_run_noalloc"])
def test_captures_of_a_library_stream_are_not_split(matmul, run):
    """Replays on another stream, beside the captured stream's own split launches: they share no memory."""
    import torch
    L, kern, a, want = matmul
    stream = _create(L)
    own = torch.cuda.ExternalStream(stream.value)
    outs = [torch.empty((ROWS, COLS), dtype=torch.int8, device="cuda") for _ in range(8)]
    call = lambda out: getattr(L, run)(kern._h, a.data_ptr(), ROWS, out.data_ptr(), stream)
    split = _splits(L)
    torch.cuda.synchronize()
    assert call(outs[0]) == lib.MI_OK and _splits(L) == split + 1
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=own):
        assert call(outs[1]) == lib.MI_OK and call(outs[2]) == lib.MI_OK
    assert _splits(L) == split + 1
    other = torch.cuda.Stream()
    for _ in range(20):
        for out in outs:
            out.fill_(55)
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            graph.replay()
        for out in outs[3:]:
            assert call(out) == lib.MI_OK
        torch.cuda.synchronize()
        assert all(torch.equal(out, want) for out in outs[1:])
    assert _splits(L) == split + 101
    _destroy(L, [stream])


FIRST_USE = """
import threading
import torch
from mindspore_amd import lib
x = torch.zeros(1000, device="cuda")
stream, graph, started = torch.cuda.Stream(), torch.cuda.CUDAGraph(), []
torch.cuda.synchronize()

def start():
    L = lib.init()
    started.append(L)
    stream = lib.C.c_void_p(None)
    assert L.mi_stream_create(lib.C.byref(stream)) == lib.MI_OK and L.mi_stream_destroy(stream) == lib.MI_OK

with torch.cuda.graph(graph, stream=stream, capture_error_mode="%s"):
    x.add_(1)
    thread = threading.Thread(target=start)
    thread.start()
    thread.join()
    x.add_(1)
for i in range(3):
    graph.replay()
    torch.cuda.synchronize()
    assert started and torch.equal(x, torch.full_like(x, 2 * i + 2))
import numpy as np
from mindspore_amd import kernels as K
w = np.ones((1000, 4096), np.int8)
kern = K.MatmulInt8Kernel(w, None, K.QuantParam(0.02, 0), [K.QuantParam(0.004, 0)], K.QuantParam(1.0, 0), True, 0)
y = kern.run(torch.ones((150, 4096), dtype=torch.int8, device="cuda"))
assert bool((y == 0).all()) and started[0].mi_debug_split_launches(None, None) == 1
print("ok")
"""


@pytest.mark.parametrize("mode", ["global", "relaxed"])
def test_the_first_use_of_the_library_beside_a_capture(mode):
    """Another thread's capture survives mi_init and the life of a stream, and K is split afterwards."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", FIRST_USE % mode], cwd=root, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.endswith("ok\n"), out.stdout + out.stderr[-2000:]
