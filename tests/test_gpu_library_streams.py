"""MatMuls whose K is split over workgroups on streams of mi_stream_create: the memory in which they hand over their sums comes
and goes with the streams."""
import ctypes as C

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
    assert torch.equal(kern.run(a), want)
    return L, kern, a, want


def _create(L):
    stream = C.c_void_p(None)
    assert L.mi_stream_create(C.byref(stream)) == lib.MI_OK
    return stream


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
    try:
        for _ in range(3):
            out.fill_(55)
            torch.cuda.synchronize()
            assert L.mi_matmul_run(kern._h, a.data_ptr(), ROWS, out.data_ptr(), streams[-1]) == lib.MI_OK
            assert L.mi_stream_synchronize(streams[-1]) == lib.MI_OK
            assert torch.equal(out, want)
        assert torch.cuda.mem_get_info()[0] == before
    finally:
        L.mi_debug_fail_alloc(0)
    for stream in streams:
        assert L.mi_stream_destroy(stream) == lib.MI_OK
