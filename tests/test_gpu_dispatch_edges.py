"""Sizes at the edges of the rules by which the library picks a kernel: the last size of one variant and the first of
the next, remainders, misaligned operands.  Full-tensor, bit-exact comparisons with the oracle."""
import re

import numpy as np
import pytest

from mindspore_amd import kernels as K

pytestmark = pytest.mark.gpu


def _last_kernel():
    """What this thread launched last: the kernel's name and its template's arguments."""
    symbol = K._lib.load().mi_debug_last_kernel().decode()
    length, rest = re.match(r"_ZN2mi(\d+)(.*)", symbol).groups()
    return rest[:int(length)], [int(v) for v in re.findall(r"L(?:[a-z]|NS_\d+[A-Za-z]+E)(\d+)E", rest[int(length):])]


def _values(rng, n):
    x = rng.standard_normal(n, dtype=np.float32)
    x[rng.integers(0, n, max(1, n // 100))] *= 50
    return x


@pytest.mark.parametrize("symmetric", [False, True])
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1024, 1027, 1028, 4096, 4100, 8195, 8196, 262144, 262147, 262148, 524288,
                               524292, 1048579, 1048580, 2097155, 2097156, 3145731, 3145732, 6291460, 8388612,
                               12582916, 16777220, 25165827, 25165828])
def test_dynamic_quant_one_launch_sizes(orc, n, symmetric):
    import torch
    rng = np.random.default_rng(n)
    x = _values(rng, n + 1)
    dev = torch.from_numpy(x).cuda()
    dq = K.DynamicQuantKernel(symmetric)
    for lead in (0, 1):  # 1: the tensor starts 4 bytes past a 16-byte boundary
        for repeat in range(2):  # the exchange between workgroups alternates between two halves of its slots
            q, p = dq.run(dev[lead:lead + n])
            want, scale, zp = orc.dynamic_quant(x[lead:lead + n], symmetric)
            assert np.array_equal(q.cpu().numpy(), want) and (p.scale, p.zero_point) == (scale, zp), (n, lead, repeat)


@pytest.mark.parametrize("special", [np.nan, np.inf, -np.inf, 0.0])
@pytest.mark.parametrize("n", [5, 40000, 3000001])
def test_dynamic_quant_one_launch_special_values(orc, n, special):
    import torch
    x = _values(np.random.default_rng(n), n)
    for where in ([0], [n - 1], list(range(n))):
        y = x.copy()
        y[where] = special
        dq = K.DynamicQuantKernel(False)
        q, p = dq.run(torch.from_numpy(y).cuda())
        want, scale, zp = orc.dynamic_quant(y)
        assert np.array_equal(q.cpu().numpy(), want), (n, special, where[:2])
        assert np.array_equal([p.scale], [scale], equal_nan=True) and p.zero_point == zp


@pytest.mark.parametrize("rows,unit", [(1, 1), (3, 255), (511, 259), (512, 259), (512, 260), (600, 515), (513, 771), (700, 1027),
                                       (255, 1028), (256, 1028), (300, 2051), (257, 3075), (256, 4099), (20, 4100), (7, 8195),
                                       (5, 8196), (3, 12292), (2, 16387), (2, 16388), (2, 65539), (2, 65540)])
def test_dynamic_quant_row_sizes(orc, rows, unit):
    import torch
    x = _values(np.random.default_rng(rows * unit), rows * unit).reshape(rows, unit)
    dq = K.DynamicQuantKernel(True)
    q, params = dq.run_rows(torch.from_numpy(x).cuda())
    want, scales, zps = orc.dynamic_quant_segments(x, True)
    got = params.cpu().numpy().view([("scale", "f8"), ("scale_f", "f4"), ("zp", "i4"), ("lo", "f4"), ("hi", "f4")])
    assert np.array_equal(q.cpu().numpy(), want)
    assert np.array_equal(got["scale"], scales) and np.array_equal(got["zp"], zps)


def test_dynamic_quant_parameters_follow_their_run(orc):
    """Parameters fetched run after run, after runs whose parameters nobody asked for, and from a stream that is being
    replayed as a graph: always those of the last run."""
    import torch
    rng = np.random.default_rng(3)
    xs = [_values(rng, n) * s for n, s in ((5000, 1.0), (40000, 3.0), (200000, 0.2), (26000000, 2.0), (700, 9.0))]
    devs = [torch.from_numpy(x).cuda() for x in xs]
    want = [orc.dynamic_quant(x)[1:] for x in xs]
    dq = K.DynamicQuantKernel(False)
    for fetch in (1, 1, 0, 1, 0, 0, 1, 1):
        for x, w in zip(devs, want):
            q, p = dq.run(x, fetch_params=bool(fetch))
            assert not fetch or (p.scale, p.zero_point) == w
    lib, p = K._lib, K._lib.DqParams()
    L = lib.load()
    side = torch.cuda.Stream()
    x = torch.empty_like(devs[1])
    with torch.cuda.stream(side):
        x.copy_(devs[1])
        dq.run(x)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            dq.run(x, fetch_params=False)
        for scale in (1.0, 2.0, 0.5, 4.0):
            x.copy_(devs[1] * scale)
            graph.replay()
            for fetch in (L.mi_dynquant_get_params, L.mi_dynquant_await_params):
                assert fetch(dq._h, side.cuda_stream, p) == lib.MI_OK
                assert (p.scale, p.zero_point) == orc.dynamic_quant(xs[1] * np.float32(scale))[1:]
        dq.run(devs[0])


@pytest.mark.parametrize("kernel,ic,oc", [((7, 7), 3, 64), ((5, 5), 3, 33), ((3, 3), 3, 32), ((3, 3), 5, 65), ((1, 1), 24, 130),
                                          ((5, 3), 10, 6), ((3, 8), 4, 31), ((16, 1), 16 + 1, 40), ((8, 4), 8, 64),
                                          ((9, 2), 16 - 1, 68), ((17, 3), 3, 36), ((4, 4), 8, 96), ((3, 11), 3, 32)])
@pytest.mark.parametrize("asymmetric", [False, True])
def test_first_layer_convolution_windows(orc, kernel, ic, oc, asymmetric):
    """One and two 16-byte chunks per window row, every remainder of the contraction steps, the first window rows the
    kernel does not take; images whose first and last bytes are inside padded windows."""
    import torch
    from oracle import pyoracle
    rng = np.random.default_rng(kernel[0] * 1000 + kernel[1] * 100 + ic)
    zp = rng.integers(-9, 10, oc).astype(np.int32) if asymmetric else np.zeros(oc, np.int32)
    w = rng.integers(-128, 128, (oc, *kernel, ic), dtype=np.int8)
    sw = rng.uniform(0.001, 0.01, oc).astype(np.float32).astype(np.float64)
    bias = rng.integers(-2000, 2001, oc).astype(np.int32)
    for (ih, iw), stride, pad in (((kernel[0], kernel[1]), (1, 1), (0, 0, 0, 0)), ((21, 19), (1, 2), (3, 2, 4, 1)),
                                  ((40, 35), (2, 1), (kernel[0] // 2, kernel[0] // 2, kernel[1] // 2, kernel[1] // 2))):
        x = rng.integers(-128, 128, (2, ih, iw, ic), dtype=np.int8)
        shape = pyoracle.conv_shape(2, ih, iw, ic, oc, kernel, stride, (1, 1), pad)
        conv = K.ConvolutionInt8Kernel(w, bias, K.QuantParam(0.02, 4), [K.QuantParam(float(s), int(z)) for s, z in zip(sw, zp)],
                                       K.QuantParam(0.2, -6), stride, (1, 1), pad, 1, K.ACT_RELU, exact_3x3=True)
        want = orc.conv_int8(x, w, bias, shape, 0.02, 4, sw, zp, 0.2, -6, K.ACT_RELU)
        assert np.array_equal(conv.run(torch.from_numpy(x).cuda()).cpu().numpy(), want), (kernel, ic, oc, ih, iw)
        flat = torch.zeros(x.size + 3, dtype=torch.int8, device="cuda")  # an image at an odd address
        flat[3:] = torch.from_numpy(x.reshape(-1)).cuda()
        assert np.array_equal(conv.run(flat[3:].view(x.shape)).cpu().numpy(), want), (kernel, ic, oc, ih, iw)


@pytest.mark.parametrize("kernel,ic,oc", [((7, 7), 3, 64), ((7, 7), 3, 33), ((3, 3), 3, 32), ((5, 5), 3, 40), ((4, 3), 10, 64)])
@pytest.mark.parametrize("h,w,stride,pad,batch", [(7, 102, (1, 1), 0, 2), (9, 139, (1, 2), 0, 1), (13, 150, (2, 2), 2, 3),
                                                  (11, 64 + 6, (3, 1), 1, 5), (70, 71, (1, 1), 3, 1)])
def test_first_layer_convolution_long_rows(orc, kernel, ic, oc, h, w, stride, pad, batch):
    """Output rows longer than a tile of 32 pixels: tiles wholly inside the image, up to the last bytes of the tensor."""
    import torch
    from oracle import pyoracle
    rng = np.random.default_rng(h * w + kernel[1])
    x = rng.integers(-128, 128, (batch, h, w, ic), dtype=np.int8)
    wt = rng.integers(-128, 128, (oc, *kernel, ic), dtype=np.int8)
    sw = rng.uniform(0.001, 0.01, oc).astype(np.float32).astype(np.float64)
    bias, zp = rng.integers(-2000, 2001, oc).astype(np.int32), np.zeros(oc, np.int32)
    shape = pyoracle.conv_shape(batch, h, w, ic, oc, kernel, stride, (1, 1), (pad,) * 4)
    conv = K.ConvolutionInt8Kernel(wt, bias, K.QuantParam(0.02, 4), [K.QuantParam(float(s), 0) for s in sw], K.QuantParam(0.2, -6),
                                   stride, (1, 1), (pad,) * 4, 1, K.ACT_NONE, exact_3x3=True)
    want = orc.conv_int8(x, wt, bias, shape, 0.02, 4, sw, zp, 0.2, -6, K.ACT_NONE)
    assert np.array_equal(conv.run(torch.from_numpy(x).cuda()).cpu().numpy(), want)


# 1x1 into more than 32 MB: both groups of 64 or 96 channels by one wave; whole groups, a last quad, a last byte; one to four steps of K, each
# with both kinds of group, odd rows, a last tile of pixels that is partly there
@pytest.mark.parametrize("pixels,k,n", [((17, 103, 115), 24, 192), ((1, 500, 560), 40, 120), ((3, 300, 331), 33, 113), ((1, 479, 501), 100, 144),
                                        ((2, 401, 299), 128, 161), ((1, 539, 541), 20, 116), ((2, 311, 301), 48, 180), ((1, 571, 569), 72, 104),
                                        ((3, 257, 233), 96, 192), ((1, 523, 523), 120, 125)])
@pytest.mark.parametrize("act", [K.ACT_NONE, K.ACT_RELU6])
def test_convolution_1x1_into_large_images(orc, pixels, k, n, act):
    import torch
    from oracle import pyoracle
    rng = np.random.default_rng(n)
    w = rng.integers(-128, 128, (n, 1, 1, k), dtype=np.int8)
    sw = rng.uniform(0.001, 0.01, n).astype(np.float32).astype(np.float64)
    bias, zp = rng.integers(-2000, 2001, n).astype(np.int32), np.zeros(n, np.int32)
    x = rng.integers(-128, 128, (*pixels, k), dtype=np.int8)
    assert x.size // k * n > 32 << 20
    so = float(np.float32(0.02 * 0.0055 * k ** 0.5 * 150))
    conv = K.ConvolutionInt8Kernel(w, bias, K.QuantParam(0.02, 4), [K.QuantParam(float(s), 0) for s in sw], K.QuantParam(so, -6), (1, 1), (1, 1),
                                   (0, 0, 0, 0), 1, act, exact_3x3=True)
    got = conv.run(torch.from_numpy(x).cuda()).cpu().numpy().reshape(-1, n)
    kernel, form = _last_kernel()
    assert kernel == "conv_thin_kernel" and form[:2] + form[3:] == [(k + 31) // 32, 3 if n > 128 else 2, 1, 2]
    some = np.unique(np.r_[np.arange(64), rng.integers(0, len(got), 20000), np.arange(len(got) - 64, len(got))])
    shape = pyoracle.conv_shape(1, 1, some.size, k, n, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0))
    orc.set_threads(16)
    want = orc.conv_int8(np.ascontiguousarray(x.reshape(-1, k)[some]).reshape(1, 1, some.size, k), w, bias, shape, 0.02, 4, sw, zp, so, -6, act)
    assert np.array_equal(got[some], want.reshape(-1, n))


# windows in LDS against 65 to 128 channels: three blocks of 32 and four, the last of them full or not; strides, dilations and uneven pads; a
# rectangle that fills the LDS (64 -> 128, stride 2).  Not on windows: fewer rectangles than the rule's least, and one round more than the GEMM's,
# of three blocks and of four; few rectangles of a first layer; four blocks with ragged stores; more pixels than the taps read
@pytest.mark.parametrize("b,ih,iw,ic,oc,taps,stride,dil,pad,windows", [
    (2, 170, 166, 16, 65, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), True), (8, 56, 56, 32, 96, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), True),
    (24, 56, 50, 16, 97, (3, 3), (1, 1), (1, 1), (0, 2, 1, 0), False), (20, 56, 50, 64, 97, (3, 3), (1, 1), (1, 1), (0, 2, 1, 0), True), (60, 29, 31, 32, 128, (2, 3), (1, 1), (1, 2), (1, 0, 2, 1), True),
    (50, 56, 56, 64, 128, (3, 3), (2, 2), (1, 1), (1, 1, 1, 1), True), (30, 60, 61, 48, 96, (3, 3), (2, 2), (1, 1), (1, 1, 1, 1), True),
    (7, 56, 56, 96, 90, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), True), (19, 56, 56, 16, 80, (3, 5), (1, 1), (2, 1), (2, 2, 2, 2), True),
    (2, 224, 224, 3, 96, (7, 7), (2, 2), (1, 1), (3, 3, 3, 3), True), (2, 220, 227, 3, 128, (7, 7), (2, 2), (1, 1), (3, 2, 3, 2), True),
    (1, 170, 163, 4, 70, (5, 5), (1, 1), (1, 1), (2, 2, 2, 2), True), (2, 113, 120, 3, 101, (9, 3), (1, 1), (2, 1), (4, 4, 1, 1), False), (4, 113, 120, 3, 101, (9, 3), (1, 1), (2, 1), (4, 4, 1, 1), True),
    (6, 56, 56, 32, 96, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), False), (11, 56, 56, 64, 128, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), False),
    (19, 56, 56, 96, 96, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), False), (19, 56, 56, 64, 128, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), False),
    (1, 224, 224, 3, 96, (7, 7), (2, 2), (1, 1), (3, 3, 3, 3), False),
    # rectangles of more pixels than the taps read: too few, in two rounds, far more; and in one round, and where two have a CU
    (67, 40, 40, 128, 96, (1, 2), (2, 2), (1, 1), (0, 0, 1, 1), False), (23, 112, 112, 64, 80, (1, 3), (2, 2), (1, 1), (0, 0, 1, 1), False),
    (96, 28, 28, 64, 96, (5, 1), (2, 2), (1, 1), (2, 2, 0, 0), False), (96, 56, 56, 64, 96, (3, 1), (3, 3), (1, 1), (1, 1, 0, 0), False),
    (57, 56, 56, 80, 96, (3, 1), (2, 2), (1, 1), (1, 1, 0, 0), True), (96, 56, 56, 16, 96, (1, 2), (2, 2), (1, 1), (0, 0, 1, 1), True)])
@pytest.mark.parametrize("act", [K.ACT_NONE, K.ACT_RELU])
def test_convolution_windows_of_more_channels(orc, b, ih, iw, ic, oc, taps, stride, dil, pad, windows, act):
    import torch
    from oracle import pyoracle
    rng = np.random.default_rng(oc * 100 + ic)
    w = rng.integers(-128, 128, (oc, *taps, ic), dtype=np.int8)
    sw = rng.uniform(0.001, 0.01, oc).astype(np.float32).astype(np.float64)
    bias, zp = rng.integers(-2000, 2001, oc).astype(np.int32), np.zeros(oc, np.int32)
    x = rng.integers(-128, 128, (b, ih, iw, ic), dtype=np.int8)
    shape = pyoracle.conv_shape(b, ih, iw, ic, oc, taps, stride, dil, pad)
    so = float(np.float32(0.02 * 0.0055 * (taps[0] * taps[1] * ic) ** 0.5 * 150))
    conv = K.ConvolutionInt8Kernel(w, bias, K.QuantParam(0.02, 4), [K.QuantParam(float(s), 0) for s in sw], K.QuantParam(so, -6), stride, dil,
                                   pad, 1, act, exact_3x3=True)
    orc.set_threads(16)
    want = orc.conv_int8(x, w, bias, shape, 0.02, 4, sw, zp, so, -6, act)
    got = conv.run(torch.from_numpy(x).cuda())
    kernel, form = _last_kernel()
    assert (kernel == "conv_window_kernel") == windows and (not windows or form[:2] == [(oc + 31) // 32, ic <= 4])
    assert np.array_equal(got.cpu().numpy(), want)
    assert torch.equal(conv.run(torch.from_numpy(x).cuda()), got)


@pytest.mark.parametrize("ic,oc,stride", [(64, 64, 1), (32, 96, 1), (64, 128, 2)])
def test_convolution_without_memory_for_its_window_weights(orc, ic, oc, stride):
    """They are a second copy: the handle is created without, and images run on the kernels that read the others."""
    import torch
    from mindspore_amd import lib
    from oracle import pyoracle
    rng = np.random.default_rng(oc)
    w = rng.integers(-128, 128, (oc, 3, 3, ic), dtype=np.int8)
    sw = rng.uniform(0.001, 0.01, oc).astype(np.float32).astype(np.float64)
    bias, zp = rng.integers(-2000, 2001, oc).astype(np.int32), np.zeros(oc, np.int32)
    x = rng.integers(-128, 128, (48, 56, 56, ic), dtype=np.int8)
    so = float(np.float32(0.02 * 0.0055 * (9 * ic) ** 0.5 * 150))
    make = lambda: K.ConvolutionInt8Kernel(w, bias, K.QuantParam(0.02, 4), [K.QuantParam(float(s), 0) for s in sw], K.QuantParam(so, -6),
                                           (stride, stride), (1, 1), (1, 1, 1, 1), 1, K.ACT_NONE, exact_3x3=True)
    L = lib.init(0)
    assert L.mi_debug_fail_alloc((oc + 31) // 32 * (9 * ic // 32) * 1024 + 16) == 0
    try:
        conv = make()
    finally:
        L.mi_debug_fail_alloc(0)
    orc.set_threads(16)
    want = orc.conv_int8(x, w, bias, pyoracle.conv_shape(48, 56, 56, ic, oc, (3, 3), (stride, stride), (1, 1), (1, 1, 1, 1)),
                         0.02, 4, sw, zp, so, -6, K.ACT_NONE)
    for c in (conv, make()):
        assert np.array_equal(c.run(torch.from_numpy(x).cuda()).cpu().numpy(), want)


def _matmul_pair(rng, n, k, asymmetric, dynamic, **kw):
    w = rng.integers(-128, 128, (n, k), dtype=np.int8)
    sw = rng.uniform(0.001, 0.01, n).astype(np.float32).astype(np.float64)
    zw = rng.integers(-9, 10, n) if asymmetric else np.zeros(n, np.int64)
    if dynamic:
        zw[:] = zw[0]
    qp = [K.QuantParam(float(s), int(z)) for s, z in zip(sw, zw)]
    if dynamic:
        bias = rng.standard_normal(n).astype(np.float32)
        make = lambda pack: K.MatmulDynamicInt8Kernel(w, bias, qp, decode_pack=pack)
    else:
        bias = rng.integers(-5000, 5001, n).astype(np.int32)
        make = lambda pack: K.MatmulInt8Kernel(w, bias, K.QuantParam(0.02, 7), qp,
                                               K.QuantParam(float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3), decode_pack=pack)
    return w, bias, sw, zw.astype(np.int32), make


# the rule picks, in this order: 64 x 64 (one K block), 32 x 32 (0: gemm_short.hip; two K blocks and more), 64 x 128, 128 x 128, 192 x 128 (the
# last tile reaches past the packed weights), 128 x 256, 256 x 128, 192 x 256, 256 x 256 tiles, and again 64 x 64 (two K blocks, more than the
# ring is deep).  tile: 10 x channels / 64 + rows / 64
@pytest.mark.parametrize("m,n,k,tile", [(65, 250, 128, 11), (65, 250, 144, 0), (130, 200, 1040, 0), (129, 257, 1000, 0), (700, 2100, 160, 12),
                                        (700, 2101, 1025, 12), (1000, 2500, 176, 22), (1000, 2503, 1040, 22), (513, 9003, 1040, 32),
                                        (1100, 6001, 1040, 24), (300, 21000, 1040, 42), (1201, 8302, 1100, 34), (1500, 9000, 1030, 44),
                                        (700, 1100, 144, 11), (300, 1700, 1040, 11), (200, 3000, 1552, 11)])
@pytest.mark.parametrize("dynamic,asymmetric", [(False, False), (False, True), (True, False), (True, True)])
def test_matmul_tile_shapes(orc, m, n, k, tile, dynamic, asymmetric):
    """Against the oracle where that takes seconds at most, against the row-major kernels (which have tests of their own)
    everywhere."""
    import torch
    rng = np.random.default_rng(m + n + k)
    w, bias, sw, zw, make = _matmul_pair(rng, n, k, asymmetric, dynamic)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    dev = torch.from_numpy(a).cuda()
    args = dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
    got = make(True).run(dev, **args).cpu().numpy()
    kernel, form = _last_kernel()
    if tile == 0:
        assert kernel == "gemm_short_kernel"
    else:
        assert kernel in ("gemm_ring_kernel", "gemm_kblock_kernel") and form[:2] == [tile // 10, tile % 10]
    assert np.array_equal(got, make(False).run(dev, **args).cpu().numpy())
    if m * n * k < 2e9:
        orc.set_threads(16)
        if dynamic:
            want = orc.dynamic_matmul(a, w, bias, 0.03, -5, sw, zw)
        else:
            want = orc.matmul_int8(a, w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3)
        assert np.array_equal(got, want)


# groups on 64 x 64 (a member of one channel, rows to be padded), 64 x 128, 128 x 128, 192 x 128, 128 x 256, 256 x 128,
# 256 x 256 and 192 x 256 tiles, a pair that gains nothing by one launch, pairs of 128 x 128 tiles
@pytest.mark.parametrize("m,k,ns", [(65, 1024, (65, 1, 200)), (130, 1030, (500, 131)), (70, 1024, (9000, 4100)),
                                    (300, 1024, (5000, 5000)), (257, 1030, (12000, 3001)), (500, 1024, (8192, 8000)),
                                    (300, 1024, (6000, 6000, 6000)), (700, 1024, (11008, 11008)), (513, 1040, (8200, 8201)),
                                    (1030, 2048, (9000, 9000)), (1878, 4320, (3929, 349))])
@pytest.mark.parametrize("how", ["static", "value", "rows"])
def test_matmul_group_on_tiles(orc, m, k, ns, how):
    """A group's launch against a launch per member (whose tiles have tests of their own), and the smallest against the oracle."""
    import torch
    rng = np.random.default_rng(m + k + sum(ns))
    members = [_matmul_pair(rng, n, k, False, how != "static") for n in ns]
    kernels = [make(True) for *_, make in members]
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    dev, args = torch.from_numpy(a).cuda(), {}
    if how == "value":
        args = dict(in_quant=K.QuantParam(0.03, -5))
    if how == "rows":
        dev, params = K.DynamicQuantKernel(True).run_rows(torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda())
        args = dict(row_params=params)
    outs = K.matmul_run_group(kernels, dev) if how == "static" else K.dynmm_run_group(kernels, dev, **args)
    for kern, y in zip(kernels, outs):
        assert torch.equal(y, kern.run(dev, **args))
    if m * k * sum(ns) < 2e8 and how != "rows":
        for (w, bias, sw, zw, _), y in zip(members, outs):
            want = (orc.dynamic_matmul(a, w, bias, 0.03, -5, sw, zw) if how == "value" else
                    orc.matmul_int8(a, w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3))
            assert np.array_equal(y.cpu().numpy(), want)


# members that are small products alone: one launch of 64 x 64 tiles as long as that is quicker than a launch each
@pytest.mark.parametrize("m,k,ns,together", [(65, 2048, (256, 256), True), (100, 2048, (64, 64), True), (128, 1024, (64, 64), True),
                                             (100, 4080, (64, 64), False), (64, 3072, (512, 512), False)])
@pytest.mark.parametrize("how", ["static", "value"])
def test_matmul_group_of_small_products(m, k, ns, together, how):
    import torch
    rng = np.random.default_rng(m + k + sum(ns))
    kernels = [_matmul_pair(rng, n, k, False, how != "static")[4](True) for n in ns]
    a = torch.from_numpy(rng.integers(-128, 128, (m, k), dtype=np.int8)).cuda()
    args = dict(in_quant=K.QuantParam(0.03, -5)) if how == "value" else {}
    want = [kern.run(a, **args) for kern in kernels]
    assert _last_kernel()[0] == "gemm_short_kernel"
    got = K.matmul_run_group(kernels, a) if how == "static" else K.dynmm_run_group(kernels, a, **args)
    assert ("_group_" in _last_kernel()[0]) == together
    assert all(torch.equal(x, y) for x, y in zip(got, want))


# ragged rows: members that read them as they are, alone, in pairs and beside one that needs the copy (decode-sized; on tiles of
# another size); a copy for three and more; one launch on a copy
@pytest.mark.parametrize("m,k,ns,copies", [(333, 1000, (1001,), False), (333, 1000, (1001, 1000), False), (70, 500, (65, 260), False),
                                           (40, 500, (4100, 300), True), (600, 1000, (100, 3000), True), (200, 770, (768, 768, 768), True),
                                           (333, 1400, (1000, 1000), True), (100, 200, (30, 30, 30, 30, 30), True)])
@pytest.mark.parametrize("how", ["static", "value", "rows"])
def test_matmul_group_on_ragged_rows(m, k, ns, copies, how):
    """Against a call per member, with and without the room for a padded copy of the rows."""
    import torch
    rng = np.random.default_rng(m + k + sum(ns))
    a = torch.from_numpy(rng.integers(-128, 128, (m, k), dtype=np.int8)).cuda()
    args = dict(in_quant=K.QuantParam(0.03, -5)) if how == "value" else {}
    if how == "rows":
        a, params = K.DynamicQuantKernel(True).run_rows(torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).cuda())
        args = dict(row_params=params)
    make = lambda: [_matmul_pair(np.random.default_rng(n), n, k, False, how != "static")[4](True) for n in ns]
    run = lambda kernels: K.matmul_run_group(kernels, a) if how == "static" else K.dynmm_run_group(kernels, a, **args)
    want = [kern.run(a, **args) for kern in make()]
    for kernels in (make(), make()):
        for _ in range(2):
            assert all(torch.equal(x, y) for x, y in zip(run(kernels), want))
    L, kernels = K._lib.load(), make()
    assert L.mi_debug_fail_alloc(m * ((k + 15) // 16 * 16)) == 0
    try:
        if copies:
            with pytest.raises(K._lib.MiError) as e:
                run(kernels)
            assert e.value.code == K._lib.MI_MEMORY_FAILED
        else:
            assert all(torch.equal(x, y) for x, y in zip(run(kernels), want))
    finally:
        L.mi_debug_fail_alloc(0)


# both sides of each line between few ragged rows as they are and on a copy: rows x K up to 16 rows against few channels, 4097 to
# 8191 channels, more than 16 rows, more than 48
@pytest.mark.parametrize("m,k,n,copies", [(8, 13007, 33, False), (16, 8191, 33, False), (16, 8193, 33, True), (9, 14563, 33, False),
                                          (9, 14565, 33, True), (8, 501, 4100, False), (9, 501, 4096, False), (9, 501, 4097, True),
                                          (16, 4001, 8191, True), (16, 4001, 8192, False), (16, 4097, 8192, True), (17, 501, 4097, False),
                                          (17, 3071, 4097, False), (17, 3073, 4097, True), (32, 4095, 8192, False), (32, 4097, 33, True),
                                          (48, 4095, 33, False), (49, 2559, 33, False), (49, 2561, 33, True)])
@pytest.mark.parametrize("dynamic", [False, True])
def test_matmul_few_ragged_rows_copied_or_not(orc, m, k, n, copies, dynamic):
    import torch
    L = K._lib.init()
    rng = np.random.default_rng(n + k)
    w, bias, sw, zw, make = _matmul_pair(rng, n, k, True, dynamic)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    dev, args = torch.from_numpy(a).cuda(), dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
    kern = make(True)
    assert L.mi_debug_fail_alloc(m * ((k + 15) // 16 * 16)) == 0
    try:
        if copies:
            with pytest.raises(K._lib.MiError) as e:
                kern.run(dev, **args)
            assert e.value.code == K._lib.MI_MEMORY_FAILED
        else:
            kern.run(dev, **args)
    finally:
        L.mi_debug_fail_alloc(0)
    orc.set_threads(16)
    if dynamic:
        want = orc.dynamic_matmul(a, w, bias, 0.03, -5, sw, zw)
    else:
        want = orc.matmul_int8(a, w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3)
    assert np.array_equal(kern.run(dev, **args).cpu().numpy(), want)


# a group of one on the decode kernels: one row, few, more than go out as one launch; rows shorter than a chunk, and too many long
# ones, are copied as they are for the member alone
@pytest.mark.parametrize("m,k,n,copies", [(1, 1001, 300, False), (8, 11009, 40, False), (16, 1001, 300, False), (33, 250, 300, False),
                                          (64, 1001, 768, False), (5, 9, 300, True), (64, 8003, 300, True)])
@pytest.mark.parametrize("how", ["static", "value"])
def test_matmul_group_of_one_on_few_ragged_rows(m, k, n, copies, how):
    """As the member alone, with and without the room for a padded copy of the rows."""
    import torch
    L = K._lib.init()
    a = torch.from_numpy(np.random.default_rng(k).integers(-128, 128, (m, k), dtype=np.int8)).cuda()
    args = dict(in_quant=K.QuantParam(0.03, -5)) if how == "value" else {}
    make = lambda: _matmul_pair(np.random.default_rng(n), n, k, False, how != "static")[4](True)
    group = lambda kern: (K.matmul_run_group([kern], a) if how == "static" else K.dynmm_run_group([kern], a, **args))[0]
    want = make().run(a, **args)
    assert torch.equal(group(make()), want)
    alone, member = make(), make()
    assert L.mi_debug_fail_alloc(m * ((k + 15) // 16 * 16)) == 0
    try:
        for run in (lambda: alone.run(a, **args), lambda: group(member)):
            if copies:
                with pytest.raises(K._lib.MiError) as e:
                    run()
                assert e.value.code == K._lib.MI_MEMORY_FAILED
            else:
                assert torch.equal(run(), want)
    finally:
        L.mi_debug_fail_alloc(0)


# small products, whose K the waves of a workgroup share: two K blocks (half the waves have none), the last with one byte, a chunk and all but
# one; up to 12 blocks and beyond (four and eight waves), 64 channels x 32 rows, one tile past 256 of each kind (tile 0: another kernel); last
# rows and channels that are partly there.  tile: 10 x waves + blocks of 32 channels; copied: odd rows come as whole chunks of a padded copy; None:
# only odd rows run here, and whole chunks of int8 on another kernel
@pytest.mark.parametrize("m,n,k,tile,copied", [
    (3, 1, 129, 41, False), (32, 31, 144, 41, False), (33, 65, 255, 41, False), (64, 4095, 256, 41, False), (65, 2700, 257, 41, False),
    (95, 96, 1535, 41, False), (97, 33, 1537, 81, False), (64, 100, 1536, 41, False), (40, 4096, 1552, 81, False), (130, 1600, 1040, 41, False),
    (257, 1793, 897, 0, False), (256, 2048, 896, 82, False), (129, 2, 4095, 81, False), (70, 300, 4080, 81, False), (60, 700, 4113, 81, True),
    (500, 520, 300, 41, False), (33, 1001, 9001, 81, True), (4, 24576, 768, 41, False), (16, 8192, 1024, 41, False), (17, 8193, 1024, 0, False),
    (16, 7168, 1536, 41, True), (32, 8192, 1536, 41, False),
    # up to 32 rows, both sides of the lines at 4, 8 and 16 rows and at 768, 2048, 4096, 8192 and 12288 channels
    (4, 2048, 512, 41, False), (4, 2048, 513, 0, False), (4, 2049, 384, 41, False), (4, 2049, 385, 0, False), (4, 4097, 896, 41, False),
    (4, 4097, 897, 0, False), (3, 8192, 384, 41, False), (3, 12288, 400, 0, False), (3, 12289, 400, 41, False), (5, 2048, 768, 41, False),
    (8, 2048, 769, 0, False), (8, 2049, 640, 41, False), (8, 4096, 641, 0, False), (8, 4097, 1536, 41, False), (8, 8192, 656, 0, False),
    (9, 768, 1536, 41, False), (16, 769, 1024, 41, False), (9, 769, 1025, 0, False), (32, 4096, 1040, 0, False), (32, 4097, 1536, 41, False),
    (17, 8191, 1041, 41, False),
    # five row tiles that nearly fill the device, and on the other side of that line
    (160, 2817, 1280, 82, None), (129, 3200, 2560, 82, None), (160, 2816, 1280, 82, False), (129, 3200, 2576, 82, False)])
@pytest.mark.parametrize("dynamic,asymmetric", [(False, False), (False, True), (True, False), (True, True)])
def test_matmul_small_products(orc, m, n, k, tile, copied, dynamic, asymmetric):
    """Against the oracle, bit by bit (integer sums, then a fixed sequence of rounded steps): rows at an aligned and at an odd address,
    in the middle of larger ones' bytes, which must not count; and with a scale per row."""
    import torch
    rng = np.random.default_rng(m + n + k)
    w, bias, sw, zw, make = _matmul_pair(rng, n, k, asymmetric, dynamic)
    kern, a = make(True), rng.integers(-128, 128, (m, k), dtype=np.int8)
    args = dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
    orc.set_threads(16)
    if dynamic:
        want = orc.dynamic_matmul(a, w, bias, 0.03, -5, sw, zw)
    else:
        want = orc.matmul_int8(a, w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3)
    for before in (0, 16, 1, 11):
        flat = torch.full((before + m * k + 64,), 99, dtype=torch.int8, device="cuda")
        flat[before:before + m * k] = torch.from_numpy(a.reshape(-1)).cuda()
        rows = flat[before:before + m * k].view(m, k)
        got = kern.run(rows, **args).cpu().numpy()
        kernel, form = _last_kernel()
        odd = (rows.data_ptr() | k) % 16 != 0
        here = tile != 0 and (copied is not None or odd or dynamic)
        assert (kernel == "gemm_short_kernel") == here
        if here:
            assert form[:2] + form[-1:] == [tile // 10, tile % 10, odd and not copied], before
        assert np.array_equal(got.view(np.int8), want.view(np.int8)), before
    if dynamic:
        x = rng.standard_normal((m, k)).astype(np.float32)
        q, params = K.DynamicQuantKernel(True).run_rows(torch.from_numpy(x).cuda())
        q_want, scale, zp = orc.dynamic_quant_segments(x, True)
        sure = orc.dynamic_matmul_rows(q_want, w, bias, scale.astype(np.float32), int(zp[0]), sw, zw)
        assert np.array_equal(kern.run(q, row_params=params).cpu().numpy().view(np.int8), sure.view(np.int8))


@pytest.mark.parametrize("taps", [3, 5])
@pytest.mark.parametrize("b,ih,iw,ch,pad", [(1, 5, 5, 4, (0, 0, 0, 0)), (1, 5, 6, 8, (1, 1, 1, 1)), (2, 7, 9, 12, (2, 0, 0, 2)),
                                            (1, 9, 11, 20, (4, 4, 4, 4)), (3, 6, 8, 192, (1, 2, 3, 0)), (1, 33, 31, 36, (1, 1, 1, 1)),
                                            (4, 61, 53, 192, (1, 1, 1, 1)), (9, 70, 127, 96, (2, 2, 2, 2)),
                                            (16, 75, 77, 192, (1, 1, 1, 1))])
def test_depthwise_stride_one_tiles(orc, b, ih, iw, ch, pad, taps):
    """Partial tiles on either side, windows that reach over every border, one, two and four output rows per thread."""
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(ih * iw + taps)
    orc.set_threads(16)
    for act in (0, 3):
        case = _conv_case(rng, b, ih, iw, ch, ch, (taps, taps), (1, 1), (1, 1), pad, True, False, True, act, dw=True)
        case["w"].reshape(ch, -1)[:2] = -128  # the largest products
        got = _gpu_conv(case, (1, 1), (1, 1), pad, ch, device_tensors=True)
        assert np.array_equal(got, orc.conv_dw_int8(**case)), act


@pytest.mark.parametrize("b,ih,iw,ic,oc", [(1, 12, 11, 1, 5),  # one byte of K, the tensor's end inside many loads
                                           (1, 13, 10, 15, 33), (2, 9, 9, 24, 144), (1, 40, 33, 32, 192), (3, 21, 19, 100, 31),
                                           (1, 30, 30, 240, 40), (1, 17, 17, 480, 256), (1, 13, 10, 1024, 64),
                                           (9, 130, 131, 16, 96)])  # several tiles per wave
def test_conv_1x1_few_channels(orc, b, ih, iw, ic, oc):
    """Contractions and channel counts around the batches of steps and the blocks of channels, with and without weight zero
    points, per-tensor and per-channel scales."""
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(ih * iw + oc)
    orc.set_threads(16)
    pad = (0, 0, 0, 0)
    for it in range(3):
        case = _conv_case(rng, b, ih, iw, ic, oc, (1, 1), (1, 1), (1, 1), pad, it != 1, it == 1, it != 2, [0, 1, 3][it])
        got = _gpu_conv(case, (1, 1), (1, 1), pad, 1, device_tensors=True)
        assert np.array_equal(got, orc.conv_int8(**case)), it


@pytest.mark.parametrize("b,ih,iw,ic,oc", [(1, 12, 11, 16, 7), (2, 31, 33, 48, 64), (1, 40, 41, 32, 65), (2, 91, 90, 16, 130),
                                           # rows of 128 pixels: 771, K = 144: 64 x 64 tiles, with up to 32 channels 64 x 256
                                           (8, 111, 111, 16, 64), (8, 111, 111, 16, 32),
                                           (8, 110, 111, 16, 33),  # 764: 64 x 64
                                           (8, 111, 111, 32, 64),  # 771, K = 288: 64 x 256
                                           (8, 128, 128, 32, 50), (8, 128, 129, 32, 50),  # 1024: 64 x 256; 1032: 64 x 64
                                           (4, 219, 219, 96, 37), (4, 221, 219, 96, 37)])  # 1499, 1513, K = 864: either side
def test_conv_gather_tiles(orc, b, ih, iw, ic, oc):
    """Either side of the rules by which the gathering GEMM picks its tile, with and without weight zero points."""
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(ih * iw + oc)
    orc.set_threads(16)
    pad = (1, 1, 1, 1)
    for it in range(2):
        case = _conv_case(rng, b, ih, iw, ic, oc, (3, 3), (1, 1), (1, 1), pad, True, it == 1, True, it)
        got = _gpu_conv(case, (1, 1), (1, 1), pad, 1, device_tensors=True, exact_3x3=True)
        assert np.array_equal(got, orc.conv_int8(**case)), it


def test_dynamic_quant_parameters_of_a_handle_first_run_under_capture(orc):
    """A handle whose very first run was captured: its graph may be replayed at any time, also between an eager run and
    the fetch that follows, and the fetch returns the parameters of whatever ran last."""
    import torch
    rng = np.random.default_rng(5)
    one, other = _values(rng, 40000), _values(rng, 5000) * 7
    other_dev = torch.from_numpy(other).cuda()
    lib, p = K._lib, K._lib.DqParams()
    L = lib.load()
    K.DynamicQuantKernel(False).run(torch.from_numpy(one).cuda())  # the kernels are loaded before the capture
    side = torch.cuda.Stream()
    x = torch.from_numpy(one).cuda()
    torch.cuda.synchronize()
    dq = K.DynamicQuantKernel(False)
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            dq.run(x, fetch_params=False)
        scale = np.float32(1.0)
        for fetch in (L.mi_dynquant_get_params, L.mi_dynquant_await_params):
            for eager_fetch in (None, False, True, False):
                if eager_fetch is not None:
                    _, q = dq.run(other_dev, fetch_params=eager_fetch)
                    assert not eager_fetch or (q.scale, q.zero_point) == orc.dynamic_quant(other)[1:]
                scale *= np.float32(1.5)
                x.copy_(torch.from_numpy(one * scale))
                graph.replay()
                assert fetch(dq._h, side.cuda_stream, p) == lib.MI_OK
                assert (p.scale, p.zero_point) == orc.dynamic_quant(one * scale)[1:], (fetch.__name__, eager_fetch)


@pytest.mark.parametrize("n,k,rows", [(201, 512, 8), (201, 512, 100), (1030, 4096, 300), (7, 48, 1)])
def test_first_run_of_odd_output_rows_under_capture(orc, n, k, rows):
    """Rows of a length the kernels store in place, from an aligned activation tensor: no run allocates, so the very first
    may be captured, and none leaves the handle holding memory."""
    import torch
    rng = np.random.default_rng(n + rows)
    orc.set_threads(16)
    w, bias, sw, zw, make = _matmul_pair(rng, n, k, False, False)
    make(True).run(torch.zeros((rows, k), dtype=torch.int8, device="cuda"))  # the kernels are loaded before the capture
    kern = make(True)
    a = torch.from_numpy(rng.integers(-128, 128, (rows, k), dtype=np.int8)).cuda()
    out = torch.zeros((rows, n), dtype=torch.int8, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            kern.run(a, out=out)
    for _ in range(3):
        a.copy_(torch.from_numpy(rng.integers(-128, 128, (rows, k), dtype=np.int8)))
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        want = orc.matmul_int8(a.cpu().numpy(), w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3)
        assert np.array_equal(out.cpu().numpy(), want)
        assert np.array_equal(kern.run(a).cpu().numpy(), want)
    many = (64 << 20) // k  # 64 MiB of activation rows
    a = torch.zeros((many, k), dtype=torch.int8, device="cuda")
    out = torch.zeros((many, n), dtype=torch.int8, device="cuda")
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    kern.run(a, out=out)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] < 32 << 20


@pytest.mark.parametrize("unfetched", [0, 2])
def test_dynamic_quant_parameters_do_not_wait_for_later_work(orc, unfetched):
    """The parameters of a run are known before the work that was queued behind it: for a new handle's first run, and for one
    whose first runs nobody asked about, from the run after its first fetch on."""
    import time
    import torch
    lib, p = K._lib, K._lib.DqParams()
    L = lib.load()
    x = _values(np.random.default_rng(8), 197 * 768)
    dev, big = torch.from_numpy(x).cuda(), torch.randn(4096, 4096, device="cuda")
    side = torch.cuda.Stream()
    K.DynamicQuantKernel(False).run(dev)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        big @ big
        dq = K.DynamicQuantKernel(False)
        for _ in range(unfetched):
            dq.run(dev, fetch_params=False)
        if unfetched:
            dq.run(dev)
        torch.cuda.synchronize()
        began = time.perf_counter()
        dq.run(dev, fetch_params=False)
        for _ in range(64):  # tens of milliseconds
            y = big @ big
        queued = time.perf_counter()
        assert L.mi_dynquant_await_params(dq._h, side.cuda_stream, p) == lib.MI_OK
        known = time.perf_counter()
        side.synchronize()
        done = time.perf_counter()
    assert (p.scale, p.zero_point) == orc.dynamic_quant(x)[1:]
    assert known - queued < 0.25 * (done - began), (queued - began, known - queued, done - began)


def test_dynamic_quant_runs_that_overlapped_spoil_no_later_run(orc):
    """Runs of one handle that overlap on two streams have unspecified results (every wait in the kernel is bounded); those
    that follow in order are right and wait for nobody."""
    import torch
    lib = K._lib
    L = lib.load()
    rng = np.random.default_rng(12)
    xs = [_values(rng, n) for n in (40000, 260000, 1200000, 9000)]
    devs = [torch.from_numpy(x).cuda() for x in xs]
    qs = [torch.empty(x.size, dtype=torch.int8, device="cuda") for x in xs]
    want = [orc.dynamic_quant(x) for x in xs]
    dq = K.DynamicQuantKernel(False)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()

    def run(i, stream):
        assert L.mi_dynquant_run(dq._h, devs[i].data_ptr(), xs[i].size, qs[i].data_ptr(), stream.cuda_stream) == lib.MI_OK

    for overlap in range(5):
        for it in range(20):
            run(it % 4, streams[0])
            run((it + 1 + overlap) % 4, streams[1])
        torch.cuda.synchronize()
        for i in range(4):
            qs[i].zero_()
        torch.cuda.synchronize()
        for i in range(4):
            run(i, streams[0])
        streams[0].synchronize()
        for i in range(4):
            assert np.array_equal(qs[i].cpu().numpy(), want[i][0]), (overlap, i)
        first, last = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        with torch.cuda.stream(streams[0]):
            first.record()
            for it in range(40):
                run(it % 4, streams[0])
            last.record()
        last.synchronize()
        assert first.elapsed_time(last) / 40 < 0.15, "ms per run; a workgroup that waits in vain takes 0.2"


def test_dynamic_quant_handles_by_the_hundred(orc):
    """More handles than one page of parameter notes holds, some destroyed and made again: each fetches its own parameters."""
    import torch
    x = _values(np.random.default_rng(2), 3000)
    dev = torch.from_numpy(x).cuda()
    want = {}
    handles = {}
    for turn in range(3):
        for i in range(130):
            if i % 3 == turn:
                handles.pop(i, None)
                handles[i] = K.DynamicQuantKernel(False)
            elif i not in handles:
                handles[i] = K.DynamicQuantKernel(True)
        for repeat in range(2):
            for i, dq in handles.items():
                n = 1000 + 10 * i
                key = (n, i % 3 <= turn)
                if key not in want:
                    want[key] = orc.dynamic_quant(x[:n], not key[1])[1:]
                _, p = dq.run(dev[:n])
                assert (p.scale, p.zero_point) == want[key], (turn, i)


@pytest.mark.parametrize("torch_is", ["none", "without HIP"])
def test_host_tensors_without_torch(orc, tmp_path, torch_is):
    from tests.test_abi_cpu import run_without_torch
    rng = np.random.default_rng(6)
    w, bias, sw, _, _ = _matmul_pair(rng, 40, 64, False, False)
    a, x = rng.integers(-128, 128, (9, 64), dtype=np.int8), _values(rng, 700)
    np.savez(tmp_path / "case.npz", w=w, bias=bias, sw=sw, a=a, x=x, want=orc.matmul_int8(a, w, bias, 0.02, 7, sw, np.zeros(40, np.int32), 0.5, 3),
             q=orc.dynamic_quant(x)[0])
    run_without_torch(tmp_path, torch_is, """
c = np.load("case.npz")
kern = K.MatmulInt8Kernel(c["w"], c["bias"], K.QuantParam(0.02, 7), [K.QuantParam(float(s), 0) for s in c["sw"]], K.QuantParam(0.5, 3))
assert np.array_equal(kern.run(c["a"]), c["want"])
assert np.array_equal(K.DynamicQuantKernel(False).run(c["x"])[0], c["q"])
""")


def test_dynamic_matmul_argument_forms(orc):
    """The input's quantisation as Python programs hold it: whole and floating zero points, device addresses as numbers and as
    ctypes pointers, for one kernel and for a group."""
    import ctypes as C
    import torch
    rng = np.random.default_rng(9)
    w, bias, sw, zw, make = _matmul_pair(rng, 48, 96, True, True)
    kern = make(True)
    x = _values(rng, 5 * 96).reshape(5, 96)
    dq = K.DynamicQuantKernel(False)
    q, p = dq.run(torch.from_numpy(x).cuda())
    want = orc.dynamic_matmul(q.cpu().numpy(), w, bias, p.scale, p.zero_point, sw, zw)

    def check(**args):
        for y in [kern.run(q, **args)] + K.dynmm_run_group([kern, kern], q, **args):
            assert np.array_equal(y.cpu().numpy().view(np.uint32), want.view(np.uint32)), args

    for scale in (p.scale, np.float64(p.scale), np.array(p.scale)):
        for zero_point in (p.zero_point, float(p.zero_point), np.float32(p.zero_point), np.int64(p.zero_point)):
            check(in_quant=K.QuantParam(scale, zero_point))
    addr = dq.device_params()
    for params in (addr, C.c_void_p(addr), C.cast(addr, C.POINTER(K._lib.DqParams))):
        check(params_dev=params)
    with pytest.raises((TypeError, C.ArgumentError)):
        kern.run(q, params_dev=1.5)


def test_dynamic_matmul_refuses_a_null_parameter_block():
    import ctypes as C
    import torch
    kern = K.MatmulDynamicInt8Kernel(np.ones((8, 16), np.int8), None, [K.QuantParam(0.1, 0)])
    q = torch.ones((2, 16), dtype=torch.int8, device="cuda")
    for null in (0, C.c_void_p(None)):
        with pytest.raises(K._lib.MiError) as e:
            kern.run(q, params_dev=null)
        assert e.value.code == K._lib.MI_NULL_PTR


@pytest.mark.parametrize("dynamic", [False, True])
def test_group_of_many_kernels(dynamic):
    import torch
    rng = np.random.default_rng(10)
    kernels = [_matmul_pair(rng, n, 32, False, dynamic)[4](True) for n in range(1, 101)]
    a = torch.from_numpy(rng.integers(-128, 128, (3, 32), dtype=np.int8)).cuda()
    args = dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
    outs = K.dynmm_run_group(kernels, a, **args) if dynamic else K.matmul_run_group(kernels, a)
    assert len(outs) == 100
    for kern, y in zip(kernels, outs):
        assert torch.equal(y, kern.run(a, **args))


@pytest.fixture
def host_slots():
    """Page-locked slots of both sizes for several callers at once: calls go without until they have lost the price of a set."""
    import threading
    rng = np.random.default_rng(78)
    work = [(_matmul_pair(rng, n, k, False, False)[4](True), rng.integers(-128, 128, (rows, k), dtype=np.int8))
            for rows, k, n in ((1000, 2000, 1500), (100, 300, 500)) * 6]

    def go(kern, a):
        for _ in range(80):
            kern.run(a)

    threads = [threading.Thread(target=go, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    yield  # (they stay while these kernels do)
    work.clear()


# one chunk, a last chunk of one byte, as many chunks as slots, slots used several times, on the way in, out and both
@pytest.mark.parametrize("rows,k,n", [(1, 1, 1), (3, 70001, 2), (65537, 1, 1), (517, 1000, 64), (2099, 1001, 5), (2100, 7, 1001),
                                      (3001, 1500, 1401)])
@pytest.mark.parametrize("slots", [False, True])
def test_host_tensors_in_and_out(request, rows, k, n, slots):
    """Against the same kernels on device tensors."""
    import torch
    if slots:
        request.getfixturevalue("host_slots")
    rng = np.random.default_rng(rows + k)
    a = rng.integers(-128, 128, (rows, k), dtype=np.int8)
    dev = torch.from_numpy(a).cuda()
    for dynamic in (False, True):
        kern = _matmul_pair(rng, n, k, False, dynamic)[4](True)
        args = dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
        want = kern.run(dev, **args).cpu().numpy()
        for _ in range(2):
            assert np.array_equal(kern.run(a, **args), want)
        locked = torch.from_numpy(a).pin_memory().numpy()  # goes past the slots
        assert np.array_equal(kern.run(locked, **args), want)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    for per_row in (False, True):
        dq = K.DynamicQuantKernel(per_row)
        there = dq.run_rows(torch.from_numpy(x).cuda())[0] if per_row else dq.run(torch.from_numpy(x).cuda())[0]
        assert np.array_equal(dq.run_rows(x)[0] if per_row else dq.run(x)[0], there.cpu().numpy())


@pytest.mark.parametrize("slots", [False, True])
def test_host_tensors_from_several_threads(request, slots):
    import threading
    import torch
    if slots:
        request.getfixturevalue("host_slots")
    rng = np.random.default_rng(77)
    work = []
    for rows, k, n in ((700, 900, 1100), (64, 64, 64), (1500, 2000, 300), (2000, 300, 2000), (1, 5, 9)):
        a = rng.integers(-128, 128, (rows, k), dtype=np.int8)
        kern = _matmul_pair(rng, n, k, False, False)[4](True)
        work.append((kern, a, kern.run(torch.from_numpy(a).cuda()).cpu().numpy()))
    bad = []

    def go(kern, a, want):
        for _ in range(6):
            if not np.array_equal(kern.run(a), want):
                bad.append(a.shape)

    threads = [threading.Thread(target=go, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


# rows of one block, of one set of four blocks, just into the next set, of three sets, the first that are padded; a chunk, a dword and a byte past a block;
# one tile and several, with rows and channels past their last one
@pytest.mark.parametrize("m,n,k", [(65, 20, 129), (64, 64, 511), (130, 257, 513), (333, 1001, 1000), (70, 260, 1535), (200, 31, 1291),
                                   (129, 65, 1537)])
@pytest.mark.parametrize("dynamic,asymmetric", [(False, False), (False, True), (True, False), (True, True)])
def test_matmul_rows_of_any_length(orc, m, n, k, dynamic, asymmetric):
    """Against the oracle, and at addresses that are no multiple of 16 against the aligned run; one of them with k % 16 == 0."""
    import torch
    rng = np.random.default_rng(m + n + k)
    orc.set_threads(16)
    for depth in (k, (k + 15) // 16 * 16):
        w, bias, sw, zw, make = _matmul_pair(rng, n, depth, asymmetric, dynamic)
        a = rng.integers(-128, 128, (m, depth), dtype=np.int8)
        kern, args = make(True), dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
        if dynamic:
            want = orc.dynamic_matmul(a, w, bias, 0.03, -5, sw, zw)
        else:
            want = orc.matmul_int8(a, w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * depth ** 0.5 * 140)), 3)
        for shift in (0, 1, 4, 15):
            flat = torch.zeros(a.size + shift, dtype=torch.int8, device="cuda")  # ends with the tensor's last byte
            flat[shift:] = torch.from_numpy(a.reshape(-1)).cuda()
            got = kern.run(flat[shift:].view(a.shape), **args).cpu().numpy()
            assert np.array_equal(got, want), (depth, shift)


# one chunk per pixel and five, odd and even numbers of contraction steps and fewer than the late loads' ones; three and four
# channels, one and two chunks per window row; rectangles that the image cuts off, channels that end inside a block and a quad;
# windows over every border, a stride and a dilation; with and without an activation
@pytest.mark.parametrize("ic,oc,kernel,stride,dilation,pad", [(64, 64, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),
                                                              (48, 37, (3, 3), (1, 1), (1, 1), (0, 2, 1, 0)),
                                                              (16, 32, (3, 3), (1, 2), (1, 1), (1, 1, 1, 1)),
                                                              (16, 7, (1, 3), (1, 1), (1, 1), (0, 0, 1, 1)),
                                                              (32, 64, (5, 5), (1, 1), (1, 1), (2, 2, 2, 2)),
                                                              (80, 33, (2, 3), (1, 1), (2, 1), (2, 0, 3, 1)),
                                                              (32, 20, (3, 3), (2, 2), (1, 3), (3, 1, 2, 4)),
                                                              (3, 64, (7, 7), (2, 2), (1, 1), (3, 3, 3, 3)),
                                                              (3, 21, (9, 3), (1, 1), (1, 1), (4, 4, 1, 1)),
                                                              (4, 42, (5, 8), (1, 2), (2, 1), (0, 4, 7, 2)),
                                                              (4, 32, (10, 4), (2, 1), (1, 1), (0, 1, 5, 0))])
@pytest.mark.parametrize("batch,h,w,act", [(16, 61, 53, 1), (5, 131, 90, 0), (208, 11, 19, 3), (3, 300, 67, 0), (171, 16, 16, 1)])
def test_window_convolution_rectangles(orc, ic, oc, kernel, stride, dilation, pad, batch, h, w, act):
    import torch
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(ic * oc + h)
    orc.set_threads(16)
    case = _conv_case(rng, batch, h, w, ic, oc, kernel, stride, dilation, pad, True, False, True, act)
    assert np.array_equal(_gpu_conv(case, stride, dilation, pad, 1, device_tensors=True, exact_3x3=True), orc.conv_int8(**case))


# rectangles of 77, 78 and 70 KiB of LDS, on three and four channels
@pytest.mark.parametrize("ic,kernel,stride,batch,size", [(3, (8, 8), (8, 8), 11, 512), (3, (7, 7), (8, 8), 11, 512),
                                                         (4, (16, 8), (5, 5), 5, 512)])
@pytest.mark.parametrize("act", [0, 1])
def test_window_convolution_most_of_the_lds(orc, ic, kernel, stride, batch, size, act):
    import torch
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(ic + size)
    orc.set_threads(16)
    pad = (0, 0, 0, 0)
    case = _conv_case(rng, batch, size, size, ic, 64, kernel, stride, (1, 1), pad, True, False, True, act)
    assert np.array_equal(_gpu_conv(case, stride, (1, 1), pad, 1, device_tensors=True), orc.conv_int8(**case))


# two to five blocks of channels in a workgroup, whole and not, one group and two, K of one step to several and no multiple of them
@pytest.mark.parametrize("ic,oc,act", [(16, 64, 0), (40, 40, 1), (24, 96, 0), (32, 112, 1), (32, 128, 0), (33, 128, 1), (200, 128, 3),
                                       (24, 160, 1), (77, 160, 0), (16, 192, 1), (64, 256, 1), (40, 256, 0), (128, 256, 3)])
def test_thin_convolution_channel_blocks(orc, ic, oc, act):
    import torch
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(ic * oc)
    orc.set_threads(16)
    case = _conv_case(rng, 3, 113, 141, ic, oc, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), True, False, True, act)
    assert np.array_equal(_gpu_conv(case, (1, 1), (1, 1), (0, 0, 0, 0), 1, device_tensors=True), orc.conv_int8(**case))


# channels of which every lane has all of its quads or none, some of them, and part of one; one group and several; whole tiles of
# pixels and a last one; the three kernels that store them (1x1, first layer, window)
@pytest.mark.parametrize("oc", [4, 24, 36, 40, 44, 60, 64, 72, 74, 80, 144, 176, 240])
@pytest.mark.parametrize("ic,kernel,batch,size", [(24, (1, 1), 3, 113), (3, (3, 3), 3, 113), (16, (3, 3), 5, 97)])
def test_convolution_stores_of_partial_blocks(orc, ic, kernel, batch, size, oc):
    import torch
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(ic * oc)
    orc.set_threads(16)
    pad = (kernel[0] // 2,) * 4
    for act in (0, 1):
        case = _conv_case(rng, batch, size, size + 2, ic, oc, kernel, (1, 1), (1, 1), pad, True, False, True, act)
        assert np.array_equal(_gpu_conv(case, (1, 1), (1, 1), pad, 1, device_tensors=True, exact_3x3=True), orc.conv_int8(**case))


# with and without an activation, channels below and from where the stores are non-temporal, tiles of one to four rows
@pytest.mark.parametrize("ch", [4, 124, 128, 132])
@pytest.mark.parametrize("b,ih,iw", [(1, 9, 11), (3, 50, 63), (6, 77, 81)])
@pytest.mark.parametrize("taps,act", [(3, 0), (3, 1), (5, 3), (5, 0)])
def test_depthwise_stride_one_activations(orc, b, ih, iw, ch, taps, act):
    import torch
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(ch * taps + act)
    orc.set_threads(16)
    pad = (taps // 2,) * 4
    case = _conv_case(rng, b, ih, iw, ch, ch, (taps, taps), (1, 1), (1, 1), pad, True, False, True, act, dw=True)
    assert np.array_equal(_gpu_conv(case, (1, 1), (1, 1), pad, ch, device_tensors=True), orc.conv_dw_int8(**case))


# strides and pads at and past the 16 bits in which the gathering kernels take them; past them the window buffer serves
@pytest.mark.parametrize("ic,kernel", [(3, (3, 3)), (16, (1, 3))])
@pytest.mark.parametrize("far", [32767, 32768, 40000])
def test_convolution_wide_strides_and_pads(orc, ic, kernel, far):
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(far + ic)
    pad, stride = (kernel[0] // 2, kernel[0] // 2, far, far), (1, far)
    case = _conv_case(rng, 2, 60, 9, ic, 40, kernel, stride, (1, 1), pad, True, False, True, 1)
    assert np.array_equal(_gpu_conv(case, stride, (1, 1), pad, 1, device_tensors=True, exact_3x3=True), orc.conv_int8(**case))


def _split_launches():
    """(how many split launches so far, tile and parts of the last one)"""
    import ctypes as C
    tile, parts = C.c_int32(0), C.c_int32(0)
    return K._lib.load().mi_debug_split_launches(C.byref(tile), C.byref(parts)), tile.value, parts.value


# K in several parts a tile, as choose_split deals it out: tile (10 x channels / 64 + rows / 64) and parts, up to the most of each
# tile; parts of unequal length, a last block, last rows and channels that are partly there, rows to be padded first; 0 and 1: where
# unsplit 64 x 64 tiles are quicker
@pytest.mark.parametrize("m,n,k,tile,parts", [(70, 200, 5632, 11, 5), (100, 256, 8200, 11, 6), (129, 257, 4100, 11, 5), (200, 1000, 4700, 11, 3),
                                              (70, 64, 11008, 11, 8), (65, 65, 16400, 11, 8), (80, 300, 8900, 11, 7),
                                              (100, 3330, 8368, 11, 2), (128, 4096, 11008, 12, 4), (176, 2407, 7360, 11, 2),
                                              (331, 1783, 11040, 12, 3), (300, 4096, 8192, 22, 2), (512, 4000, 11008, 22, 2),
                                              (250, 4000, 11008, 0, 1), (144, 3756, 10336, 0, 1), (199, 2252, 7888, 0, 1),
                                              (232, 2905, 10016, 0, 1), (213, 2175, 10848, 0, 1), (273, 2188, 9744, 0, 1)])
@pytest.mark.parametrize("dynamic,asymmetric", [(False, False), (False, True), (True, False)])
def test_matmul_with_k_in_parts(orc, m, n, k, tile, parts, dynamic, asymmetric):
    """On the null stream, where K is split, and on another, where it is not: the same sums.  Against the oracle too: all rows of
    small ones, rows at the tiles' edges of the others."""
    import torch
    rng = np.random.default_rng(m + n + k)
    w, bias, sw, zw, make = _matmul_pair(rng, n, k, asymmetric, dynamic)
    kern = make(True)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    dev = torch.from_numpy(a).cuda()
    args = dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
    torch.cuda.synchronize()
    other = torch.cuda.Stream()
    so_far = _split_launches()[0]
    with torch.cuda.stream(other):
        want = kern.run(dev, **args)
    other.synchronize()
    assert _split_launches()[0] == so_far
    for _ in range(4):  # (the counters are left as they were found)
        got = [kern.run(dev, **args) for _ in range(3)]
        torch.cuda.synchronize()
        for y in got:
            assert torch.equal(y.view(torch.int8), want.view(torch.int8))
    assert _split_launches()[0] == so_far + (12 if parts > 1 else 0)
    assert parts == 1 or _split_launches()[1:] == (tile, parts)
    rows = np.arange(m) if m * n * k < 1e9 else np.unique(np.r_[0, 1, 31, 63:65, 127:129, m // 2, m - 2, m - 1] % m)
    orc.set_threads(16)
    if dynamic:
        sure = orc.dynamic_matmul(a[rows], w, bias, 0.03, -5, sw, zw)
    else:
        sure = orc.matmul_int8(a[rows], w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3)
    assert np.array_equal(want.cpu().numpy()[rows], sure)


# both sides of the line between a group's one launch and members whose K is split: at one and two row tiles and beyond, rows to be padded
# first, members of unequal size, more than two
@pytest.mark.parametrize("m,ns,k,apart", [(70, (64, 64), 11008, True), (70, (64, 64), 7100, True), (70, (64, 64), 5120, False),
                                          (128, (512, 512), 8192, True), (128, (512, 512), 7168, False), (65, (1024, 64), 11008, True),
                                          (100, (1024, 1024), 8192, False), (100, (256, 250, 256), 14336, True),
                                          (100, (256, 250, 256), 11008, False), (200, (64, 64), 16384, True),
                                          (200, (512, 500), 11008, False), (70, (64, 64, 64, 64), 16384, False)])
@pytest.mark.parametrize("how", ["static", "value"])
def test_matmul_group_apart_where_members_are_split(orc, m, ns, k, apart, how):
    """On the null stream; on another, where nothing is split, the one launch in any case: the same sums."""
    import torch
    rng = np.random.default_rng(m + k)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    dev, dynamic = torch.from_numpy(a).cuda(), how == "value"
    args = dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
    pairs = [_matmul_pair(rng, n, k, False, dynamic) for n in ns]
    kernels = [pair[4](True) for pair in pairs]
    group = lambda: K.dynmm_run_group(kernels, dev, **args) if dynamic else K.matmul_run_group(kernels, dev)
    torch.cuda.synchronize()
    so_far = _split_launches()[0]
    other = torch.cuda.Stream()
    with torch.cuda.stream(other):
        want = group()
    other.synchronize()
    assert _split_launches()[0] == so_far
    got = group()
    torch.cuda.synchronize()
    assert _split_launches()[0] == so_far + (len(ns) if apart else 0)
    rows = np.unique(np.r_[0, 1, 31, 63:65, m // 2, m - 2, m - 1])
    orc.set_threads(16)
    for (w, bias, sw, zw, _), y, z in zip(pairs, got, want):
        assert torch.equal(y.view(torch.int8), z.view(torch.int8))
        if dynamic:
            sure = orc.dynamic_matmul(a[rows], w, bias, 0.03, -5, sw, zw)
        else:
            sure = orc.matmul_int8(a[rows], w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3)
        assert np.array_equal(y.cpu().numpy()[rows], sure)


def test_matmul_with_k_in_parts_on_library_streams():
    """Two threads, each with a stream of the library and a handle of its own, beside the null stream."""
    import ctypes as C
    import threading
    import torch
    L = K._lib.load()
    rng = np.random.default_rng(5)
    work = []
    for i in range(3):
        kern = _matmul_pair(rng, 1000, 4096, False, False)[4](True)
        dev = torch.from_numpy(rng.integers(-128, 128, (150, 4096), dtype=np.int8)).cuda()
        work.append((kern, dev, kern.run(dev), torch.empty((150, 1000), dtype=torch.int8, device="cuda")))
    torch.cuda.synchronize()
    failed = []

    def go(kern, dev, want, out, own):
        stream = C.c_void_p(None)
        if own and L.mi_stream_create(C.byref(stream)) != 0:
            failed.append("stream")
        for _ in range(200):
            if L.mi_matmul_run(kern._h, C.c_void_p(dev.data_ptr()), 150, C.c_void_p(out.data_ptr()), stream) != 0:
                failed.append("run")
        if _split_launches()[0] != 200:  # (of this thread)
            failed.append("not split")
        L.mi_stream_synchronize(stream)
        if not torch.equal(out, want):
            failed.append("result")
        if own and L.mi_stream_destroy(stream) != 0:
            failed.append("destroy")

    threads = [threading.Thread(target=go, args=w + (i > 0,)) for i, w in enumerate(work)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed


# row sums on the matrix cores: K that ends at every 16 bytes of a block of 128, fewer blocks than stages and more, rows and
# channels that end inside a tile; extreme values, whose sums are the largest
@pytest.mark.parametrize("k", [16, 48, 128, 144, 176, 400, 640, 1008, 1040, 2032, 4112])
@pytest.mark.parametrize("m,n", [(65, 65), (131, 300), (200, 1000)])
@pytest.mark.parametrize("dynamic", [False, True])
def test_matmul_row_sums(orc, m, n, k, dynamic):
    import torch
    rng = np.random.default_rng(m + n + k)
    w, bias, sw, zw, make = _matmul_pair(rng, n, k, True, dynamic)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    a[1], a[m // 2], a[m - 1] = -128, 127, -128
    orc.set_threads(16)
    if dynamic:
        want = orc.dynamic_matmul(a, w, bias, 0.03, -5, sw, zw)
    else:
        want = orc.matmul_int8(a, w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3)
    args = dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
    assert np.array_equal(make(True).run(torch.from_numpy(a).cuda(), **args).cpu().numpy(), want)


# few rows that are no whole 16-byte chunks, or start anywhere: shorter than a chunk and just longer, ends at each part of a chunk, of a
# 64-byte step, of a wave's slice of K and of the row lengths at which the kernels change; 8200 channels for the wide form
@pytest.mark.parametrize("k,n", [(9, 40), (17, 40), (31, 300), (63, 40), (127, 40), (250, 1001), (1001, 96), (1023, 40), (2049, 40), (4095, 33),
                                 (6151, 40), (7005, 40), (12281, 33), (13007, 33), (770, 8200), (64, 40), (1024, 40)])
@pytest.mark.parametrize("dynamic,asymmetric", [(False, False), (False, True), (True, False), (True, True)])
def test_matmul_few_rows_of_any_length(orc, k, n, dynamic, asymmetric):
    import torch
    rng = np.random.default_rng(n + k)
    w, bias, sw, zw, make = _matmul_pair(rng, n, k, asymmetric, dynamic)
    kern = make(True)
    args = dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
    orc.set_threads(16)
    for m in (1, 2, 3, 5, 8, 13, 16, 17, 32, 33, 64):
        a = rng.integers(-128, 128, (m, k), dtype=np.int8)
        if dynamic:
            want = orc.dynamic_matmul(a, w, bias, 0.03, -5, sw, zw)
        else:
            want = orc.matmul_int8(a, w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3)
        for start in (0, 1, 6, 15):
            held = torch.full((start + m * k,), 77, dtype=torch.int8, device="cuda")
            held[start:] = torch.from_numpy(a).cuda().reshape(-1)
            got = kern.run(held[start:].view(m, k), **args).cpu().numpy()
            assert np.array_equal(got, want), (m, start)


# rows of less than one block of K, at any address, where the next chunk of a row lies in the rows behind it or behind the last one
@pytest.mark.parametrize("k", [16, 17, 33, 47, 65, 100, 127])
@pytest.mark.parametrize("m,n", [(65, 40), (130, 65), (1000, 300)])
@pytest.mark.parametrize("dynamic,asymmetric", [(False, False), (False, True), (True, True)])
def test_matmul_short_rows_of_any_length(orc, m, n, k, dynamic, asymmetric):
    import torch
    rng = np.random.default_rng(m + n + k)
    w, bias, sw, zw, make = _matmul_pair(rng, n, k, asymmetric, dynamic)
    a = rng.integers(-128, 128, (m, k), dtype=np.int8)
    orc.set_threads(16)
    if dynamic:
        want = orc.dynamic_matmul(a, w, bias, 0.03, -5, sw, zw)
    else:
        want = orc.matmul_int8(a, w, bias, 0.02, 7, sw, zw, float(np.float32(0.02 * 0.0055 * k ** 0.5 * 140)), 3)
    kern = make(True)
    args = dict(in_quant=K.QuantParam(0.03, -5)) if dynamic else {}
    for start in (0, 1, 15):
        held = torch.full((start + m * k,), 77, dtype=torch.int8, device="cuda")
        held[start:] = torch.from_numpy(a).cuda().reshape(-1)
        assert np.array_equal(kern.run(held[start:].view(m, k), **args).cpu().numpy(), want), start


# values that leave the range the quick rounding holds for, or are no numbers (0x7fa00000: a signalling NaN), in tensors and rows of every
# kernel form; most of a tensor stays ordinary, and the parameters are the oracle's
@pytest.mark.parametrize("bits", [0x7fc00000, 0xffc00001, 0x7fa00000, 0xffa00000, 0x7f800000, 0xff800000, 0x7f7fffff, 0x00000001, 0x80000000])
@pytest.mark.parametrize("symmetric", [False, True])
def test_dynamic_quant_values_out_of_line(orc, bits, symmetric):
    import torch
    special = np.array([bits], np.uint32).view(np.float32)[0]
    dq = K.DynamicQuantKernel(symmetric)
    for n in (3, 700, 4099, 8195, 40003, 300002, 1500001, 6300003, 27000003):
        for scale in (1.0, 1e-30):
            x = _values(np.random.default_rng(n), n) * np.float32(scale)
            x.view(np.uint32)[[0, n // 2, n - 1]] = bits
            q, p = dq.run(torch.from_numpy(x).cuda())
            want, s, zp = orc.dynamic_quant(x, symmetric)
            assert np.array_equal(q.cpu().numpy(), want), (n, scale, special)
            assert np.array_equal([p.scale], [s], equal_nan=True) and p.zero_point == zp
    for rows, unit in ((3, 255), (600, 515), (513, 771), (256, 1028), (257, 3075), (5, 8196), (2, 16388), (2, 65540)):
        x = _values(np.random.default_rng(rows * unit), rows * unit).reshape(rows, unit)
        x.view(np.uint32)[rows // 2, [0, unit // 2, unit - 1]] = bits
        q, params = dq.run_rows(torch.from_numpy(x).cuda())
        want, scales, zps = orc.dynamic_quant_segments(x, symmetric)
        got = params.cpu().numpy().view([("scale", "f8"), ("scale_f", "f4"), ("zp", "i4"), ("lo", "f4"), ("hi", "f4")])
        assert np.array_equal(q.cpu().numpy(), want), (rows, unit, special)
        assert np.array_equal(got["scale"].reshape(-1), scales.reshape(-1), equal_nan=True) and np.array_equal(got["zp"].reshape(-1), zps.reshape(-1))


# channels that end inside and just past the parameters' padding, 8 and 16 of them a thread and one; left shifts (sums of a few units) and none
@pytest.mark.parametrize("left_shifts", [False, True])
@pytest.mark.parametrize("ch", [5, 8, 256, 264, 1008])
@pytest.mark.parametrize("taps,stride,dil", [(3, 2, 1), (5, 2, 1), (7, 1, 1), (3, 1, 2)])
def test_depthwise_parameters_of_many_channels(orc, taps, stride, dil, ch, left_shifts):
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(ch * taps + left_shifts)
    strides, dils, pad = (stride, stride), (dil, dil), (taps // 2,) * 4
    case = _conv_case(rng, 2, 9, 8, ch, ch, (taps, taps), strides, dils, pad, True, False, not left_shifts, 0, dw=True)
    if left_shifts:
        case["x"] = (case["zx"] + rng.integers(-1, 2, case["x"].shape)).astype(np.int8)
        case["w"] = rng.integers(-3, 4, case["w"].shape, dtype=np.int8)
        case["so"] = float(case["sx"] * case["sw"].mean() / 2)
    got = _gpu_conv(case, strides, dils, pad, ch, device_tensors=True)
    assert np.array_equal(got, orc.conv_dw_int8(**case))


# as above, where a lane reads four channels at a time of all parameters
@pytest.mark.parametrize("left_shifts", [False, True])
@pytest.mark.parametrize("oc", [4, 28, 32, 36, 128])
def test_short_convolution_parameters(orc, oc, left_shifts):
    from tests.test_gpu_parity import _conv_case, _gpu_conv
    rng = np.random.default_rng(oc + left_shifts)
    pad, dil = (1, 1, 2, 2), (1, 2)
    case = _conv_case(rng, 2, 12, 13, 3, oc, (3, 3), (1, 1), dil, pad, True, True, not left_shifts, 0)
    if left_shifts:
        case["x"] = (case["zx"] + rng.integers(-1, 2, case["x"].shape)).astype(np.int8)
        case["w"] = rng.integers(-3, 4, case["w"].shape, dtype=np.int8)
        case["zw"] = rng.integers(-1, 2, case["zw"].shape).astype(np.int32)
        case["so"] = float(case["sx"] * case["sw"].mean() / 2)
    assert np.array_equal(_gpu_conv(case, (1, 1), dil, pad, 1, device_tensors=True), orc.conv_int8(**case))
