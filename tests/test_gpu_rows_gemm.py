"""The few-row quantized GEMM against float64 products of the dequantized
weights, at the edges of its tiles and of its dispatch rule.

Bounds, per element and relative to sum |x w|: one f16 rounding (2^-11) of
each activation and each weight, plus f32 sums, stay below 2^-10 (1 + 2^-4).
Q4_0 at 7 to 16 rows: activations, levels and products are exact, and what is
left is the f32 sums, of fewer than K / 16 + 24 partial sums 2^-24 each."""
import numpy as np
import pytest
import torch

from synapse_amd import hip

pytestmark = pytest.mark.gpu

EL = {hip.FMT_Q4_0: 32, hip.FMT_Q8_0: 32, hip.FMT_Q4_K: 256, hip.FMT_Q6_K: 256}
NAME = {hip.FMT_Q4_0: "q4_0", hip.FMT_Q8_0: "q8_0", hip.FMT_Q4_K: "q4_k", hip.FMT_Q6_K: "q6_k"}


@pytest.fixture(scope="module", autouse=True)
def gpu():
    hip.init(0)


def _linear(fmt, n, k, seed):
    """a handle and its float64 weights"""
    rng = np.random.default_rng(seed)
    w = rng.standard_normal((n, k)).astype(np.float32) * 0.05
    if fmt == hip.FMT_Q4_0:
        raw = rng.integers(0, 256, (n * k // 32, 18), dtype=np.uint8)
        d = (rng.random(n * k // 32) * 0.01 + 1e-3).astype(np.float16)
        raw[:, :2] = d.view(np.uint8).reshape(-1, 2)
        q = np.empty((n * k // 32, 32))
        q[:, 0::2], q[:, 1::2] = raw[:, 2:] & 15, raw[:, 2:] >> 4
        return (hip.QLinear.q4_0(raw.reshape(-1), n, k),
                ((q - 8) * d.astype(np.float64)[:, None]).reshape(n, k))
    blocks = hip.kquant_encode(fmt, w)
    return (hip.QLinear.gguf(fmt, blocks, n, k),
            hip.kquant_decode(fmt, blocks).astype(np.float64).reshape(n, k))


def _check(lin, w, x, split):
    m, k = x.shape
    got = lin.forward(x).astype(np.float64)
    want = x.astype(np.float64) @ w.T
    size = np.abs(x).astype(np.float64) @ np.abs(w).T
    bound = 2.0**-21 + (k / 16 + 16) * 2.0**-24 if split else 2.0**-10 * (1 + 2.0**-4)
    worst = float((np.abs(got - want) / size).max())
    print(NAME[lin.fmt], "m", m, "n", w.shape[0], "k", k, "worst", worst, "bound", bound, flush=True)
    assert worst <= bound, (m, worst, bound)
    return worst


# rows: one and two tiles of 32, one and two passes of 64, the rule's lines
# at 128 / 129 and 256 / 257; K: one step, an odd number of half steps, fewer
# and more steps than waves, a K split; N: a part of a panel, several panels
@pytest.mark.parametrize("fmt", sorted(EL), ids=lambda f: NAME[f])
@pytest.mark.parametrize("n,k", [(36, 256), (100, 512), (64, 2304), (320, 4096)])
def test_rows_gemm_edges(fmt, n, k):
    lin, w = _linear(fmt, n, k, n + k)
    rng = np.random.default_rng(k)
    x = rng.standard_normal((260, k)).astype(np.float32)
    x[:, rng.integers(0, k, 3)] *= 50
    x[3] *= 1e-7
    x[5] *= 1e6
    for m in (9, 16, 17, 31, 32, 33, 64, 65, 127, 128, 129, 256, 257):
        _check(lin, w, x[:m], fmt == hip.FMT_Q4_0 and m <= 16)
    lin.close()


@pytest.mark.parametrize("fmt", [hip.FMT_Q4_0, hip.FMT_Q8_0], ids=lambda f: NAME[f])
@pytest.mark.parametrize("k", [32, 96, 1056])
def test_rows_gemm_half_step_tail(fmt, k):
    lin, w = _linear(fmt, 72, k, k)
    x = np.random.default_rng(k).standard_normal((40, k)).astype(np.float32)
    for m in (9, 16, 17, 40):
        _check(lin, w, x[:m], fmt == hip.FMT_Q4_0 and m <= 16)
    lin.close()


def test_split_rows_seven_and_eight():
    # 7 and 8 rows take the matrix cores from 24e6 weights on; both sides of the line
    for n, k in ((8192, 3072), (1024, 2048)):
        lin, w = _linear(hip.FMT_Q4_0, n, k, 3)
        x = np.random.default_rng(5).standard_normal((8, k)).astype(np.float32)
        for m in (6, 7, 8):
            _check(lin, w, x[:m], True)
        lin.close()


def test_split_rows_extremes():
    # a row of subnormals, a zero row, rows at the ends of the f32 range; a
    # NaN or an infinity stays in its own row
    k, n = 256, 64
    lin, w = _linear(hip.FMT_Q4_0, n, k, 8)
    x = np.random.default_rng(9).standard_normal((12, k)).astype(np.float32)
    x[0] *= np.float32(1e-41)
    x[1] = 0
    x[2] *= np.float32(1e-30)
    x[3] *= np.float32(1e30)
    x[4, 7] = np.inf
    x[5, 9] = np.nan
    got = lin.forward(x)
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.T
        inf_row = (np.inf * w[:, 7]).astype(np.float32)
    assert not got[1].any()
    assert np.isnan(got[5]).all()
    # infinity times a weight of zero is a NaN, else an infinity of its sign
    np.testing.assert_array_equal(got[4], inf_row)
    for r in (0, 2, 3, 6, 7, 8, 9, 10, 11):
        size = np.abs(x[r]).astype(np.float64) @ np.abs(w).T
        # subnormal outputs round to 2^-149
        assert (np.abs(got[r] - want[r]) <= 1e-6 * size + 2.0**-148).all(), r
    lin.close()


@pytest.mark.parametrize("d", [2.0**13, 65504.0])
def test_wide_scales_keep_the_gemv(d):
    # 8 d beyond f16: the levels are scaled in f32
    n, k, m = 64, 512, 12
    rng = np.random.default_rng(21)
    raw = rng.integers(0, 256, (n * k // 32, 18), dtype=np.uint8)
    dd = np.full(n * k // 32, 0.01, np.float16)
    dd[5] = d
    raw[:, :2] = dd.view(np.uint8).reshape(-1, 2)
    raw[5, 2] = 0x00  # nibble 0: -8 d
    q = np.empty((n * k // 32, 32))
    q[:, 0::2], q[:, 1::2] = raw[:, 2:] & 15, raw[:, 2:] >> 4
    w = ((q - 8) * dd.astype(np.float64)[:, None]).reshape(n, k)
    lin = hip.QLinear.q4_0(raw.reshape(-1), n, k)
    _check(lin, w, rng.standard_normal((m, k)).astype(np.float32), True)
    lin.close()


# y over x, or over its upper part, where K splits add into rows that are cleared first: 24 rows
# of the few-row kernel, 512 of the tiled one (two splits each on separate buffers)
@pytest.mark.parametrize("m", [24, 512])
@pytest.mark.parametrize("offset", [0, 64], ids=["same", "shifted"])
def test_k_split_in_place(m, offset):
    n = k = 4096
    lin, w = _linear(hip.FMT_Q8_0, n, k, 4)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    buf = hip.DeviceBuffer(4 * (m * k + offset))
    buf.upload(np.concatenate([x.ravel(), np.zeros(offset, np.float32)]))
    lin.forward_dev(m, buf.ptr, buf.ptr + 4 * offset)
    hip.check(hip.lib().syn_hip_stream_synchronize(None))
    got = buf.download(m * k + offset, np.float32)[offset:].reshape(m, n).astype(np.float64)
    size = np.abs(x).astype(np.float64) @ np.abs(w).T
    worst = float((np.abs(got - x.astype(np.float64) @ w.T) / size).max())
    print("m", m, "offset", offset, "worst", worst, flush=True)
    assert worst <= 2.0**-10 * (1 + 2.0**-4)
    buf.close()
    lin.close()


def _raw(fmt, n, k, seed):
    """a handle over random bytes with scales of about 0.01, and the bytes"""
    size, at = {hip.FMT_Q4_0: (18, (0,)), hip.FMT_Q8_0: (34, (0,)), hip.FMT_Q4_K: (144, (0, 2)),
                hip.FMT_Q6_K: (210, (208,))}[fmt]
    rng = np.random.default_rng(seed)
    raw = rng.integers(0, 256, (n * k // EL[fmt], size), dtype=np.uint8)
    d = (rng.random(len(raw)) * 0.01 + 0.005).astype(np.float16).view(np.uint8).reshape(-1, 2)
    for a in at:
        raw[:, a:a + 2] = d
    if fmt == hip.FMT_Q4_0:
        return hip.QLinear.q4_0(raw.reshape(-1), n, k), raw
    return hip.QLinear.gguf(fmt, raw.reshape(-1), n, k), raw


# shapes whose least time by the launch rule's count is at three or four K splits, on grids where
# at most two are taken: the same bits from call to call
@pytest.mark.parametrize("fmt,m,n,k", [(hip.FMT_Q8_0, 15, 20040, 9216),
                                       (hip.FMT_Q4_K, 26, 17000, 10752),
                                       (hip.FMT_Q6_K, 9, 16388, 14336)])
def test_bits_repeat(fmt, m, n, k):
    lin, _ = _raw(fmt, n, k, m)
    x = np.random.default_rng(k).standard_normal((m, k)).astype(np.float32)
    first = lin.forward(x).view(np.uint32)
    for _ in range(6):
        np.testing.assert_array_equal(lin.forward(x).view(np.uint32), first)
    lin.close()


# both sides of the lines to the tiled kernels: 128 rows on full and part rounds of columns and at
# K of 1536, the columns of 129 to 256 rows, the products m n and m n k, 512 and 1024 rows
@pytest.mark.parametrize("fmt,n,k,rows", [
    (hip.FMT_Q8_0, 28548, 256, (64, 65, 128)), (hip.FMT_Q4_K, 28676, 256, (64, 65, 128)),
    (hip.FMT_Q6_K, 28676, 1792, (65, 128)), (hip.FMT_Q8_0, 28676, 1536, (128,)),
    (hip.FMT_Q8_0, 7168, 8192, (129, 256)), (hip.FMT_Q8_0, 7172, 8192, (129, 256)),
    (hip.FMT_Q4_K, 8196, 512, (128, 129)), (hip.FMT_Q4_0, 3128, 512, (511, 512)),
    (hip.FMT_Q8_0, 256, 4128, (1024, 1025)), (hip.FMT_Q8_0, 256, 6144, (953, 954)),
    (hip.FMT_Q6_K, 64, 512, (512, 513, 1024, 1025)), (hip.FMT_Q4_K, 260, 8192, (1024,))])
def test_dispatch_lines(fmt, n, k, rows):
    lin, raw = _raw(fmt, n, k, n)
    if fmt == hip.FMT_Q4_0:
        q = np.empty((len(raw), 32), np.float32)
        q[:, 0::2], q[:, 1::2] = raw[:, 2:] & 15, raw[:, 2:] >> 4
        w = (q - 8) * raw[:, :2].copy().view(np.float16).astype(np.float32)
    else:
        w = hip.kquant_decode(fmt, raw.reshape(-1))
    w = w.astype(np.float64).reshape(n, k)
    x = np.random.default_rng(k).standard_normal((max(rows), k)).astype(np.float32)
    for m in rows:
        _check(lin, w, x[:m], False)
    lin.close()


def _q4_0(n, k, d, seed):
    """a Q4_0 handle's bytes with the block scales d, and its float64 weights"""
    raw = np.random.default_rng(seed).integers(0, 256, (n * k // 32, 18), dtype=np.uint8)
    raw[:, :2] = d.view(np.uint8).reshape(-1, 2)
    q = np.empty((len(raw), 32))
    q[:, 0::2], q[:, 1::2] = raw[:, 2:] & 15, raw[:, 2:] >> 4
    return raw, ((q - 8) * d.astype(np.float64)[:, None]).reshape(n, k)


# an activation 2^30 times the others, on weights of zero: the others keep all of their bits
@pytest.mark.parametrize("k", [64, 2048])
def test_q4_0_rows_beside_an_outlier(k):
    n, m = 96, 12
    rng = np.random.default_rng(k)
    raw, w = _q4_0(n, k, (rng.random(n * k // 32) * 0.01 + 1e-3).astype(np.float16), k)
    raw.reshape(n, -1, 18)[:, 1, 2 + 3] = 0x88  # elements 6 and 7 of every row's second block
    w[:, 32 + 6:32 + 8] = 0
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[:, 32 + 6] = 2.0**30
    lin = hip.QLinear.q4_0(raw.reshape(-1), n, k)
    _check(lin, w, x, True)
    lin.close()


# subnormal block scales, as IEEE values and (GGUF) halved, in the K split and without it
@pytest.mark.parametrize("gguf", [False, True])
@pytest.mark.parametrize("m", [9, 16])
def test_q4_0_rows_subnormal_scales(m, gguf):
    n, k = 72, 1056
    rng = np.random.default_rng(m)
    d = (rng.random(n * k // 32) * 0.01 + 1e-3).astype(np.float16)
    d[::3] = rng.integers(1, 1024, len(d[::3]), dtype=np.uint16).view(np.float16)
    raw, w = _q4_0(n, k, d, m)
    if gguf:
        w.reshape(-1, 32)[::3] *= 0.5
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[:, 96:128] *= 1e4  # a block whose scale is subnormal counts
    lin = hip.QLinear.q4_0(raw.reshape(-1), n, k, gguf_dequant=gguf)
    _check(lin, w, x, True)
    lin.close()


# columns of 32 and 64 a workgroup (the line at 8192) with parts of the last one, block counts that
# are no whole steps of four, K splits
@pytest.mark.parametrize("n,k", [(8196, 288), (8192, 96), (8188, 1056), (16404, 160), (1000, 14336),
                                 (40, 2112), (15300, 64)])
def test_q4_0_rows_columns(n, k):
    rng = np.random.default_rng(n)
    raw, w = _q4_0(n, k, (rng.random(n * k // 32) * 0.01 + 1e-3).astype(np.float16), n)
    x = rng.standard_normal((16, k)).astype(np.float32)
    x[0, 5], x[3, 7], x[4, 8] = np.inf, 1e38, np.nan
    lin = hip.QLinear.q4_0(raw.reshape(-1), n, k)
    for m in (9, 16):
        got = lin.forward(x[:m]).astype(np.float64)
        assert np.isnan(got[4]).all() and not np.isfinite(got[0]).any()
        rows = [r for r in range(m) if r not in (0, 4)]
        size = np.abs(x[rows]).astype(np.float64) @ np.abs(w).T
        worst = float((np.abs(got[rows] - x[rows].astype(np.float64) @ w.T) / size).max())
        print("n", n, "k", k, "m", m, "worst", worst, flush=True)
        assert worst <= (k / 16 + 24) * 2.0**-24
    lin.close()


# grids without a K split use no scratch: the first call may be recorded into a graph, and two
# streams may run one handle at once
def test_q4_0_rows_capture_and_streams():
    n, k, m = 16384, 512, 12
    lin, _ = _raw(hip.FMT_Q4_0, n, k, 2)
    xs = [torch.randn(m, k, device="cuda", generator=torch.Generator("cuda").manual_seed(i))
          for i in range(2)]
    ys = [torch.zeros(m, n, device="cuda") for _ in range(2)]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=streams[0]):
        lin.forward_dev(m, xs[0].data_ptr(), ys[0].data_ptr(), stream=streams[0].cuda_stream)
    want = [torch.from_numpy(lin.forward(x.cpu().numpy())).cuda() for x in xs]
    for _ in range(3):
        ys[0].zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(ys[0], want[0])
    for _ in range(20):
        for x, y, s in zip(xs, ys, streams):
            lin.forward_dev(m, x.data_ptr(), y.data_ptr(), stream=s.cuda_stream)
    torch.cuda.synchronize()
    for y, v in zip(ys, want):
        assert torch.equal(y, v)
    lin.close()


# 64 columns a workgroup (over 8192), a part of the last one, one and two tiles of 32 rows, block
# counts that leave half a step over
@pytest.mark.parametrize("fmt", sorted(EL), ids=lambda f: NAME[f])
@pytest.mark.parametrize("n", [8196, 14340])
def test_rows_gemm_wide(fmt, n):
    k = 512 if EL[fmt] == 256 else 288
    lin, w = _linear(fmt, n, k, n)
    x = np.random.default_rng(n).standard_normal((64, k)).astype(np.float32)
    for m in (9, 16, 17, 32, 33, 64):
        _check(lin, w, x[:m], fmt == hip.FMT_Q4_0 and m <= 16)
    lin.close()


# rows of y that are no whole 16 bytes, or start off them, are not cleared 16 bytes at a time
@pytest.mark.parametrize("n,offset", [(1021, 0), (1024, 1), (1022, 3)])
def test_k_split_unaligned_output(n, offset):
    m, k = 24, 4096
    lin, w = _linear(hip.FMT_Q8_0, n, k, n)
    x = np.random.default_rng(n).standard_normal((m, k)).astype(np.float32)
    bx, by = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(4 * (m * n + 8))
    by.upload(np.full(m * n + 8, 7, np.float32))
    lin.forward_dev(m, bx.ptr, by.ptr + 4 * offset)
    hip.check(hip.lib().syn_hip_stream_synchronize(None))
    y = by.download(m * n + 8, np.float32)
    got = y[offset:offset + m * n].reshape(m, n).astype(np.float64)
    size = np.abs(x).astype(np.float64) @ np.abs(w).T
    assert (np.abs(got - x.astype(np.float64) @ w.T) / size).max() <= 2.0**-10 * (1 + 2.0**-4)
    assert (y[:offset] == 7).all() and (y[offset + m * n:] == 7).all()
    for b in (bx, by):
        b.close()
    lin.close()


# y over x, and from x's second row on
@pytest.mark.parametrize("n,k", [(2048, 2048), (8224, 4096)])
@pytest.mark.parametrize("row", [0, 1])
def test_q4_0_rows_in_place(n, k, row):
    m = 12
    lin, _ = _raw(hip.FMT_Q4_0, n, k, 5)
    x = np.random.default_rng(n).standard_normal((m, k)).astype(np.float32)
    want = lin.forward(x)
    size = row * k + m * max(n, k)
    buf = hip.DeviceBuffer(4 * size)
    for _ in range(3):
        buf.upload(np.concatenate([x.ravel(), np.zeros(size - m * k, np.float32)]))
        lin.forward_dev(m, buf.ptr, buf.ptr + 4 * row * k)
        hip.check(hip.lib().syn_hip_stream_synchronize(None))
        got = buf.download(size, np.float32)[row * k:row * k + m * n].reshape(m, n)
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    buf.close()
    lin.close()
