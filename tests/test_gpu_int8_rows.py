"""The row quantizer's vector form and the one-launch INT8 forward at their
edges: the same bits as the oracle's quantizer and, for the forward, as
quantizing first and multiplying then."""
import numpy as np
import pytest

import oracle as O
from synapse_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    hip.init(0)


def _rows(m, k, seed):
    x = np.random.default_rng(seed).standard_normal((m, k)).astype(np.float32)
    x[:, seed % k] *= 40
    return x


# a row per block of 256 x 4 values and its neighbours, the register forms'
# lines at 1024, 4096 and 16384, rows that are not whole 16-byte groups
@pytest.mark.parametrize("k", [1, 4, 1020, 1023, 1024, 1028, 4096, 4100, 16384, 16388])
def test_quantize_rows_vector_form(k):
    x = _rows(5, k, k)
    x[1] = 0
    x[2] *= np.float32(1e-30)
    q, s = hip.quantize_per_channel_int8(x)
    wq, ws = O.quantize_per_channel_int8(x)
    np.testing.assert_array_equal(q, wq)
    np.testing.assert_array_equal(s.view(np.uint32), ws.view(np.uint32))


def _both(lin, x, offset=0):
    """(forward, quantize then multiply) of one row at a byte offset"""
    n, k = lin.n, lin.k
    buf = hip.DeviceBuffer(4 * k + 64)
    ldq = (k + 15) // 16 * 16
    xq, sx, y, y2 = (hip.DeviceBuffer(b) for b in (ldq, 16, 4 * n, 4 * n))
    try:
        raw = np.zeros(k + 16, np.float32)
        raw[offset // 4:offset // 4 + k] = x
        buf.upload(raw)
        xq.zero()
        L = hip.lib()
        lin.forward_dev(1, buf.ptr + offset, y.ptr)
        hip.check(L.syn_hip_quantize_rows(buf.ptr + offset, 1, k, k, xq.ptr, ldq, sx.ptr, None))
        lin.forward_pre_quantized_dev(1, xq.ptr, ldq, sx.ptr, y2.ptr)
        hip.check(L.syn_hip_stream_synchronize(None))
        return y.download(n, np.uint32), y2.download(n, np.uint32)
    finally:
        for b in (buf, xq, sx, y, y2):
            b.close()


# K: parts of a 16-byte chunk, one chunk, fewer chunks than waves, splits, the
# line at 16384; N: part of a panel, a K split, no K split, the line at 512
# workgroups
@pytest.mark.parametrize("k,n", [(4, 5), (16, 64), (20, 70), (1000, 100), (1024, 1024),
                                 (2052, 3000), (16384, 130), (16388, 130), (64, 32768),
                                 (64, 32769), (4096, 16500)])
def test_one_launch_forward(k, n):
    rng = np.random.default_rng(k + n)
    lin = hip.QLinear.int8(rng.integers(-128, 128, (n, k), dtype=np.int8),
                           (rng.random(n) * 1e-3 + 1e-4).astype(np.float32), hip.LAYOUT_NK)
    cases = [_rows(1, k, n)[0], np.zeros(k, np.float32)]
    odd = _rows(1, k, n + 1)[0]
    odd[k // 2] = np.nan
    cases.append(odd)
    odd = odd.copy()
    odd[0] = np.inf
    cases.append(odd)
    for i, x in enumerate(cases):
        for offset in (0, 4):  # 4: not 16-byte aligned, the two-launch form
            a, b = _both(lin, x, offset)
            np.testing.assert_array_equal(a, b, err_msg=f"case {i} offset {offset}")
        a2, _ = _both(lin, x)  # the K split's accumulators were left clear
        np.testing.assert_array_equal(a2, b)
    lin.close()


def test_forward_in_place():
    # y over x: every row is quantized before any of y is written
    n = k = 4096
    rng = np.random.default_rng(6)
    lin = hip.QLinear.int8(rng.integers(-128, 128, (n, k), dtype=np.int8),
                           (rng.random(n) * 1e-3 + 1e-4).astype(np.float32), hip.LAYOUT_NK)
    x = _rows(1, k, 11)[0]
    want, _ = _both(lin, x)
    buf = hip.DeviceBuffer(8 * k)
    for offset in (0, 16):  # words of x between its start and that of y
        buf.upload(np.concatenate([x, np.zeros(k, np.float32)]))
        lin.forward_dev(1, buf.ptr, buf.ptr + 4 * offset)
        hip.check(hip.lib().syn_hip_stream_synchronize(None))
        np.testing.assert_array_equal(buf.download(2 * k, np.uint32)[offset:offset + n], want)
    buf.close()
    lin.close()
