"""Softmax and argmax on rows a workgroup holds, and gemv on rows that do not fill the chip or do
not start 16-byte aligned: lengths around the register forms' limits and the 4-wide remainder."""
import numpy as np
import pytest

import mensurflow_amd as mf
from helpers import quarter_matrix, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [1025, 2049, 2051, 8191, 8192, 8193, 16384, 16387, 32003, 32768,
                                   32769])
def test_softmax_and_argmax(stream, oracle, width):
    rng = np.random.default_rng(width)
    x = (4 * rng.standard_normal((7, width))).astype(np.float32)
    x[1, width // 2] = np.nan
    x[2, :] = -np.inf
    x[3, 5:] = -np.inf
    x[4, width - 1] = np.inf
    x[5, [3, width - 1]] = 100.0  # a tie: the lower index
    x[6, :] = 0.0
    x[6, 1::2] = -0.0
    x_d = mf.DeviceArray.from_numpy(x, stream)
    got = mf.softmax(x_d).numpy()
    want = oracle.softmax(x)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    # Within 4 units in the last place (the exponential's 1 or 2, the scale's rounding).
    ulp = np.spacing(np.maximum(want[ok], np.finfo(np.float32).tiny))
    assert np.all(np.abs(got[ok] - want[ok]) <= 4 * ulp)
    choice = mf.argmax(x_d).numpy()
    assert choice.tolist() == oracle.argmax(x).tolist()
    x[0, [7, 9]] = np.nan  # the first NaN
    assert mf.argmax(mf.DeviceArray.from_numpy(x, stream)).numpy()[0] == 7
    inplace = mf.DeviceArray.from_numpy(x[5:], stream)
    mf.softmax(inplace, out=inplace)
    assert same_bits(inplace.numpy(), got[5:])


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 2), (1, 4099), (64, 5), (2047, 257),
                                       (2048, 1024), (2050, 1023), (8191, 300), (4001, 512), (8200, 64),
                                       (300, 16383), (4093, 1023), (16, 20000)])
def test_gemv_exact(stream, rows, cols):
    """Quarter integers: exact sums, so exact results, N and T, on whole and offset storage."""
    a = quarter_matrix(rows, cols, rows + cols)
    y0n, y0t = quarter_matrix(1, rows, 1)[0], quarter_matrix(1, cols, 2)[0]
    xn, xt = quarter_matrix(1, cols, 3)[0], quarter_matrix(1, rows, 4)[0]
    a64 = a.astype(np.float64)
    for offset in (0, 1):
        store = np.zeros((rows, cols + 3), np.float32)
        store[:, offset:offset + cols] = a
        a_d = mf.DeviceArray.from_numpy(store, stream).slice(1, offset, offset + cols)
        for trans, x, y0 in ((False, xn, y0n), (True, xt, y0t)):
            pad = np.concatenate([np.zeros(offset, np.float32), x])
            x_d = mf.DeviceArray.from_numpy(pad, stream).slice(0, offset, offset + x.size)
            y = mf.sgemv(a_d, x_d, alpha=2.0, beta=0.5,
                         y0=mf.DeviceArray.from_numpy(y0, stream), trans=trans).numpy()
            want = 2.0 * ((a64.T if trans else a64) @ x.astype(np.float64)) + 0.5 * y0
            assert same_bits(y, want.astype(np.float32)), (rows, cols, trans, offset)


@pytest.mark.parametrize("rows,width", [(4096, 1024), (4096, 1025), (4097, 1025),
                                        (4097, 3072), (4097, 3073)])
def test_argmax_many_rows(stream, rows, width):
    """Both sides of the line between a wavefront and a workgroup a row, ties to the lower index."""
    x = np.random.default_rng(rows).integers(-500, 500, (rows, width)).astype(np.float32)
    x[::7, width - 1] = np.nan
    got = mf.argmax(mf.DeviceArray.from_numpy(x, stream)).numpy()
    assert np.array_equal(got, np.argmax(np.where(np.isnan(x), np.inf, x), axis=1))
