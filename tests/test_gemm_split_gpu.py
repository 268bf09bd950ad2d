"""The GEMM tiles on the bf16 matrix cores (three bf16 parts per operand element) where the parts
could miss the fp32 product: non-finite and huge operands, tiny ones, sums that are zero or
underflow, at tile edges and remainders of the 16- and 32-deep slices. Against float64 products
rounded to float32, within the summation bound k * 2^-24 of sum |a b| (plus the float32 product's
own underflow, 2^-149 per term)."""
import numpy as np
import pytest

import mensurflow_amd as mf
from helpers import quarter_matrix, same_bits

pytestmark = pytest.mark.gpu

TILES = [mf.abi.TILE_256x256, mf.abi.TILE_128x128, mf.abi.TILE_128x64, mf.abi.TILE_64x128,
         mf.abi.TILE_64x64]


def check(stream, a, b, tile, trans_a=False, trans_b=False, splits=1):
    """One product against its float64 value; returns the result."""
    m, k = a.shape
    n = b.shape[1]
    a_d = mf.DeviceArray.from_numpy(np.ascontiguousarray(a.T if trans_a else a), stream)
    b_d = mf.DeviceArray.from_numpy(np.ascontiguousarray(b.T if trans_b else b), stream)
    got = mf.gemm(a_d, b_d, trans_a=trans_a, trans_b=trans_b, tile=tile, splits=splits,
                  stage=mf.abi.STAGE_NEVER).numpy()
    with np.errstate(all="ignore"):
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        want = (a64 @ b64).astype(np.float32)
        scale = np.abs(a64) @ np.abs(b64)
    what = f"tile {tile} {m}x{n}x{k} ta {trans_a} tb {trans_b}"
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)), what
    assert np.array_equal(got[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)]), what
    bound = scale * k * 2.0**-24 + k * 2.0**-149
    err = np.abs(got[finite].astype(np.float64) - want[finite].astype(np.float64))
    assert np.all(err <= bound[finite]), (what, float(np.max(err / bound[finite])))
    return got


def normal(shape, seed, scale=1.0):
    return (np.random.default_rng(seed).standard_normal(shape) * scale).astype(np.float32)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k", [(1, 1, 65), (37, 70, 80), (130, 257, 95), (64, 64, 1000),
                                   (300, 260, 129), (1000, 1000, 97)])
def test_normal_operands(stream, tile, m, n, k):
    for ta in (False, True):
        for tb in (False, True):
            check(stream, normal((m, k), 1), normal((k, n), 2), tile, ta, tb)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("case", ["inf", "inf times zero", "nan", "huge", "overflow", "tiny",
                                  "tiny and large", "tiny product", "denormal", "zero rows",
                                  "zeros", "few tiny", "identity", "zero rows, tiny columns",
                                  "tiny by ordinary", "one tiny row"])
def test_extreme_operands(stream, tile, case):
    # 16 x 16 tiles of 64x64: the register form; fewer workgroups than half the CUs: the other; at
    # most 32 rows: the 32x64 form, with and without its loop of two steps in flight.
    for m, n, k in ((1000, 1000, 71), (150, 90, 200), (20, 150, 71), (20, 150, 500)):
        a, b = normal((m, k), 3), normal((k, n), 4)
        if case == "inf":
            a[5, 3], a[m - 1, k - 1], b[7, 11] = np.inf, -np.inf, np.inf
        elif case == "inf times zero":
            a[5, 3], b[3, 8], a[6, 3] = np.inf, 0.0, 1.0
        elif case == "nan":
            a[m - 1, 0], b[k - 1, n - 1] = np.nan, np.nan
        elif case == "huge":  # above the largest bf16, the products finite
            a[2, 1], b[1, :] = 3.4e38, np.float32(1e-3)
            a[9, 4], b[4, :] = -3.4e38, np.float32(2.0**-40)
        elif case == "overflow":
            a[2, :], b[:, 9] = 1e30, 1e30
        elif case == "tiny":
            a = normal((m, k), 3, 1e-36)
        elif case == "tiny and large":
            a, b = normal((m, k), 3, 1e-38), normal((k, n), 4, 1e30)
        elif case == "tiny product":
            a, b = normal((m, k), 3, 1e-20), normal((k, n), 4, 1e-19)
        elif case == "denormal":
            a = normal((m, k), 3, 1e-41)
            b = normal((k, n), 4, 1e20)
        elif case == "zero rows":
            a[m // 3: m // 2], b[:, n // 2:] = 0.0, 0.0
            a[m // 3, 2] = 1e-40
        elif case == "zeros":
            a[:] = 0.0
        elif case == "few tiny":  # sums clear of what the tiny elements can lose
            a[:, 1::3] = normal((m, k), 5, 1e-39)[:, 1::3]
        elif case == "zero rows, tiny columns":
            a[m // 3: m // 2], b[:, ::5] = 0.0, b[:, ::5] * np.float32(1e-38)
        elif case == "tiny by ordinary":
            a = normal((m, k), 3, 1e-20)
        elif case == "one tiny row":
            a[7] *= np.float32(1e-37)
        elif case == "identity":  # every element comes back exactly
            b = np.zeros((k, n), np.float32)
            b[np.arange(min(k, n)), np.arange(min(k, n))] = 1.0
        got = check(stream, a, b, tile)
        if case == "identity":
            q = min(k, n)
            assert np.array_equal(got[:, :q], a[:, :q])


def test_one_zero_sum(stream):
    """A sum that is exactly zero among ordinary ones (its row and column are read again)."""
    for tile in TILES:
        a, b = normal((300, 128), 6), normal((128, 300), 7)
        a[17, 64:] = -a[17, :64]
        b[64:, 31] = b[:64, 31]
        got = check(stream, a, b, tile)
        assert abs(got[17, 31]) <= 128 * 2.0**-24 * np.abs(a[17]) @ np.abs(b[:, 31])


@pytest.mark.parametrize("splits", [2, 5])
def test_extremes_in_depth_ranges(stream, splits):
    a, b = normal((200, 700), 8), normal((700, 130), 9)
    a[3, 10], b[650, 100], a[50] = np.inf, np.nan, 1e-41
    check(stream, a, b, mf.abi.TILE_64x64, splits=splits)


def test_no_larger_error_than_fp32_chains(stream):
    """The 2-norm error on uniform and normal operands stays under a sequential fp32 sum's
    (sqrt(k) / 4 roundings of 2^-24 at the sum's size), whatever the tile."""
    for k in (128, 1024, 4096):
        a = np.random.default_rng(k).uniform(-1, 1, (256, k)).astype(np.float32)
        b = np.random.default_rng(k + 1).uniform(-1, 1, (k, 256)).astype(np.float32)
        want = a.astype(np.float64) @ b.astype(np.float64)
        for tile in TILES:
            got = mf.gemm(mf.DeviceArray.from_numpy(a, stream),
                          mf.DeviceArray.from_numpy(b, stream), tile=tile, splits=1).numpy()
            rel = np.linalg.norm(got - want) / np.linalg.norm(want)
            assert rel <= np.sqrt(k) * 2.0**-24 * 0.3, (k, tile, rel)


@pytest.mark.parametrize("m,n,k", [(256, 256, 256), (20, 250, 500), (200, 250, 71), (130, 70, 40),
                                   (300, 260, 71), (2100, 2100, 40)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_lines_that_run_backwards(stream, m, n, k, ta, tb):
    """Operands whose lines lie a negative stride apart (the descriptor takes any element strides):
    quarter integers, so the product is exact on AUTO (which would peel a strip off a 256x256 tile, or take the panel path,
    were the lines in order) and on every tile."""
    a, b = quarter_matrix(m, k, 1), quarter_matrix(k, n, 2)
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    # Stored along k or along m (n), the lines in reverse order.
    a_d = mf.DeviceArray.from_numpy(np.ascontiguousarray((a.T if ta else a)[::-1]), stream)
    b_d = mf.DeviceArray.from_numpy(np.ascontiguousarray((b.T if tb else b)[::-1]), stream)
    c = mf.DeviceArray.empty((m, n), stream)
    d = mf.GemmDesc()
    d.m, d.n, d.k, d.alpha = m, n, k, 1.0
    d.a = a_d.ptr + 4 * (a.size - (m if ta else k))
    d.a_rs, d.a_cs = (1, -m) if ta else (-k, 1)
    d.b = b_d.ptr + 4 * (b.size - (k if tb else n))
    d.b_rs, d.b_cs = (1, -k) if tb else (-n, 1)
    d.c, d.c_rs, d.stage = c.ptr, n, mf.abi.STAGE_NEVER
    for tile in [mf.abi.TILE_AUTO] + TILES[1:]:  # the 256x256 tile refuses such lines
        d.tile = tile
        mf.fill(c, 7.0)
        mf.sgemm(stream, d)
        assert np.array_equal(c.numpy(), want), (tile, m, n, k, ta, tb)


@pytest.mark.parametrize("tile", TILES)
def test_no_depth_gelu(stream, oracle, tile):
    """A depth of 0 on a fixed tile: gelu(beta C0 + bias) bit for bit in every wavefront, the exp
    table in LDS written before any of them reads it, right after a product that left other values
    there."""
    m, n = 300, 260
    c0, bias = normal((m, n), 10), normal((n,), 11)
    want = oracle.gelu(oracle.bias_add(np.float32(0.5) * c0, bias), approximate=True)
    dev = lambda x: mf.DeviceArray.from_numpy(x, stream)  # noqa: E731
    c0_d, bias_d = dev(c0), dev(bias)
    a, b = mf.DeviceArray.empty((m, 0), stream), mf.DeviceArray.empty((0, n), stream)
    other = dev(normal((512, 512), 12))
    c = mf.DeviceArray.empty((m, n), stream)
    for _ in range(5):
        mf.gemm(other, other, tile=tile)
        mf.fill(c, 7.0)
        mf.gemm(a, b, c0=c0_d, beta=0.5, bias=bias_d, act=mf.ACT_GELU_TANH, tile=tile, out=c)
        assert same_bits(c.numpy(), want)


@pytest.mark.parametrize("batch", [256, 257, 513])
@pytest.mark.parametrize("k", [72, 127, 128, 511, 512])
def test_few_rows_batched_exact(stream, batch, k):
    """At most 32 rows and one 64-column tile a matrix: both sides of the register form's lines, in
    tiles and in depth, exact on quarter integers."""
    m, n = 19, 61
    a = quarter_matrix(batch * m, k, 1).reshape(batch, m, k)
    b = quarter_matrix(batch * k, n, 2).reshape(batch, k, n)
    want = (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)
    a_d = mf.DeviceArray.from_numpy(a, stream)
    c = mf.DeviceArray.empty((batch, m, n), stream)
    for tb in (False, True):
        b_d = mf.DeviceArray.from_numpy(np.ascontiguousarray(np.swapaxes(b, 1, 2) if tb else b), stream)
        mf.gemm_batched(a_d, b_d.transpose(-2, -1) if tb else b_d, c)
        assert np.array_equal(c.numpy(), want), tb


@pytest.mark.parametrize("nonzeros,k", [(1, 512), (2, 512), (4, 512), (8, 1024), (32, 4096),
                                        (500, 1000)])
def test_sparse_and_wide_rows(stream, nonzeros, k):
    """Rows with few nonzeros, and rows of widely differing sizes, within (2 + 6 s) 2^-24 of
    sum |a b|: s steps of 16 depths with a nonzero, six roundings each, the products left out and the
    last rounding."""
    rng = np.random.default_rng(k)
    sparse = np.zeros((200, k), np.float32)
    for row in sparse:
        row[rng.choice(k, nonzeros, replace=False)] = rng.standard_normal(nonzeros)
    wide = (rng.standard_normal((200, k)) * np.exp(3 * rng.standard_normal((200, k)))).astype(np.float32)
    b = normal((k, 150), 2)
    for a in (sparse, wide):
        padded = np.pad(a != 0, ((0, 0), (0, -k % 16))).reshape(200, -1, 16)
        steps = padded.any(axis=2).sum(axis=1)[:, None]
        want = a.astype(np.float64) @ b.astype(np.float64)
        scale = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
        for tile in TILES:
            got = mf.gemm(mf.DeviceArray.from_numpy(a, stream),
                          mf.DeviceArray.from_numpy(b, stream), tile=tile, splits=1).numpy()
            assert np.all(np.abs(got - want) <= (2 + 6 * steps) * 2.0**-24 * scale), tile
            if a is sparse:
                # One rounding for a nonzero's own products and six a step that add up as their root:
                # at most 2^-24 each, 0.58 of it root mean square where the adder truncates, times
                # the share of a partial sum in the whole (0.71 on average). 0.40 is measured.
                rel = np.linalg.norm(got - want) / np.linalg.norm(want)
                assert rel <= 0.5 * 2.0**-24 * np.sqrt(1 + 6 * min(nonzeros, k // 16 + 1)), tile


@pytest.mark.parametrize("m,n,k", [(1, 300, 1000), (20, 130, 400), (32, 513, 4096), (64, 64, 1024),
                                   (200, 130, 500)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_every_part_counts(stream, m, n, k, ta, tb):
    """AUTO and many depth ranges in every layout, full mantissas: the 2-norm error stays under 0.3
    sqrt(k) 2^-24 (test_no_larger_error_than_fp32_chains), where losing the third part of either
    operand (2^-19 of it root mean square) alone would be 1.9e-6, past the bound at any depth here."""
    a, b = normal((m, k), 13), normal((k, n), 14)
    want = a.astype(np.float64) @ b.astype(np.float64)
    a_d = mf.DeviceArray.from_numpy(np.ascontiguousarray(a.T if ta else a), stream)
    b_d = mf.DeviceArray.from_numpy(np.ascontiguousarray(b.T if tb else b), stream)
    for tile, splits in ((0, 0), (0, 1), (mf.abi.TILE_64x64, 12), (mf.abi.TILE_128x64, 3)):
        got = mf.gemm(a_d, b_d, trans_a=ta, trans_b=tb, tile=tile, splits=splits).numpy()
        rel = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert rel <= 0.3 * np.sqrt(k) * 2.0**-24, (tile, splits, rel)


@pytest.mark.parametrize("tile", TILES)
def test_identity_gives_b_exactly(stream, tile):
    """The identity times b: every part of b counts (test_extreme_operands has a times it)."""
    for m, n in ((300, 260), (20, 150), (130, 70)):
        b = normal((m, n), 15)
        got = mf.gemm(mf.DeviceArray.from_numpy(np.eye(m, dtype=np.float32), stream),
                      mf.DeviceArray.from_numpy(b, stream), tile=tile, splits=1).numpy()
        assert np.array_equal(got, b)
