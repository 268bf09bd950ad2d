"""The fused attention on the bf16 matrix cores where its parts could miss the fp32 values: infinite,
NaN, huge and tiny operands, in the first and the last key block, causal and masked, for every head
size and both workgroup sizes; against float64 with the fused kernel's bound."""
import numpy as np
import pytest

import mensurflow_amd as mf

pytestmark = pytest.mark.gpu


def reference(q, k, v, keep, scale=None):
    with np.errstate(all="ignore"):
        s = q.astype(np.float64) @ np.swapaxes(k.astype(np.float64), -1, -2)
        s = s * (1 / np.sqrt(q.shape[-1]) if scale is None else scale)
        s = np.where(keep, s, -np.inf)
        top = np.max(s, axis=-1, keepdims=True)
        p = np.exp(s - np.where(top == -np.inf, 0.0, top))
        total = p.sum(axis=-1, keepdims=True)
        p = np.where(total == 0, 0.0, p / total)
        out = np.zeros(q.shape[:-1] + (v.shape[-1],))
        mag = np.zeros_like(out)
        # A removed key adds nothing here; the weight 0 of a kept one still meets its value.
        for idx in np.ndindex(q.shape[:-2]):
            out[idx] = p[idx] @ v[idx].astype(np.float64)
            mag[idx] = p[idx] @ np.abs(v[idx].astype(np.float64))
    return out, mag


@pytest.mark.parametrize("d", [32, 64, 96, 128])
@pytest.mark.parametrize("case", ["value inf", "value nan", "key -inf", "key nan", "huge value",
                                  "tiny values", "huge scores", "tiny keys", "tiny queries",
                                  "huge scale", "small values", "smaller values", "one tiny value",
                                  "tiny column", "values of the least weights"])
def test_extreme_operands(stream, d, case):
    for batch, lq, lk, causal in (((2,), 70, 150, False), ((2,), 260, 260, True),
                                  ((70, 4), 300, 64, False)):
        rng = np.random.default_rng(d)
        q = rng.standard_normal(batch + (lq, d)).astype(np.float32)
        k = rng.standard_normal(batch + (lk, d)).astype(np.float32)
        v = rng.standard_normal(batch + (lk, d)).astype(np.float32)
        one = (0,) * len(batch)
        if case == "value inf":
            v[one + (0, 3)] = np.inf   # kept by every query
        elif case == "value nan":
            v[one + (0, d - 1)] = np.nan
        elif case == "key -inf":
            q[..., 0] = np.abs(q[..., 0]) + 0.1
            k[one + (5, 0)] = -np.inf  # a weight of 0
        elif case == "key nan":
            k[one + (0, 1)] = np.nan
        elif case == "huge value":
            v[one + (0, slice(None))] = 3.4e38  # above the largest bf16
            v[one + (slice(1, None), slice(None))] = 0.0
        elif case == "tiny values":
            v *= np.float32(1e-37)
        elif case == "huge scores":
            q *= np.float32(1e18)
            k *= np.float32(1e18)
        elif case in ("tiny keys", "tiny queries"):  # ordinary scores of parts under 2^-126
            q, k = q * np.float32(1e36), k * np.float32(1e-36)
            if case == "tiny queries":
                q, k = q * np.float32(1e-36) * np.float32(1e-36), k * np.float32(1e36) * np.float32(1e36)
        elif case == "huge scale":  # scale q overflows, scale (q k) does not
            q, k = q * np.float32(1e35), k * np.float32(1e-39)
        elif case == "small values":
            v *= np.float32(2.0**-60)
        elif case == "smaller values":
            v *= np.float32(2.0**-95)
        elif case == "one tiny value":
            v[one + (0, 0)] = 1e-37
        elif case == "tiny column":
            v[..., 1] *= np.float32(1e-33)
        elif case == "values of the least weights":  # the likeliest keys' values are 0
            # Scores up to 25 in size: their rounding moves a weight by 25 * 2^-22, 6e-6 of it.
            k *= np.float32(4.0)
            top = np.argmax(q @ np.swapaxes(k, -1, -2), axis=-1)
            for idx in np.ndindex(batch):
                v[idx][np.unique(top[idx]), 2] = 0.0
        scale = 1e4 if case == "huge scale" else None
        keep = np.tril(np.ones((lq, lk), bool)) if causal else np.ones((lq, lk), bool)
        dev = lambda x: mf.DeviceArray.from_numpy(x, stream)  # noqa: E731
        got = mf.attention_fused(dev(q), dev(k), dev(v), causal=causal, scale=scale or 0.0).numpy()
        want, mag = reference(q, k, v, keep, scale)
        what = (case, d, batch, lq, lk)
        assert np.array_equal(np.isnan(got), np.isnan(want)), what
        ok = np.isfinite(want)
        assert np.array_equal(got[~ok & ~np.isnan(want)], want[~ok & ~np.isnan(want)]), what
        if case != "huge scores":  # there the scores' own rounding moves the weights
            bound = 1e-5 * np.sqrt(lk) * mag + lk * 2.0**-149
            assert np.all(np.abs(got[ok] - want[ok]) <= bound[ok]), what


@pytest.mark.parametrize("form", ["row", "rows", "strided"])
def test_mask_forms(stream, form):
    """A mask row shared by all queries, a row each, and a row whose bytes are not adjacent, with
    key counts around the 4-byte words and the 32-key blocks."""
    for d in (32, 64, 128):
        for lk in (5, 32, 63, 97, 130):
            rng = np.random.default_rng(lk)
            b, lq = 3, 40
            q, k, v = (rng.standard_normal((b, n, d)).astype(np.float32) for n in (lq, lk, lk))
            dev = lambda x: mf.DeviceArray.from_numpy(np.ascontiguousarray(x), stream)  # noqa: E731
            if form == "row":
                keep = rng.random((b, 1, lk)) < 0.5
                mask = dev(keep.astype(np.uint8))
            elif form == "rows":
                keep = rng.random((b, lq, lk)) < 0.5
                keep[:, 3] = False
                mask = dev(keep.astype(np.uint8))
            else:
                keep = rng.random((b, lq, lk)) < 0.5
                mask = dev(np.swapaxes(keep, 1, 2).astype(np.uint8)).T
            full = np.broadcast_to(keep, (b, lq, lk))
            got = mf.attention_fused(dev(q), dev(k), dev(v), mask=mask).numpy()
            want, mag = reference(q, k, v, full)
            assert np.all(np.abs(got - want) <= 1e-5 * np.sqrt(lk) * mag), (form, d, lk)


@pytest.mark.parametrize("d", [32, 64, 96, 128])
def test_causal_rerun_reads_no_key_past_the_wavefront(stream, d):
    """A value too small for its parts sends every wavefront through the fp32 matrix cores again;
    the wavefronts whose queries come before a non-finite value stay finite."""
    for batch, n in (((2,), 200), ((70, 4), 500)):  # 4 and 8 wavefronts a workgroup
        rng = np.random.default_rng(d)
        q, k, v = (rng.standard_normal(batch + (n, d)).astype(np.float32) for _ in range(3))
        v[..., :64, 0] = 1e-37
        keep = np.tril(np.ones((n, n), bool))
        want, mag = reference(q, k, v, keep)
        v[..., 64:, 1] = np.nan  # from the third wavefront's first query on
        dev = lambda x: mf.DeviceArray.from_numpy(x, stream)  # noqa: E731
        got = mf.attention_fused(dev(q), dev(k), dev(v), causal=True).numpy()
        bound = 1e-5 * np.sqrt(n) * mag + n * 2.0**-149
        assert np.all(np.abs(got - want)[..., :64, :] <= bound[..., :64, :]), (d, batch)
        assert np.all(np.isnan(got[..., 96:, 1])), (d, batch)


@pytest.mark.parametrize("d", [64, 96])
@pytest.mark.parametrize("lq,lk", [(5, 512), (128, 512), (128, 513), (129, 100), (33, 33)])
def test_workgroup_sizes(stream, d, lq, lk):
    """Workgroups of 4 and of 8 wavefronts, on enough heads for either."""
    rng = np.random.default_rng(lq + lk)
    q, k, v = (rng.standard_normal((520, n, d)).astype(np.float32) for n in (lq, lk, lk))
    dev = lambda x: mf.DeviceArray.from_numpy(x, stream)  # noqa: E731
    for causal in (False, True):
        keep = np.tril(np.ones((lq, lk), bool)) if causal else np.ones((lq, lk), bool)
        got = mf.attention_fused(dev(q), dev(k), dev(v), causal=causal).numpy()
        want, mag = reference(q[::40], k[::40], v[::40], keep)
        assert np.all(np.abs(got[::40] - want) <= 1e-5 * np.sqrt(lk) * mag), causal


@pytest.mark.parametrize("d", [32, 64, 96, 128])
@pytest.mark.parametrize("lq,lk", [(150, 1024), (520, 333)])
def test_every_part_counts(stream, d, lq, lk):
    """The 2-norm error on normal operands is the fp32 sums' own (2.8e-7 to 5.3e-7 measured): a lost
    part of q, k, v or the weights, 2^-17 of it, would be 10 times the bound."""
    rng = np.random.default_rng(d)
    q, k, v = (rng.standard_normal((3, n, d)).astype(np.float32) for n in (lq, lk, lk))
    dev = lambda x: mf.DeviceArray.from_numpy(x, stream)  # noqa: E731
    got = mf.attention_fused(dev(q), dev(k), dev(v)).numpy()
    want, _ = reference(q, k, v, np.ones((lq, lk), bool))
    assert np.linalg.norm(got - want) <= 8e-7 * np.linalg.norm(want)
