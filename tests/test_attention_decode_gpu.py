"""Attention of 1 to 4 queries (the decode form): key counts around a wavefront's and a range's
edges, every head size, masks, causal, broadcast keys, NaN and fully masked rows, against float64
with the fused kernel's bound 1e-5 * sqrt(lk) of sum_j |p_ij v_jc|."""
import numpy as np
import pytest

import mensurflow_amd as mf

pytestmark = pytest.mark.gpu


def reference(q, k, v, keep):
    """Output and its magnitude sum_j p_ij |v_jc| in float64; keep [.., lq, lk] of booleans."""
    q, k, v = (t.astype(np.float64) for t in (q, k, v))
    s = q @ np.swapaxes(k, -1, -2) / np.sqrt(q.shape[-1])
    s = np.where(keep, s, -np.inf)
    top = np.max(s, axis=-1, keepdims=True)
    p = np.exp(s - np.where(np.isfinite(top), top, 0.0))
    total = p.sum(axis=-1, keepdims=True)
    p = np.divide(p, total, out=np.zeros_like(p), where=total > 0)
    return p @ v, p @ np.abs(v)


def check(stream, batch, lq, lk, d, causal=False, masked=False, broadcast=False, seed=0):
    rng = np.random.default_rng(seed)
    kv_batch = (batch[0],) + (1,) * (len(batch) - 1) if broadcast else batch
    q = rng.standard_normal(batch + (lq, d)).astype(np.float32)
    k = rng.standard_normal(kv_batch + (lk, d)).astype(np.float32)
    v = rng.standard_normal(kv_batch + (lk, d)).astype(np.float32)
    keep = np.ones(batch + (lq, lk), bool)
    mask_d = None
    if masked:
        keep = rng.random(batch + (lq, lk)) < 0.6
        keep[..., 0, :] = False  # a fully masked row
        mask_d = mf.DeviceArray.from_numpy(keep.astype(np.uint8), stream)
    if causal:
        keep = keep & np.tril(np.ones((lq, lk), bool))
    dev = lambda x: mf.DeviceArray.from_numpy(x, stream)  # noqa: E731
    got = mf.attention_fused(dev(q), dev(k).expand(batch + (lk, d)), dev(v).expand(batch + (lk, d)),
                             mask=mask_d, causal=causal).numpy()
    want, scale = reference(q, k, v, keep)
    bound = 1e-5 * np.sqrt(lk) * scale
    assert np.all(np.abs(got - want) <= bound), (batch, lq, lk, d, causal, masked)


@pytest.mark.parametrize("d", [16, 32, 48, 64, 80, 96, 112, 128])
@pytest.mark.parametrize("lq,lk", [(1, 1), (1, 7), (1, 255), (2, 256), (3, 257), (4, 1000),
                                   (1, 4097), (4, 16384)])
def test_head_sizes_and_key_counts(stream, d, lq, lk):
    check(stream, (2, 3), lq, lk, d, seed=d + lk)


@pytest.mark.parametrize("lq,lk", [(1, 33), (2, 300), (4, 2049)])
def test_masks_causal_broadcast(stream, lq, lk):
    for d in (32, 64, 128):
        check(stream, (2, 3), lq, lk, d, causal=True, seed=1)
        check(stream, (2, 3), lq, lk, d, masked=True, seed=2)
        check(stream, (2, 4), lq, lk, d, masked=True, causal=True, broadcast=True, seed=3)
    check(stream, (300, 5), lq, lk, 64, seed=4)  # as many heads as ranges fill the chip: one range
    check(stream, (), lq, lk, 64, seed=5)


def test_nan_and_infinite_keys(stream):
    """A NaN score makes its row NaN and leaves other rows alone, in the last range too."""
    for lk in (100, 5000):
        rng = np.random.default_rng(lk)
        q, k, v = (rng.standard_normal((3, n, 64)).astype(np.float32) for n in (2, lk, lk))
        k[1, lk - 1, 5] = np.nan
        dev = lambda x: mf.DeviceArray.from_numpy(x, stream)  # noqa: E731
        got = mf.attention_fused(dev(q), dev(k), dev(v)).numpy()
        assert np.all(np.isnan(got[1])) and np.all(np.isfinite(got[[0, 2]]))
        want, scale = reference(q, k, v, np.ones((3, 2, lk), bool))
        assert np.all(np.abs(got - want)[[0, 2]] <= 1e-5 * np.sqrt(lk) * scale[[0, 2]])


@pytest.mark.parametrize("lq,lk", [(1, 1), (1, 5000), (2, 300), (3, 2), (4, 4096), (40, 50)])
@pytest.mark.parametrize("d", [32, 64, 80])
def test_causal_reads_no_key_past_the_queries(stream, d, lq, lk):
    """A long buffer whose keys and values past the queries were never written."""
    rng = np.random.default_rng(lk)
    q, k, v = (rng.standard_normal((2, 3, n, d)).astype(np.float32) for n in (lq, lk, lk))
    keep = np.tril(np.ones((lq, lk), bool))
    want, scale = reference(q, k, v, keep)
    k[..., lq:, :], v[..., lq:, :] = np.nan, np.inf
    dev = lambda x: mf.DeviceArray.from_numpy(x, stream)  # noqa: E731
    got = mf.attention_fused(dev(q), dev(k), dev(v), causal=True).numpy()
    assert np.all(np.abs(got - want) <= 1e-5 * np.sqrt(lk) * scale)


@pytest.mark.parametrize("lk", [300, 5000])
def test_scale_applies_to_the_scores(stream, lk):
    """scale q overflows where scale (q k) is ordinary."""
    rng = np.random.default_rng(lk)
    q, k, v = (rng.standard_normal((2, 3, n, 64)).astype(np.float32) for n in (1, lk, lk))
    q, k = q * np.float32(2.0**112), k * np.float32(2.0**-132)
    want, scale = reference(q.astype(np.float64) * 2.0**20, k, v, np.ones((1, lk), bool))
    dev = lambda x: mf.DeviceArray.from_numpy(x, stream)  # noqa: E731
    got = mf.attention_fused(dev(q), dev(k), dev(v), scale=2.0**20 / 8).numpy()
    assert np.all(np.abs(got - want) <= 1e-5 * np.sqrt(lk) * scale)


@pytest.mark.parametrize("d,lq,lk", [(16, 2, 256), (32, 2, 128), (64, 3, 128), (32, 4, 256),
                                     (32, 4, 2048), (128, 4, 64), (48, 4, 256), (16, 3, 1024)])
def test_form_lines(stream, d, lq, lk):
    """Both sides of the lines between the decode form and the tile kernels, in keys and heads."""
    for heads in (127, 128, 129, 257):
        for keys in (lk - 1, lk):
            check(stream, (heads,), lq, keys, d, seed=heads + keys)


def test_captured_call_keeps_no_workspace():
    """A captured call's graph is replayed after eager calls on the same stream have used and grown
    the stream's workspace, and after the inputs changed."""
    import ctypes

    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime that the library has loaded

    def call(name, *args):
        assert getattr(hip, name)(*args) == 0, name

    heads, lk, d = 6, 4096, 64
    rng = np.random.default_rng(7)
    host = lambda n: rng.standard_normal((heads, n, d)).astype(np.float32)  # noqa: E731
    with mf.Stream(0) as stream:
        q, k, v = (mf.DeviceArray.from_numpy(host(n), stream) for n in (1, lk, lk))
        out = mf.DeviceArray.empty((heads, 1, d), stream)

        def check():
            want, scale = reference(q.numpy(), k.numpy(), v.numpy(), np.ones((heads, 1, lk), bool))
            assert np.all(np.abs(out.numpy() - want) <= 1e-5 * np.sqrt(lk) * scale)

        mf.attention_fused(q, k, v, out=out)  # the workspace holds the ranges' results from here on
        check()
        handle = ctypes.c_void_p(stream.hip_stream())
        graph, run = ctypes.c_void_p(), ctypes.c_void_p()
        thread_local = 1  # hipStreamCaptureModeThreadLocal
        call("hipStreamBeginCapture", handle, ctypes.c_int(thread_local))
        mf.attention_fused(q, k, v, out=out)
        call("hipStreamEndCapture", handle, ctypes.byref(graph))
        call("hipGraphInstantiate", ctypes.byref(run), graph, None, None, ctypes.c_size_t(0))
        for size in (256, 4096, 16384):  # y = A^T x: partial sums, a larger workspace each time
            a = mf.DeviceArray.from_numpy(rng.standard_normal((2048, size)).astype(np.float32), stream)
            x = mf.DeviceArray.from_numpy(rng.standard_normal(2048).astype(np.float32), stream)
            mf.sgemv(a, x, trans=True)
            q.upload(host(1))
            v.upload(host(lk))
            mf.fill(out, 7.0)
            call("hipGraphLaunch", run, handle)
            check()
        call("hipGraphExecDestroy", run)
        call("hipGraphDestroy", graph)
