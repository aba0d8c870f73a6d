"""FP32 projections and attention as products of bf16 planes: every tile shape
and its edges against float64 sums, and what the planes cannot hold against fp32
rules.

The bound of a projection is that of any fp32 sum of K products: (K + 2) roundings of 2^-24
relative to sum |x w| (the planes themselves lose 2^-25 of a product)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def backend():
    from funasrnet_amd.hip import HipBackend
    b = HipBackend(0, minimum_operations=0)
    yield b
    b.close()


def run(backend, x, w, b=None):
    out = np.full((x.shape[0], w.shape[0]), np.nan, np.float32)
    assert backend.try_linear(x, x.shape[0], w, b, out.reshape(-1))
    return out


def check(got, x, w, b=None):
    x, w = x.astype(np.float64), w.astype(np.float64)
    bias = 0.0 if b is None else b.astype(np.float64)
    bound = (x.shape[1] + 2) * 2.0**-24 * (np.abs(x) @ np.abs(w).T + np.abs(bias)) + 2.0**-149
    assert np.all(np.abs(got - (x @ w.T + bias)) <= bound)


# 32 x 32 tiles, 32 x 64 from 128 of them on, 64 x 128 from 224 (eight waves) and 257 (four) on.
@pytest.mark.parametrize("frames,cols,rows", [(5, 4, 1), (31, 33, 31), (33, 128, 33), (64, 132, 65), (511, 60, 500),
                                              (513, 96, 511), (1023, 36, 1793), (1025, 260, 2049), (2100, 31, 1100)])
@pytest.mark.parametrize("biased", [False, True])
def test_split_tiles(backend, frames, cols, rows, biased):
    rng = np.random.default_rng(frames)
    x = rng.standard_normal((frames, cols)).astype(np.float32)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    b = rng.standard_normal(rows).astype(np.float32) if biased else None
    check(run(backend, x, w, b), x, w, b)


# The same tiles above 192 columns and at odd widths, and either side of the sizes
# that fp32 MFMA takes: up to 256 tiles of 64 x 128 of 192 columns from 17 frames on,
# up to 320 and 513 to 600 of 64 columns, and up to 32 frames of 28,672 rows or more.
@pytest.mark.parametrize("frames,cols,rows", [(9, 193, 33), (31, 200, 31), (33, 257, 33), (64, 260, 65), (511, 196, 500),
                                              (513, 225, 511), (1023, 196, 1793), (2100, 199, 1100), (17, 65, 40),
                                              (16, 192, 31), (17, 192, 31), (1000, 192, 2100), (1001, 192, 2100),
                                              (2000, 64, 2000), (1280, 64, 2048), (1281, 64, 2048), (2048, 64, 2048),
                                              (2049, 64, 2048), (2432, 64, 2000), (1300, 64, 3600), (32, 196, 28672), (33, 196, 28672)])
def test_gemm_choice(backend, frames, cols, rows):
    rng = np.random.default_rng(cols)
    x = rng.standard_normal((frames, cols)).astype(np.float32)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    check(run(backend, x, w), x, w)


# The GEMV of one, up to four and up to eight frames: parts of a chunk of 1,024 k,
# aligned and not, and the row counts where four rows a wave and the GEMM begin.
@pytest.mark.parametrize("frames,cols,rows", [(1, 1, 1), (1, 63, 5), (1, 1023, 9), (1, 1028, 65537), (2, 4, 3),
                                              (3, 1025, 70), (4, 2052, 65541), (5, 1024, 6), (7, 67, 8192), (8, 5000, 33),
                                              (8, 64, 8193), (1, 6148, 11), (1, 255, 9), (2, 256, 66000), (4, 260, 33),
                                              (8, 192, 3072), (6, 191, 20), (5, 512, 4096), (8, 1024, 3841), (6, 516, 3073)])
def test_gemv(backend, frames, cols, rows):
    rng = np.random.default_rng(cols)
    x = rng.standard_normal((frames, cols)).astype(np.float32)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    b = rng.standard_normal(rows).astype(np.float32)
    check(run(backend, x, w, b), x, w, b)


@pytest.mark.parametrize("frames,cols,rows", [(1, 1024, 70), (1, 516, 65541), (3, 1028, 33), (8, 2052, 65), (40, 560, 100),
                                              (600, 132, 1100)])
def test_frames_at_any_float(backend, frames, cols, rows):
    """Device frames that start at a multiple of 4 bytes give the bits that aligned ones do."""
    from funasrnet_amd import device
    from funasrnet_amd.hip import HipFloatWeight
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((frames, cols)).astype(np.float32)
    weight = HipFloatWeight(backend, rng.standard_normal((rows, cols)).astype(np.float32))
    results = []
    for offset in range(4):
        held = np.zeros(x.size + 4, np.float32)
        held[offset:offset + x.size] = x.ravel()
        dx, out = device.DeviceArray.from_numpy(held), device.DeviceArray((frames, rows), np.float32)
        backend.linear_device(dx.ptr + 4 * offset, frames, weight, None, out.ptr)
        backend.synchronize()
        results.append(out.numpy())
    for r in results[1:]:
        assert np.array_equal(r.view(np.uint32), results[0].view(np.uint32))


# (Up to 192 columns these run on fp32 MFMA, odd widths on the planes again.)
@pytest.mark.parametrize("cols", [64, 65, 260, 517])
@pytest.mark.parametrize("frames,rows", [(40, 70), (400, 700), (1100, 2100)])
def test_split_range(backend, frames, cols, rows):
    """Zero frames, tiny and huge values, infinities and NaN."""
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((frames, cols)).astype(np.float32)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    x[3] = 0.0
    check(run(backend, x, w), x, w)
    for scale in (2.0**-60, 2.0**-110, 2.0**-120, 2.0**100):
        scaled = x.copy()
        scaled[7] *= np.float32(scale)
        check(run(backend, scaled, w), scaled, w)
    # Values below the smallest bf16 give sums of zero on the planes.
    for frame, col in ((7, 5), (frames - 1, cols - 1), (32, 0)):
        scaled = x.copy()
        scaled[frame] = 0.0
        scaled[frame, col] = 2.0**-140
        check(run(backend, scaled, w), scaled, w)
    x[5, 2], x[6, 1], x[9, 0] = np.inf, np.nan, np.float32(3.4e38)
    w = w.copy()
    w[:, 0] = np.abs(w[:, 0]) * np.float32(0.1)
    got = run(backend, x, w)
    sound = np.ones(frames, bool)
    sound[[5, 6]] = False
    check(got[sound], x[sound], w)
    assert np.all(np.isnan(got[6])) and np.array_equal(got[5], np.where(w[:, 2] < 0, -np.inf, np.inf).astype(np.float32))


@pytest.mark.parametrize("cols", [100, 101, 196])
@pytest.mark.parametrize("value", [2.0**21, 2.0**-90, np.inf])
def test_weights_outside_the_planes(backend, value, cols):
    rng = np.random.default_rng(1)
    x = rng.standard_normal((200, cols)).astype(np.float32)
    w = rng.standard_normal((130, cols)).astype(np.float32)
    w[4] = np.float32(value) * (np.sign(w[4]) if np.isfinite(value) else 1)
    got = run(backend, x, w)
    if np.isfinite(value):
        check(got, x, w)
    else:
        keep = np.arange(130) != 4
        check(got[:, keep], x, w[keep])
        assert not np.any(np.isfinite(got[:, 4]))


# Their kernels: 64 x 64 and 32 x 64 tiles, 32 x 64 with K over the waves, any K.
@pytest.mark.parametrize("frames,cols,rows", [(257, 68, 1000), (33, 132, 70), (65, 260, 65), (1025, 1024, 513), (130, 75, 67)])
@pytest.mark.parametrize("biased", [False, True])
def test_fp32_tiles(backend, frames, cols, rows, biased):
    rng = np.random.default_rng(cols)
    x = rng.standard_normal((frames, cols)).astype(np.float32)
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    w[rows - 1, cols - 1] = 2.0**21
    b = rng.standard_normal(rows).astype(np.float32) if biased else None
    check(run(backend, x, w, b), x, w, b)


@pytest.mark.parametrize("rows,cols,value,planes", [(300, 31, 1.0, False), (300, 32, 1.0, True), (70, 500, 1.0, True),
                                                    (70, 500, 2.0**21, False), (1, 1, 1.0, False)])
def test_planes_memory(backend, rows, cols, value, planes):
    """Planes are kept only where products use them: three bf16 a value, rows to 32, columns to 128."""
    from funasrnet_amd.hip import HipFloatWeight
    w = np.ones((rows, cols), np.float32)
    w[-1, -1] = value
    held = HipFloatWeight(backend, w).device_bytes
    padded = -(-rows // 32) * 32 * -(-cols // 128) * 128
    assert 0 <= held - w.nbytes - (6 * padded if planes else 0) < 32
    x = np.random.default_rng(rows).standard_normal((40, cols)).astype(np.float32)
    check(run(backend, x, w), x, w)


@pytest.mark.parametrize("cols", [100, 101, 196])
@pytest.mark.parametrize("value,partner", [(2.0**-135, 2.0**80), (2.0**-125, 2.0**100), (2.0**-118, 2.0**60)])
def test_tiny_weight_beside_ordinary_ones(backend, value, partner, cols):
    """An element that the planes do not hold, in a row of ordinary ones, against
    frames that are large there and zero elsewhere."""
    rng = np.random.default_rng(4)
    x = rng.standard_normal((70, cols)).astype(np.float32)
    w = rng.standard_normal((130, cols)).astype(np.float32)
    w[9, 6] = np.float32(value * 1.2345678)
    x[[3, 40]] = 0
    x[[3, 40], 6] = np.float32(partner)
    check(run(backend, x, w), x, w)


def attend(backend, q, k, v, heads):
    out = np.full(q.shape, np.nan, np.float32)
    assert backend.try_attention(q, k, v, q.shape[0], q.shape[1], heads, out.reshape(-1))
    return out


# Tiles of 64 queries, blocks of 32 keys, one to four key shares; either side of
# the lengths from which heads of 128 and 64 take the planes. The tolerance is the
# reference's device check's (AttentionGpuChecks.cs), relative to values of 4. On the planes,
# all rows but the peaked one together: 7e-7 (2-norm). The same products in numpy, added
# exactly, are within 1.6e-7 (the kernel's fp32 sums 2.2e-7 to 4.5e-7), and off by
# 9.8e-7 or more (33 frames on) without any one of the six, in the scores or in the
# outputs.
@pytest.mark.parametrize("frames,heads,size", [(1, 2, 96), (33, 1, 96), (63, 4, 96), (65, 8, 96), (399, 1, 128),
                                               (400, 4, 128), (449, 1, 128), (513, 3, 128), (1857, 4, 128),
                                               (640, 2, 64), (671, 8, 64), (1100, 8, 64)])
def test_split_attention(backend, oracle_lib, frames, heads, size):
    rng = np.random.default_rng(frames)
    width = heads * size
    q, k, v = (rng.uniform(-s, s, (frames, width)).astype(np.float32) for s in (3, 3, 4))
    q[0] *= 8  # one peaked row
    expected = oracle_lib.attention_f64(q, k, v, frames, width, heads)
    off = attend(backend, q, k, v, heads) - expected
    assert np.abs(off).max() <= 5e-5 * 4
    rest = slice(min(1, frames - 1), None)
    if (frames, size) != (399, 128):  # (that one runs on fp32 MFMA, in longer fp32 sums)
        assert np.linalg.norm(off[rest]) <= 7e-7 * np.linalg.norm(expected[rest])


# One, two, three and four key shares, of which each takes queries of its own here.
@pytest.mark.parametrize("frames,heads,size", [(65, 8, 96), (1068, 8, 64), (1400, 4, 128), (449, 3, 128), (400, 3, 128), (1001, 3, 128)])
def test_split_attention_range_shares(backend, oracle_lib, frames, heads, size):
    """Heads that the planes do not hold, for a large value, a tiny query and an infinite value of the last key."""
    rng = np.random.default_rng(frames)
    width = heads * size
    q, k, v = (rng.uniform(-2, 2, (frames, width)).astype(np.float32) for _ in range(3))
    v[5, 3] = 2.0**70
    q[frames // 2, size + 2] = 2.0**-101
    expected = oracle_lib.attention_f64(q, k, v, frames, width, heads)
    v[frames - 1, width - 1] = np.inf
    got = attend(backend, q, k, v, heads)
    assert np.all(got[:, -1] == np.inf)
    assert np.all(np.abs(got - expected)[:, :-1] <= (5e-5 * np.maximum(4, np.abs(expected)))[:, :-1])


@pytest.mark.parametrize("value", [2.0**-101, 2.0**70, np.inf, np.nan])
def test_split_attention_range(backend, oracle_lib, value):
    """A value that the planes do not hold moves its head, and only it, to fp32."""
    rng = np.random.default_rng(3)
    frames, heads, size = 450, 3, 128
    q, k, v = (rng.uniform(-2, 2, (frames, heads * size)).astype(np.float32) for _ in range(3))
    plain = attend(backend, q, k, v, heads)
    v[7, size + 5] = value
    got = attend(backend, q, k, v, heads)
    other = np.ones(heads * size, bool)
    other[size:2 * size] = False
    assert np.array_equal(got[:, other].view(np.uint32), plain[:, other].view(np.uint32))
    if np.isfinite(value):
        expected = oracle_lib.attention_f64(q, k, v, frames, heads * size, heads)
        assert np.all(np.abs(got - expected) <= 5e-5 * np.maximum(4, np.abs(expected)))
    else:
        assert not np.any(np.isfinite(got[:, size + 5]))
    # The workspace serves the next call as before.
    v[7, size + 5] = 1.0
    again = attend(backend, q, k, v, heads)
    assert np.all(np.isfinite(again)) and np.array_equal(again, attend(backend, q, k, v, heads))


@pytest.mark.parametrize("frames,heads,size", [(400, 2, 128), (1000, 4, 128), (640, 3, 64), (130, 4, 96)])
@pytest.mark.parametrize("scale", [1e4, 1e5, 1e8, 1e16])
def test_split_attention_large_scores(backend, frames, heads, size, scale):
    """Queries and keys far above 1: a row whose largest score stands out by more than
    two fp32 scores can be off ((size + 2) 2^-24 of sum |q k| each), and by 40 beyond (e^-40 of the
    rest), is that key's value; every other row is still a mean of values."""
    rng = np.random.default_rng(frames)
    q, k = (rng.uniform(-scale, scale, (frames, heads * size)).astype(np.float32) for _ in range(2))
    v = rng.uniform(-4, 4, (frames, heads * size)).astype(np.float32)
    got = attend(backend, q, k, v, heads)
    assert np.all(np.isfinite(got)) and np.abs(got).max() <= 4 * (1 + 2.0**-16)
    clear = 0
    for h in range(0, heads * size, size):
        qh, kh = (a[:, h:h + size].astype(np.float64) for a in (q, k))
        scores = qh @ kh.T
        top = scores.argmax(axis=1)
        gap = -np.diff(np.sort(scores, axis=1)[:, -2:][:, ::-1], axis=1)[:, 0]
        error = 2 * (size + 2) * 2.0**-24 * (np.abs(qh) @ np.abs(kh).T).max(axis=1)
        sure = gap > error + 40 * size**0.5
        assert np.array_equal(got[sure, h:h + size], v[top[sure], h:h + size])
        clear += sure.sum()
    assert clear > 0.9 * frames * heads


def test_attention_workspace_grows(oracle_lib):
    """Ever longer device calls on a busy stream return before it has drained, and
    also while the thread captures another stream."""
    import ctypes
    from funasrnet_amd import device
    from funasrnet_amd.hip import HipBackend, HipFloatWeight
    backend, rt = HipBackend(0, minimum_operations=0), device.runtime()
    other, graph = ctypes.c_void_p(), ctypes.c_void_p()
    assert rt.hipStreamCreate(ctypes.byref(other)) == 0
    rng = np.random.default_rng(8)
    weight = HipFloatWeight(backend, rng.standard_normal((512, 2048)).astype(np.float32))
    x, y = device.DeviceArray((4000, 2048), np.float32), device.DeviceArray((4000, 512), np.float32)
    x.fill_zero()
    calls = []
    for frames in (400, 640, 1000, 1001):
        q, k, v = (rng.uniform(-2, 2, (frames, 256)).astype(np.float32) for _ in range(3))
        calls.append((frames, (q, k, v), [device.DeviceArray.from_numpy(a) for a in (q, k, v)],
                      device.DeviceArray((frames, 256), np.float32)))
    device.synchronize()
    for frames, _, d, out in calls:
        for _ in range(400):  # some 20 ms of work
            backend.linear_device(x.ptr, 4000, weight, None, y.ptr)
        assert rt.hipStreamBeginCapture(other, 0) == 0  # global: this thread may not allocate by itself
        backend.attention_device(d[0].ptr, d[1].ptr, d[2].ptr, frames, 256, 2, out.ptr)
        assert rt.hipStreamEndCapture(other, ctypes.byref(graph)) == 0
        assert rt.hipStreamQuery(ctypes.c_void_p(backend.stream)) == 600  # hipErrorNotReady
        rt.hipGraphDestroy(graph)
    backend.synchronize()
    for frames, host, _, out in calls:
        assert np.abs(out.numpy() - oracle_lib.attention_f64(*host, frames, 256, 2)).max() <= 5e-5 * 2
    rt.hipStreamDestroy(other)
    backend.close()


def test_output_arrays(backend):
    """Results land in the caller's array, also one that the library cannot write."""
    rng = np.random.default_rng(2)
    x, w = rng.standard_normal((9, 40)).astype(np.float32), rng.standard_normal((6, 40)).astype(np.float32)
    plain = run(backend, x, w)
    wide = np.zeros((9, 6))
    assert backend.try_linear(x, 9, w, None, wide) and np.array_equal(wide, plain)
    every_other = np.zeros(2 * 9 * 6, np.float32)[::2]
    assert backend.try_linear(x, 9, w, None, every_other) and np.array_equal(every_other, plain.ravel())
    for strided in (np.zeros((9, 12), np.float32)[:, ::2], np.zeros((6, 9), np.float32).T, np.zeros((9, 8), np.float32)[:, 1:7]):
        assert backend.try_linear(x, 9, w, None, strided) and np.array_equal(strided, plain)
    same = rng.standard_normal((6, 6)).astype(np.float32)
    expected = run(backend, same.copy(), w[:, :6].copy())
    assert backend.try_linear(same, 6, w[:, :6].copy(), None, same) and np.array_equal(same, expected)
