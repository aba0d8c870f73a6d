"""The Q8_0 GEMM's tiles and their edges, bit for bit against the oracle, with
every kind of block scale: fp16 (the term's product from the MFMA's biased
result), fp32 (converted dots), and fp16 ones that are infinite or NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def backend():
    from funasrnet_amd.hip import HipBackend
    b = HipBackend(0, minimum_operations=0)
    yield b
    b.close()


def scales(rng, kind, rows, blocks):
    s = (rng.standard_normal((rows, blocks)) * 0.02).astype(np.float16)
    s[rng.random(s.shape) < 0.05] = 0
    s[0, 0], s[-1, -1] = np.float16(65504), np.float16(6e-8)
    if kind == "odd":
        s[rows // 2, blocks // 2], s[rows // 3, 0] = np.inf, np.nan
    s = s.astype(np.float32)
    return s * np.float32(1.0001) if kind == "fp32" else s


# Tiles of 32 x 32, 32 x 64 from 448 of them on, 64 x 64 from 512 on. Rows of less
# than 512 and of 640 are q8_gemm_short_kernel's at any size, in tiles by the number of
# waves.
@pytest.mark.parametrize("frames,cols,rows", [(4, 128, 1), (31, 384, 33), (33, 640, 31), (65, 1024, 65), (225, 256, 3969),
                                              (449, 384, 2047), (513, 128, 4033), (1023, 640, 2049)])
@pytest.mark.parametrize("kind", ["fp16", "fp32", "odd"])
def test_tiles(backend, oracle_lib, frames, cols, rows, kind):
    check_tiles(backend, oracle_lib, frames, cols, rows, kind)


# Longer rows: stages of eight blocks with four left over (896, 1152, 1408) and
# whole, up to 256 tiles of 32 x 32 and more (up to 1280 short rows, from 1408 on
# not), 32 x 64 (short rows at 896 with fp32 scales) and 64 x 64 (with fp32 scales
# from 2048 waves of 32 x 32 on).
@pytest.mark.parametrize("frames,cols,rows", [(33, 896, 31), (512, 768, 512), (513, 768, 512), (300, 1280, 1000),
                                              (300, 1408, 1000), (225, 896, 3969), (225, 1152, 3969), (513, 512, 4033),
                                              (513, 768, 4033), (449, 768, 4033)])
@pytest.mark.parametrize("kind", ["fp16", "fp32", "odd"])
def test_longer_rows(backend, oracle_lib, frames, cols, rows, kind):
    check_tiles(backend, oracle_lib, frames, cols, rows, kind)


def check_tiles(backend, oracle_lib, frames, cols, rows, kind):
    from funasrnet_amd.model import Q8Tensor
    rng = np.random.default_rng(frames + cols)
    x = rng.standard_normal((frames, cols)).astype(np.float32)
    x[0] = 0
    if kind == "odd":
        x[1, 3], x[2, 0] = np.nan, np.inf
    q = rng.integers(-128, 128, (rows, cols), dtype=np.int8)
    s = scales(rng, kind, rows, cols // 32)
    bias = rng.standard_normal(rows).astype(np.float32)
    out = np.empty(frames * rows, np.float32)
    assert backend.try_quantized_linear(x.ravel(), frames, Q8Tensor("w", q, s), bias, out)
    got, expected = out.reshape(frames, rows), oracle_lib.linear(x.ravel(), q, s, bias).reshape(frames, rows)
    nan = np.isnan(expected)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint32), expected[~nan].view(np.uint32))


# Last scales that are infinite or overflow with the dot, where the last stage
# of eight blocks has four left over, and where it has none.
@pytest.mark.parametrize("cols", [128, 256, 384, 896, 1024, 1152])
def test_last_scales(backend, oracle_lib, cols):
    from funasrnet_amd.model import Q8Tensor
    rng = np.random.default_rng(cols)
    frames, rows, blocks = 40, 70, cols // 32
    x = rng.standard_normal((frames, cols)).astype(np.float32)
    x[3] = 0
    q = rng.integers(-128, 128, (rows, cols), dtype=np.int8)
    s = (rng.random((rows, blocks)) * 0.02 + 0.001).astype(np.float32)
    s[5, -1], s[6, -1], s[7, -1], s[8, -1], s[9, 0] = np.inf, -np.inf, 3e38, np.nan, 3e38
    out = np.empty((frames, rows), np.float32)
    assert backend.try_quantized_linear(x.ravel(), frames, Q8Tensor("w", q, s), None, out)
    expected = oracle_lib.linear(x.ravel(), q, s).reshape(frames, rows)
    nan = np.isnan(expected)
    assert np.isinf(expected[:, 5]).sum() > frames // 2 and np.isinf(expected[:, 7]).sum() > frames // 2
    assert np.array_equal(np.isnan(out), nan)
    assert np.array_equal(out[~nan].view(np.uint32), expected[~nan].view(np.uint32))


# The lm_head of lock-step sessions: the few-frame kernel up to seven and below
# 12,288 rows, else the GEMM; vocabularies that end inside a workgroup's 128 rows.
@pytest.mark.parametrize("count", [7, 8, 13, 16])
@pytest.mark.parametrize("vocab", [33, 4001, 12287, 12288, 12389])
def test_session_heads(backend, count, vocab):
    from funasrnet_amd import model
    from funasrnet_amd.hip import HipDecoder
    weights = model.synthetic(model.small_config(layers=1, vocab=vocab), seed=vocab)
    parent = HipDecoder(backend, weights, capacity=32)
    sessions, alone = ([parent.session(32) for _ in range(count)] for _ in range(2))
    try:
        for i, (a, b) in enumerate(zip(sessions, alone)):
            x = np.random.default_rng(i).standard_normal((5, weights.config.width)).astype(np.float32)
            a.decode(x, 5)
            b.decode(x, 5)
        tokens = HipDecoder.generate_sessions(sessions, 6)
        assert np.array_equal(tokens, np.stack([d.generate(6) for d in alone]))
    finally:
        for d in [*sessions, *alone, parent]:
            d.close()
