"""The matrix-core kernels' workgroup tiles (32 x 32, 64 x 64, 64 x 128 and 128 x
128 rows x outputs) against the oracle, bit for bit: whole and ragged rows and
outputs, one stage of 8 blocks to more than the ring of buffers holds, a bias,
a weight row slice, scales that are subnormal or not finite, a residual."""
import numpy as np
import pytest

from llama_fixtures import random_llama
from oracle import oracle
import tensomite_hip as th

pytestmark = pytest.mark.gpu

FORMATS = ["Q8_0", "Q4_0", "Q4_1"]


@pytest.fixture(scope="module")
def dev():
    return th.HIPDevice(0)


# (rows, outputs, k): on 256 compute units, 32 x 32 tiles up to one round,
# 64 x 64 up to one round, then 64 x 128 and 128 x 128; k from 1 stage to 6
SHAPES = [(32, 32, 256), (45, 203, 512), (97, 1990, 1536), (100, 130, 1280), (129, 3000, 768), (100, 16350, 256),
          (65, 16384, 1024), (512, 8192, 512), (400, 9001, 768), (385, 8065, 256)]


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("shape", SHAPES)
def test_matrix_tiles(dev, fmt, shape):
    rows, n, k = shape
    print("matrix tiles", fmt, rows, n, k, flush=True)
    rng = np.random.default_rng(rows + n + k)
    w = oracle.quantize(fmt, rng.normal(0, 0.02, (n + 8) * k).astype(np.float32))
    x = rng.normal(0, 1, (rows, k)).astype(np.float32)
    x[rows // 2] *= 1e-6  # scales that are subnormal halves
    bias = rng.normal(0, 1, n).astype(np.float32)
    rb = th.row_bytes(fmt, k)
    wb, xb = dev.from_array(w), dev.from_array(x)
    for first, b in ((0, None), (8, bias)):
        got = dev.block_matmul(fmt, wb, xb, rows, n, k, bias=None if b is None else dev.from_array(b), w_row=first)
        got = dev.to_array(got, np.float32, rows * n).reshape(rows, n)
        dev.sync()
        want = oracle.matmul(fmt, x, w[first * rb:(first + n) * rb], rows, n, k)
        if b is not None:
            want = want + b
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), first


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("shape", [(40, 200, 512), (100, 16384, 256), (256, 16384, 256)])
def test_scales_not_finite(dev, fmt, shape):
    # infinite and NaN block scales reach their own outputs and no others
    rows, n, k = shape
    rng = np.random.default_rng(n)
    w = oracle.quantize(fmt, rng.normal(0, 0.02, n * k).astype(np.float32)).copy()
    bb = th.BLOCK_BYTES[th.KINDS[fmt]]
    for row, bits in ((3, 0x7c00), (n - 1, 0xfc00), (n // 2, 0x7e00)):
        at = (row * (k // 32) + 5) * bb
        w[at:at + 2] = np.frombuffer(np.uint16(bits).tobytes(), np.uint8)
    x = rng.normal(0, 1, (rows, k)).astype(np.float32)
    x[7, 40] = np.inf
    x[rows - 1, 64] = np.nan
    got = dev.block_matmul(fmt, dev.from_array(w), dev.from_array(x), rows, n, k)
    got = dev.to_array(got, np.float32, rows * n).reshape(rows, n)
    dev.sync()
    with np.errstate(all="ignore"):
        want = oracle.matmul(fmt, x, w, rows, n, k)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])


# (width, ids): the residual added in the product, where the 32 x 32 tiles, the
# 64 x 64 and the 64 x 128 take it, and at a width that none of them takes
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("width,ids", [(256, 32), (256, 45), (576, 33), (1024, 300), (2048, 520)])
def test_residual_in_the_product(dev, fmt, width, ids):
    print("residual", fmt, width, ids, flush=True)
    config = dict(layers=1, width=width, heads=2, kv_heads=1, head_width=64, hidden=352 if width == 576 else 256,
                  vocab=300, context=ids, eps=1e-5, theta=10000.0, kind=fmt)
    weights = random_llama(config, seed=width + ids, norm_jitter=0.1)
    prompt = list(np.random.default_rng(ids).integers(0, config["vocab"], ids))
    got = th.HIPLlama(dev, config, weights, rows=1, capacity=ids, max_tokens=ids).forward(prompt, last_only=False)
    want = oracle.Llama(config, weights).forward(prompt, last_only=False)
    got, want = np.asarray(got, np.float32).reshape(ids, -1), np.asarray(want, np.float32).reshape(ids, -1)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
