"""The few-rows matrix-core kernel (9 to 16 activation rows) against the oracle,
bit for bit: rows of whole stages of 32 blocks and of 16, one stage to many,
ragged rows and outputs, narrow (a compute unit a workgroup) and wide, a bias, a
weight row slice, and scales that are subnormal or not finite."""
import numpy as np
import pytest

from oracle import oracle
import tensomite_hip as th

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return th.HIPDevice(0)


@pytest.mark.parametrize("fmt", ["Q8_0", "Q4_0", "Q4_1"])
@pytest.mark.parametrize("rows,n,k", [(9, 16, 512), (16, 1, 1024), (13, 203, 1536), (16, 250, 2048), (10, 65, 3072),
                                      (16, 144, 8192), (12, 4096, 1024), (11, 4100, 1024)])
def test_few_rows(dev, fmt, rows, n, k):
    print("few rows", fmt, rows, n, k, flush=True)
    rng = np.random.default_rng(rows + n + k)
    w = oracle.quantize(fmt, rng.normal(0, 0.02, (n + 8) * k).astype(np.float32)).copy()
    w[(n // 2 + 8) * th.row_bytes(fmt, k):][:2] = np.frombuffer(np.uint16(0x7c00).tobytes(), np.uint8)
    x = rng.normal(0, 1, (rows, k)).astype(np.float32)
    x[rows // 2] *= 1e-6  # scales that are subnormal halves
    bias = rng.normal(0, 1, n).astype(np.float32)
    rb = th.row_bytes(fmt, k)
    wb, xb = dev.from_array(w), dev.from_array(x)
    for first, b in ((0, None), (8, bias)):
        got = dev.block_matmul(fmt, wb, xb, rows, n, k, bias=None if b is None else dev.from_array(b), w_row=first)
        got = dev.to_array(got, np.float32, rows * n).reshape(rows, n)
        dev.sync()
        with np.errstate(all="ignore"):
            want = oracle.matmul(fmt, x, w[first * rb:(first + n) * rb], rows, n, k)
            if b is not None:
                want = want + b
        nan = np.isnan(want)
        assert np.array_equal(np.isnan(got), nan), first
        assert np.array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan]), first
