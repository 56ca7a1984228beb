"""The int8 prefill matmul of Q6_K (kmatmul_i8.hip) at the edges of its tiles: rows past a tile of 128 and of 16, ragged
columns, K ranges that do not start on a group of four super-blocks (the K split), 64 and 128 columns per workgroup, and
super-block sums past 2^24 (which the fp16 kernel rounds). Against the oracle's exact int32 sums: 6 + 2 nsb roundings of
2^-24 on the terms' sum of magnitudes (4 times: taken from the activations before their quantization); and bit-identical to the fp16 kernel where its sums are exact."""
import numpy as np
import pytest

import kernelcore_amd as kc
import oracle
from tests import kq
from tests.test_gpu_matmul import oracle_slots, run_matmul

pytestmark = pytest.mark.gpu
O = oracle.lib()


@pytest.fixture(scope="module", autouse=True)
def runtime():
    kc.init()
    yield
    kc.synchronize()


@pytest.mark.parametrize("rows,k,ncols", [(8, 1024, 64), (136, 1024, 65), (1000, 3072, 127), (264, 5120, 129), (2056, 1024, 200),
                                          (40, 12288, 96), (8200, 1024, 1040)])
def test_int8_prefill_matmul(rows, k, ncols):
    print(f"int8 prefill {rows}x{k} ncols={ncols}", flush=True)
    w = kq.random_blocks("q6k", rows, k, seed=rows + k + ncols)
    x = kq.randn(k * ncols, ncols + rows, 1.5)
    y, _ = run_matmul("q6k", True, w, x, rows, k, ncols)
    kc.set_option("matmul_ws", 2)  # the fp16 producer-wavefront kernel, the same K split
    yf, _ = run_matmul("q6k", True, w, x, rows, k, ncols)
    kc.set_option("matmul_ws", 0)
    assert np.array_equal(kq.bits(y), kq.bits(yf))
    check(w, x, y, rows, k, ncols)


def test_int8_prefill_sums_past_24_bits():
    rows, k, ncols = 48, 1024, 70
    blocks = kq.random_blocks("q6k", rows, k, seed=5).view(np.uint8).reshape(-1, 210).copy()
    blocks[:, :192] = 0xFF  # every q = 31
    blocks[:, 192:208] = np.where(np.arange(16) % 5, 127, 0x80)  # scales 127 and -128
    w = blocks.reshape(-1)
    x = np.abs(kq.randn(k * ncols, 3, 1.5)) + np.float32(3)
    y, _ = run_matmul("q6k", True, w, x, rows, k, ncols)
    check(w, x, y, rows, k, ncols)


@pytest.mark.parametrize("rows,ncols", [(48, 64), (16400, 200)])
def test_int8_prefill_infinite_column_scale(rows, ncols):
    """A column whose slot carries an infinite scale gives the oracle's infinities (64 and 128 columns per workgroup, the
    first super-block of each K range; columns of every block of 32), and leaves the others alone."""
    k = 1024
    w, x = kq.random_blocks("q6k", rows, k, seed=9), kq.randn(k * ncols, 4, 1.5)
    q = oracle_slots(x, k, ncols, True)
    at = {5: 0, 40: 0, 41: 2, 63: 1} | ({100: 0, 127: 2, 130: 0, 199: 0} if ncols == 200 else {})
    for c, s in at.items():
        q.reshape(ncols, -1)[c, k // 4 + s] = np.float32(np.inf).view(np.int32)
    stream, slots, y = kc.upload_weights("q6k", w, rows, k), kc.Buffer.of(q), kc.Buffer(4 * rows * ncols)
    kc.launch("matmul_q6k_q8kx8", kc.MatmulKQ8Args(stream.ptr, slots.ptr, y.ptr, None, rows, k, ncols, 8))
    got, want = y.download(np.float32).reshape(ncols, rows), np.zeros(rows * ncols, np.float32)
    O.kco_matmul_q6k_q8k(w, q, want, rows, k, ncols)
    want = want.reshape(ncols, rows)
    assert np.isinf(want[list(at)]).mean() > 0.9
    assert np.array_equal(got[list(at)], want[list(at)], equal_nan=True)
    assert np.isfinite(np.delete(got, list(at), 0)).all()
    for b in (stream, slots, y):
        b.free()


def check(w, x, y, rows, k, ncols):
    cols = np.unique(np.r_[0, ncols // 2, ncols - 1, np.arange(0, ncols, 67)])
    xs = np.ascontiguousarray(x.reshape(ncols, k)[cols]).reshape(-1)
    want = np.zeros(rows * len(cols), np.float32)
    O.kco_matmul_q6k_q8k(w, oracle_slots(xs, k, len(cols), True), want, rows, k, len(cols))
    scale = np.abs(oracle.dequant(O, "q6k", w, rows, k).reshape(rows, k)) @ np.abs(xs.reshape(len(cols), k)).T
    assert (np.abs(y[cols] - want.reshape(len(cols), rows)) <= (6 + 2 * k // 256) * 2.0 ** -24 * 4 * scale.T).all()
