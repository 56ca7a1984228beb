"""The short-batch per-256 matmul (kmatmul_short.hip) at the edges of its tiles: 1 to 4 blocks of 16 columns,
ragged columns and rows, slot rows that are not 16-byte aligned (k / 256 not a multiple of 4, and slots at an
odd word), rounds of super-blocks (long rows), both wavefront counts. Integer sums and the reference's float
operations in its order: bit-exact against the oracle."""
import numpy as np
import pytest

import kernelcore_amd as kc
import oracle
from tests import kq
from tests.model_weights import random_weights
from tests.test_gpu_matmul import oracle_slots

pytestmark = pytest.mark.gpu
O = oracle.lib()


@pytest.fixture(scope="module", autouse=True)
def runtime():
    kc.init()
    yield
    kc.synchronize()


@pytest.mark.parametrize("qtype", ["q4k", "q6k"])
@pytest.mark.parametrize("rows,k,ncols,shift", [
    (8, 256, 2, 0), (24, 1024, 16, 0), (40, 1024, 17, 0), (200, 1280, 33, 0), (1000, 2048, 63, 0), (16, 4096, 15, 0),
    (136, 12288, 40, 0), (24, 16384, 50, 0), (72, 8192, 62, 0), (48, 1024, 31, 1),
    (24, 8448, 50, 0), (72, 8192, 62, 1), (40, 33280, 17, 1),  # rounds without staging
    (9224, 1024, 2, 0), (13320, 2304, 2, 1),  # column tiles
])
def test_short_batch_is_bit_exact(qtype, rows, k, ncols, shift):
    print(f"short batch {qtype} {rows}x{k} ncols={ncols} shift={shift}", flush=True)
    w = kq.random_blocks(qtype, rows, k, seed=rows + k + ncols)
    x = kq.randn(k * ncols, ncols + rows, 1.5)
    q = oracle_slots(x, k, ncols, True)
    stream, y = kc.upload_weights(qtype, w, rows, k), kc.Buffer(4 * rows * ncols)
    at = kc.Buffer(q.nbytes + 4 * shift)
    at.upload(q, 4 * shift)
    kc.launch(f"matmul_{qtype}_q8kx8", kc.MatmulKQ8Args(stream.ptr, at.at(4 * shift), y.ptr, None, rows, k, ncols, 8))
    want = np.zeros(rows * ncols, np.float32)
    getattr(O, f"kco_matmul_{qtype}_q8k")(w, q, want, rows, k, ncols)
    assert np.array_equal(kq.bits(y.download(np.float32)), kq.bits(want))
    for b in (stream, at, y):
        b.free()


@pytest.mark.parametrize("n", [2, 37])
def test_grouped_short_batch_is_bit_exact(n):
    """The one launch of q / k / v and of gate / up with Q6_K parts first, last and between Q4_K ones (a driver's prompt, three
    layers): logits and caches by bits against a launch of column tiles per matrix."""
    cfg = dict(n_layer=3, n_embd=1280, n_head=10, n_head_kv=2, head_dim=128, n_ff=1280, n_vocab=1024, norm_eps=1e-5,
               rope_theta=500000.0, rope_neox=0, qk_norm=0, max_ctx=64, max_batch=64)
    types = [("q4k", "q4k", "q6k", "q4k", "q6k"), ("q6k", "q4k", "q4k", "q6k", "q4k"), ("q4k", "q6k", "q4k", "q6k", "q6k")]
    types = {(kc.TENSORS[name], layer): kc.QTYPE[t] for layer, ts in enumerate(types)
             for name, t in zip(("wq", "wk", "wv", "w_gate", "w_up"), ts)}
    print(f"short batch groups n={n}", flush=True)
    m = kc.Model(**cfg)
    for (tid, layer), data in random_weights(cfg, 5, types).items():
        m.set_tensor(tid, layer, data, types.get((tid, layer)))
    got = []
    for path in (0, 1):
        m.reset()
        kc.set_option("matmul_path", path)
        logits = m.forward(np.arange(3, 3 + n, dtype=np.int32))
        got.append([kq.bits(logits)] + [m.read_cache(i, which, 0, n) for i in range(3) for which in (0, 1)])
    kc.set_option("matmul_path", 0)
    assert np.isfinite(got[0][0].view(np.float32)).all()
    assert all(np.array_equal(a, b) for a, b in zip(*got))
    m.close()
