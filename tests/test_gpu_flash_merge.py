"""The merge of a long context's chunk partials (flash_decode_f16 past 16 chunks of 64 positions): 16 chunks (the
short merge), 17, a last round of one chunk, many rounds, whole wavefronts' chunks masked; head sizes 64 and 128.
Against float64 within (8 sqrt(T) 2^-24 + 2^-19) of sum_j p_j |v_j| / sum_j p_j: the f32 sums and exponents."""
import numpy as np
import pytest

import kernelcore_amd as kc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def runtime():
    kc.init()
    yield
    kc.synchronize()


@pytest.mark.parametrize("T,D,H,K,N,hole", [(1024, 128, 8, 2, 1, False), (1025, 128, 6, 2, 2, False), (1100, 64, 8, 1, 1, True),
                                            (4161, 128, 4, 4, 1, True), (4161, 64, 16, 2, 3, True), (16384, 128, 8, 1, 1, False)])
def test_long_context_merge(T, D, H, K, N, hole):
    print(f"flash merge T={T} D={D} H={H}/{K} N={N}", flush=True)
    r = np.random.default_rng(T + D)
    q = r.standard_normal((N, H, D)).astype(np.float32)
    k, v = (r.standard_normal((T, K, D)).astype(np.float16) for _ in range(2))
    tp = (T + 7) // 8 * 8
    mask = np.zeros((N, tp), np.float16)
    if hole:  # all of the first eight chunks but one position, every chunk of wavefront 3, the tail
        mask[:, 1:512] = -np.inf
        for c in range(3, (T + 63) // 64, 8):
            mask[:, 64 * c:64 * c + 64] = -np.inf
        mask[:, T - 5:] = -np.inf
    bufs = [kc.Buffer.of(a) for a in (q, k, v, mask)]
    out, part = kc.Buffer(4 * N * H * D), kc.Buffer(4 * N * H * ((T + 63) // 64) * (D + 2))
    d = kc.FaDims(H=H, T=T, D=D, group=H // K, tp=tp, k_row=K * D // 2, k_head=D // 2, v_row=K * D // 2, v_head=D // 2, N=N,
                  q_tok=H * D, q_head=D, m_row=tp // 2, has_mask=1, H_kv=K)
    kc.launch("flash_decode_f16", kc.FlashDecodeArgs(*[b.ptr for b in bufs], out.ptr, part.ptr, None, d, 0.1))
    got = out.download(np.float32).reshape(N, H, D)
    for h in range(H):
        s = 0.1 * q[:, h].astype(np.float64) @ k[:, h // (H // K)].astype(np.float64).T + mask[:, :T].astype(np.float64)
        p = np.exp(s - s.max(1, keepdims=True))
        p /= p.sum(1, keepdims=True)
        v64 = v[:, h // (H // K)].astype(np.float64)
        bound = (8 * np.sqrt(T) * 2.0 ** -24 + 2.0 ** -19) * (p @ np.abs(v64))
        assert (np.abs(got[:, h] - p @ v64) <= bound).all()
    for b in bufs + [out, part]:
        b.free()
