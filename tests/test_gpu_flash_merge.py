"""The merge of a long context's chunk partials (flash_decode_f16 past 16 chunks of 64 positions): 16 chunks (the
short merge), 17, a last round of one chunk, many rounds, whole wavefronts' chunks masked; head sizes 64 and 128.
Against float64 within (8 sqrt(T) 2^-24 + 2^-19) of sum_j p_j |v_j| / sum_j p_j: the f32 sums and exponents.

And by bits against the partials merged in chunk order on the host: scores a whole number of doublings apart, so that every
factor is a power of two, chunks that are masked whole over infinite and NaN values (they must not reach the output), an
infinity in the last chunk that is not masked (it must)."""
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


LOG2E = np.float32(1.44269504)
LN2 = next(s for s in (np.float32(1) / LOG2E + np.float32(e * 2.0 ** -24) for e in (0, 1, -1)) if s * LOG2E == 1)


def chunk_order_merge(part):
    """One head's chunk partials [nch][D + 2] (sums, maximum, sum of p) merged one after the other in f32."""
    M, L, O = np.float32(-np.inf), np.float32(0), np.zeros(part.shape[1] - 2, np.float32)
    for p in part:
        m, l = p[-2], p[-1]
        if m == -np.inf:
            continue
        if m > M:
            f = np.exp2((M - m) * LOG2E)
            L, O, M = L * f, O * f, m
        x = (m - M) * LOG2E
        assert x == np.rint(x)
        L, O = L + l * np.exp2(x), O + p[:-2] * np.exp2(x)
    return O / L


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("nch", [16, 17, 64, 65, 129])
@pytest.mark.parametrize("live_inf", [False, True])
def test_merge_is_chunk_order_and_skips_masked_chunks(nch, D, live_inf):
    print(f"flash merge bits nch={nch} D={D} live_inf={live_inf}", flush=True)
    H, K, T = 4, 2, 64 * nch - 3
    r = np.random.default_rng(nch + D)
    q = np.zeros((1, H, D), np.float32)
    k, v = np.zeros((T, K, D), np.float16), r.standard_normal((T, K, D)).astype(np.float16)
    for h in range(H):  # head h's scores are LN2 times its own component of k: whole numbers, each chunk's largest 0, 1 or 2
        q[0, h, h % 2] = 1
        top = r.integers(0, 3, nch)
        k[:, h // 2, h % 2] = np.repeat(top, 64)[:T] - r.integers(0, 3, T) * (np.arange(T) % 64 != 5)
    tp = (T + 7) // 8 * 8
    mask = np.zeros((1, tp), np.float16)
    dead = [0, nch // 2] + ([] if live_inf else [nch - 1]) + ([62, 63] if nch > 64 else [])
    for i, c in enumerate(dead):
        mask[:, 64 * c:64 * c + 64] = -np.inf
        v[64 * c:64 * c + 64] = (np.inf, np.nan, -np.inf)[i % 3]
    if live_inf:
        v[64 * (nch - 1) + 5, :, 7] = np.inf
    bufs = [kc.Buffer.of(a) for a in (q, k, v, mask)]
    out, part = kc.Buffer(4 * H * D), kc.Buffer(4 * H * nch * (D + 2))
    d = kc.FaDims(H=H, T=T, D=D, group=H // K, tp=tp, k_row=K * D // 2, k_head=D // 2, v_row=K * D // 2, v_head=D // 2, N=1,
                  q_tok=H * D, q_head=D, m_row=tp // 2, has_mask=1, H_kv=K)
    kc.launch("flash_decode_f16", kc.FlashDecodeArgs(*[b.ptr for b in bufs], out.ptr, part.ptr, None, d, float(LN2)))
    got, parts = out.download(np.float32).reshape(H, D), part.download(np.float32).reshape(H, nch, D + 2)
    assert (parts[:, dead, D] == -np.inf).all() and np.isnan(parts[:, dead, :D]).all()
    for h in range(H):
        want = chunk_order_merge(parts[h])
        assert np.isinf(want[7]) == live_inf and np.isfinite(np.delete(want, 7)).all()
        assert np.array_equal(got[h].view(np.uint32), want.view(np.uint32)), h
    for b in bufs + [out, part]:
        b.free()
