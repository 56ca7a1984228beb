// kmatmul_short.hip -- Y = W X for K-quant weights and a short batch of per-256 activation columns
// (gfx950): the per-256 matmul names below the prefill kernel's batch, and every projection of a
// prompt of that many tokens.
//
// The result is the reference's (kernels/llm/matmul_q4k_q8kx8.cu, matmul_q6k_q8kx8.cu, mirror
// llm/llm_reference.cpp:529-596) bit for bit: every super-block's two sums are exact 32-bit
// integers, its term is formed with the reference's float operations, and the terms are added in
// super-block order.
//
// What bounds it: the weight bytes (each read once per 64 columns) and, as the batch grows, the vector
// ALU. So the products run on v_mfma_i32_16x16x32_i8 (one 32-value sub-block of 16 rows times
// 16 columns per op, the activations' int8 words as they lie in the slots), and the sub-block scale is
// applied to the op's 4 sums per lane by a 24-bit multiply-add: 4 vector ops per op, whatever the scale,
// where scaling the weights before the op would need two ops per sub-block (6-bit scale times 4-bit
// value does not fit a byte). Q6_K's scales cover 16 values: each op takes half of its lanes' values
// (the other half zeroed), two ops per 32 values -- as many as the scaled weights in two bytes would take
// (kmatmul_i8.hip), a form not measured here.
//
// Measured (this kernel alone, against the column-tiled kernel): 8192 x 3072 Q4_K, 12 columns 23.0 -> 7.5 us,
// 37 columns 46.9 -> 12.4 us, 63 columns 68.7 -> 18.5 us; 3072 x 8192 Q6_K, 2 columns 21.2 -> 9.9 us, 12 columns
// 50.0 -> 9.7 us, 37 columns 50.9 -> 21.6 us. The weights' bytes alone take 2.2 and 3.2 us at 6.4 TB/s.
//
// One workgroup per 16-row tile and up to 64 columns; its wavefronts take the super-blocks in turn (so a
// small matrix still has its whole row of super-blocks in flight), each writes its super-blocks' terms
// to LDS, and after one barrier wavefront c adds column block c's terms in order. A matrix whose
// terms do not fit kLdsBytes runs in rounds.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "internal.hpp"
#include "kmatmul_short.hpp"
#include "kquant.hpp"
#include "kquant_device.hpp"

namespace kcamd {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));

constexpr int kLdsBytes = 80 * 1024;  // two workgroups per CU

__device__ __forceinline__ i32x4 mfma8(i32x2 a, i32x2 b, i32x4 c) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, a), __builtin_bit_cast(long, b), c, 0, 0, 0);
}

// Loads at (this lane's byte offset v) + (uniform byte offset s) + an immediate: one address register per
// lane and array, where pointers would take two per load. The slots are 4-byte aligned. Cache policy 2: non-temporal.
typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc bufRes(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
template <int NT = 0>
__device__ __forceinline__ i32x2 buf2(Rsrc b, uint32_t v, uint32_t s) {
    return __builtin_bit_cast(i32x2, __builtin_amdgcn_raw_buffer_load_b64(b, v, s, NT));
}
template <int NT = 0>
__device__ __forceinline__ i32x4 buf4(Rsrc b, uint32_t v, uint32_t s) {
    return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(b, v, s, NT));
}

// One super-block's pieces held by lane (r = lane % 16: the row, kg = lane / 16: the 8 of every 32
// values this lane feeds to the matrix op).
// (v0 = 16 r, vq = 16 r + 1024 (kg / 2) + 8 (kg % 2): byte offsets within a 256-byte chunk pair.)
template <bool Q6>
struct SbWeights;
template <>
struct SbWeights<false> {
    i32x4 hdr;    // d, dmin, the 12 scale / min bytes
    i32x2 q[4];   // qs bytes 32 j + 8 kg ..: sub-block 2j in the low nibbles, 2j + 1 in the high ones
    __device__ __forceinline__ void load(Rsrc w, int s, uint32_t v0, uint32_t vq) {
        const uint32_t o = (uint32_t)((s >> 2) * kQ4kSeg + (s & 3) * 256);
        hdr = buf4<2>(w, v0, o);
#pragma unroll
        for (int j = 0; j < 4; ++j) q[j] = buf2<2>(w, vq, o + (1 + 2 * j) * 1024);
    }
};
template <>
struct SbWeights<true> {
    i32x4 sc;         // 16 int8 scales
    uint32_t d;       // fp16
    i32x2 ql[2][2];   // [half n][a]: ql bytes 64 n + 32 a + 8 kg ..
    i32x2 qh[2];      // [half n]: qh bytes 32 n + 8 kg ..
    __device__ __forceinline__ void load(Rsrc w, int s, uint32_t v0, uint32_t vq) {
        const uint32_t seg = (uint32_t)((s >> 2) * kQ6kSeg), o = seg + (s & 3) * 256;
        sc = buf4<2>(w, v0, o + 12 * 1024);
        d = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(w, v0 >> 3, seg + kQ6kSlabs * 1024 + (s & 3) * 32, 0) & 0xFFFFu;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
#pragma unroll
            for (int a = 0; a < 2; ++a) ql[n][a] = buf2<2>(w, vq, o + (4 * n + 2 * a) * 1024);
            qh[n] = buf2<2>(w, vq, o + (8 + 2 * n) * 1024);
        }
    }
};

// is += sc p, one 24-bit multiply-add per value: the empty asm keeps the sums in this order (regrouped as
// sums of products they held every product of a super-block in registers and spilled at four blocks).
__device__ __forceinline__ void scaleAdd(i32x4& is, int sc, i32x4 p) {
#pragma unroll
    for (int e = 0; e < 4; ++e) is[e] += __mul24(sc, p[e]);
    asm("" : "+v"(is));
}

// Half a super-block's activations for this lane: per column block the 8 values of four sub-blocks of 32 of
// column lane % 16.
template <int C>
struct HalfActs {
    i32x2 a[C][4];
};

// is += the scaled sums of sub-blocks 4 half .. 4 half + 3: 4 columns 4 kg .. 4 kg + 3 of each block, row r.
template <int C>
__device__ __forceinline__ void halfSums(const SbWeights<false>& w, const HalfActs<C>& x, int half, int,
                                         i32x4 (&is)[C]) {
    const uint32_t h1 = w.hdr[1], h3 = w.hdr[3];
    const uint32_t scw = half ? (h3 & 0x0F0F0F0Fu) | ((h1 >> 2) & 0x30303030u) : h1 & 0x3F3F3F3Fu;
    const i32x4 zero = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int sc = (int)((scw >> (8 * j)) & 255u);
        const uint32_t q0 = (uint32_t)w.q[2 * half + (j >> 1)][0], q1 = (uint32_t)w.q[2 * half + (j >> 1)][1];
        const i32x2 b = (j & 1) ? i32x2{(int)((q0 >> 4) & kLow4), (int)((q1 >> 4) & kLow4)}
                                : i32x2{(int)(q0 & kLow4), (int)(q1 & kLow4)};
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const i32x4 p = mfma8(x.a[c][j], b, zero);  // |p| <= 32 * 127 * 15
            scaleAdd(is[c], sc, p);
        }
        __builtin_amdgcn_sched_barrier(0);  // (keeps later sub-blocks' sums out of the registers)
    }
}
template <int C>
__device__ __forceinline__ void halfSums(const SbWeights<true>& w, const HalfActs<C>& x, int half, int kg,
                                         i32x4 (&is)[C]) {
    const uint32_t scw[2] = {(uint32_t)w.sc[2 * half], (uint32_t)w.sc[2 * half + 1]};
    const i32x4 zero = {0, 0, 0, 0};
    const uint32_t lo = kg < 2 ? ~0u : 0u;  // the op of values 0..15 of a sub-block takes lanes kg 0, 1
#pragma unroll
    for (int t = 0; t < 4; ++t) {  // values 128 half + 32 t ..
        uint32_t q[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t l = (uint32_t)w.ql[half][t & 1][i], h = (uint32_t)w.qh[half][i];
            const uint32_t hb = t == 0 ? h << 4 : t == 1 ? h << 2 : t == 2 ? h : h >> 2;
            // q - 32 per byte: (0x80 + q) - 32 never borrows, and its top bit flipped is the signed byte
            q[i] = ((((l >> (4 * (t >> 1))) & kLow4) | (hb & 0x30303030u) | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
        }
        const i32x2 b0 = {(int)(q[0] & lo), (int)(q[1] & lo)}, b1 = {(int)(q[0] & ~lo), (int)(q[1] & ~lo)};
        const int sw = (int)scw[t >> 1];
        int s0 = sbyte(sw, 2 * (t & 1)), s1 = sbyte(sw, 2 * (t & 1) + 1);
        asm("" : "+v"(s0), "+v"(s1));
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const i32x4 p0 = mfma8(x.a[c][t], b0, zero), p1 = mfma8(x.a[c][t], b1, zero);  // |p| <= 16 * 127 * 32
            scaleAdd(is[c], s0, p0);
            scaleAdd(is[c], s1, p1);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The super-block's terms from its sums (xd: the columns' scales; m: column lane % 16's packed sums of 32).
template <int C>
__device__ __forceinline__ void sbTerms(const SbWeights<false>& w, const i32x4 (&m)[C], int kg, const i32x4 (&is)[C],
                                        const float4 (&xd)[C], float4 (&t)[C]) {
    const uint32_t h0 = w.hdr[0], h1 = w.hdr[1], h2 = w.hdr[2], h3 = w.hdr[3];
    (void)h1;
    const float d = f16bits(h0 & 0xFFFFu), dmin = f16bits(h0 >> 16);
    const uint32_t mw[2] = {h2 & 0x3F3F3F3Fu, ((h3 >> 4) & 0x0F0F0F0Fu) | ((h2 >> 2) & 0x30303030u)};
    const i32x4 zero = {0, 0, 0, 0};
    // the min sums: 64 sum_j m_j (B_j >> 6) + sum_j m_j (B_j & 63), the eight j as lane group 0's values
    const i32x2 bm = kg == 0 ? i32x2{(int)mw[0], (int)mw[1]} : i32x2{0, 0};
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const i32x4 hi = mfma8(i32x2{m[c][0], m[c][1]}, bm, zero);
        const i32x4 im = mfma8(i32x2{m[c][2], m[c][3]}, bm, hi << 6);
        const float xs[4] = {xd[c].x, xd[c].y, xd[c].z, xd[c].w};
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (d * xs[e]) * (float)is[c][e] - (dmin * xs[e]) * (float)im[e];
        t[c] = make_float4(o[0], o[1], o[2], o[3]);
    }
}
template <int C>
__device__ __forceinline__ void sbTerms(const SbWeights<true>& w, const i32x4 (&)[C], int, const i32x4 (&is)[C],
                                        const float4 (&xd)[C], float4 (&t)[C]) {
    const float d = f16bits(w.d);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const float xs[4] = {xd[c].x, xd[c].y, xd[c].z, xd[c].w};
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (d * xs[e]) * (float)is[c][e];
        t[c] = make_float4(o[0], o[1], o[2], o[3]);
    }
}

// The activations of half super-blocks, from the slots to the matrix op's operands.
// Direct (ST = false): each lane loads its 8 bytes of every sub-block, 16 columns' cache lines per load.
// Staged (ST = true, slots 16-byte aligned): 16-byte pieces of whole 128-byte rows go straight to a
// wavefront-private LDS tile [block][16 columns][8 pieces] (about a third of the cache-line accesses, which
// is what the direct loads cost: 3072 x 8192 Q6_K, 48 columns 30.3 -> 21.7 us), a piece p of column c at chunk p ^ (c / 2 % 8)
// so that the 16 columns an operand read touches lie in different banks.
typedef __attribute__((address_space(3))) void* LdsPtr;
template <int C, bool ST>
struct HalfLoader {
    Rsrc x;
    char* tile;
    uint32_t v[ST ? 2 * C : C];  // byte offsets at super-block 0
    int rd;                      // staged: this lane's column and byte within a piece
    int swz;
    __device__ __forceinline__ void init(Rsrc rsrc, char* lds_tile, int lane, int col0, int ncols, uint32_t slot_bytes) {
        x = rsrc;
        tile = lds_tile;
        const int r = lane & 15, kg = lane >> 4;
        rd = r * 128 + (kg & 1) * 8;
        swz = (r >> 1) & 7;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            if (ST) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int cc = i * 8 + (lane >> 3), p = (lane & 7) ^ ((cc >> 1) & 7);
                    v[(ST ? 2 : 1) * c + (ST ? i : 0)] = (uint32_t)min(col0 + c * 16 + cc, ncols - 1) * slot_bytes + p * 16;
                }
            } else {
                v[c] = (uint32_t)min(col0 + c * 16 + r, ncols - 1) * slot_bytes + kg * 8;
            }
        }
    }
    // staged: the loads of half `half` of super-block s into the tile (its earlier contents have been read)
    __device__ __forceinline__ void stage(int s, int half) const {
        if (!ST) return;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2 * C; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(x, (LdsPtr)(tile + i * 1024), 16, v[ST ? i : 0], s * 256 + half * 128,
                                                     0, 0);
    }
    __device__ __forceinline__ void get(HalfActs<C>& h, int s, int half, int kg) const {
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (ST)
                    h.a[c][j] = *reinterpret_cast<const i32x2*>(tile + c * 2048 + rd + (((2 * j + (kg >> 1)) ^ swz) * 16));
                else
                    h.a[c][j] = buf2(x, v[ST ? 0 : c] + 32 * j, s * 256 + half * 128);
            }
    }
};

// LDS: xd [rsb][16 C] floats, the packed sums of 32 [rsb][16 C] x 16 B, the terms [rsb][C][16 rows][16 columns],
// the staged activations [wavefront][C] x 2 KiB.
template <bool Q6, int C, bool ST>
__device__ __forceinline__ void shortTile(char* lds, const uint8_t* __restrict__ qw, const int* __restrict__ xq,
                                          float* __restrict__ y, int rows, int nsb, int ncols, int tile, int col0,
                                          int rsb) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int W = blockDim.x >> 6;
    const int r = lane & 15, kg = lane >> 4;
    const int slot = nsb * 85, ngroups = (nsb + kGroupSb - 1) / kGroupSb;
    const uint32_t wbytes = (uint32_t)ngroups * (Q6 ? kQ6kSeg : kQ4kSeg);
    const Rsrc tw = bufRes(qw + (size_t)tile * wbytes, wbytes);
    const uint32_t v0 = r * 16, vq = v0 + (kg >> 1) * 1024 + (kg & 1) * 8;
    float* lxd = reinterpret_cast<float*>(lds);
    i32x4* lm = reinterpret_cast<i32x4*>(lds + (size_t)rsb * C * 64);
    float4* lt = reinterpret_cast<float4*>(lds + (size_t)rsb * C * (64 + 256));
    HalfLoader<C, ST> ld;
    ld.init(bufRes(xq, (uint32_t)ncols * (uint32_t)slot * 4u), lds + (size_t)rsb * C * (64 + 256 + 1024) + wave * (C * 2048),
            lane, col0, ncols, (uint32_t)slot * 4u);
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int r0 = 0; r0 < nsb; r0 += rsb) {
        const int r1 = min(r0 + rsb, nsb), nr = r1 - r0;
        SbWeights<Q6> w;
        HalfActs<C> x0, x1;
        int s = r0 + wave;
        if (s < r1) {
            ld.stage(s, 0);
            w.load(tw, s, v0, vq);
            if (!ST) ld.get(x0, s, 0, kg);
        }
        // (consecutive lanes: consecutive super-blocks of a column, contiguous in its slot)
        for (int i = threadIdx.x; i < nr * C * 16; i += blockDim.x) {
            const int cc = i / nr, sl = i - cc * nr;
            const int* cs = xq + (size_t)min(col0 + cc, ncols - 1) * slot;
            lxd[sl * C * 16 + cc] = reinterpret_cast<const float*>(cs + nsb * 64)[r0 + sl];
            if (!Q6) {
                const int* m = cs + nsb * 81 + (r0 + sl) * 4;
                lm[sl * C * 16 + cc] = i32x4{m[0], m[1], m[2], m[3]};
            }
        }
        __syncthreads();
        for (; s < r1; s += W) {
            SbWeights<Q6> wn;
            i32x4 is[C];
#pragma unroll
            for (int c = 0; c < C; ++c) is[c] = i32x4{0, 0, 0, 0};
            const int sn = s + W < r1 ? s + W : s;  // (past the round: this one again, unused)
            if (ST) {
                // (the staged tile: half 0 was the last load issued; half 1 is followed by wn's loads only)
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                ld.get(x0, s, 0, kg);
                ld.stage(s, 1);
                __builtin_amdgcn_sched_barrier(0);
                wn.load(tw, sn, v0, vq);
                __builtin_amdgcn_sched_barrier(0);
                halfSums<C>(w, x0, 0, kg, is);
                if (Q6) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
                ld.get(x1, s, 1, kg);
                ld.stage(sn, 0);
                halfSums<C>(w, x1, 1, kg, is);
            } else {
                ld.get(x1, s, 1, kg);
                halfSums<C>(w, x0, 0, kg, is);
                wn.load(tw, sn, v0, vq);
                ld.get(x0, sn, 0, kg);
                halfSums<C>(w, x1, 1, kg, is);
            }
            float4 xd[C], t[C];
            i32x4 m[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                xd[c] = *reinterpret_cast<const float4*>(lxd + (s - r0) * C * 16 + c * 16 + kg * 4);
                if (!Q6) m[c] = lm[(s - r0) * C * 16 + c * 16 + r];
            }
            sbTerms<C>(w, m, kg, is, xd, t);
#pragma unroll
            for (int c = 0; c < C; ++c) lt[((s - r0) * C + c) * 64 + r * 4 + kg] = t[c];
            w = wn;
        }
        if (ST) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the last, unused stage)
        __syncthreads();
        if (wave < C) {  // lane (row r' = lane / 4, columns 4 (lane % 4) ..) of column block `wave`
            for (int i = 0; i < nr; ++i) {
                const float4 v = lt[(i * C + wave) * 64 + lane];
                acc.x += v.x;
                acc.y += v.y;
                acc.z += v.z;
                acc.w += v.w;
            }
        }
        if (r1 < nsb) __syncthreads();
    }
    if (wave < C) {
        const int row = tile * kTileRows + (lane >> 2), c = col0 + wave * 16 + (lane & 3) * 4;
        const float o[4] = {acc.x, acc.y, acc.z, acc.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (row < rows && c + e < ncols) y[(size_t)(c + e) * rows + row] = o[e];
    }
}

template <int C, bool ST>
__global__ __launch_bounds__(512) void matmul_short_kernel(ShortGroup g, const int* __restrict__ xq, int nsb, int ncols,
                                                           int rsb) {
    extern __shared__ int4 lds4[];
    char* lds = reinterpret_cast<char*>(lds4);
    const int bx = blockIdx.x;
    const int pi = (g.nparts > 2 && bx >= g.p[2].tile0) ? 2 : (g.nparts > 1 && bx >= g.p[1].tile0) ? 1 : 0;
    const ShortPart p = g.p[pi];
    const int col0 = blockIdx.y * (16 * C);
    if (p.q6)
        shortTile<true, C, ST>(lds, p.qw, xq, p.y, p.rows, nsb, ncols, bx - p.tile0, col0, rsb);
    else
        shortTile<false, C, ST>(lds, p.qw, xq, p.y, p.rows, nsb, ncols, bx - p.tile0, col0, rsb);
}

}  // namespace

bool matmulShortRuns(int k, int ncols) {
    // a single column: the column kernel; 32-bit slot offsets
    return option("matmul_path") != 1 && ncols > 1 && (unsigned long long)ncols * (k / 256) * 340ull < (1ull << 32);
}

int launchMatmulShort(ShortGroup g, const int* xq, int k, int ncols, hipStream_t s) {
    if (g.nparts < 1 || g.nparts > 3 || ncols < 1 || k < 256 || k % 256) return fromHip(hipErrorInvalidValue, "matmul (short batch)");
    const int nsb = k / 256;
    int tiles = 0;
    for (int i = 0; i < g.nparts; ++i) {
        g.p[i].tile0 = tiles;
        tiles += tilesOf(g.p[i].rows);
    }
    const int blocks = (ncols + 15) / 16, C = blocks < 4 ? blocks : 4;
    const bool st = nsb % 4 == 0 && (reinterpret_cast<uintptr_t>(xq) & 15) == 0;  // 16-byte aligned slot rows
    // one block of a long row: 8 wavefronts keep more of the row in flight (3072 x 8192 Q6_K, 12 columns: 9.7 us
    // against 11.8 with 4); with 12 super-blocks, or more blocks and their LDS, 4 (8192 x 3072 Q4_K: 7.5 against 8.0 us
    // at 12 columns, 12.4 against 14.6 at 37)
    const int W = C == 1 && nsb >= 16 ? 8 : 4;
    // rounds of equal size whose terms fit
    const int per = C * (1024 + 256 + 64), most = (kLdsBytes - (st ? W * C * 2048 : 0)) / per;
    const int rounds = (nsb + most - 1) / most, rsb = (nsb + rounds - 1) / rounds;
    const dim3 grid(tiles, (blocks + C - 1) / C), block(64 * W);
    const size_t lds = (size_t)rsb * per + (st ? W * C * 2048 : 0);
#define KC_SHORT(CC, SS)                                                                                             \
    if (C == CC && st == SS) {                                                                                       \
        static const int attr = (int)hipFuncSetAttribute(reinterpret_cast<const void*>(matmul_short_kernel<CC, SS>), \
                                                         hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);     \
        if (attr != 0) return fromHip(attr, "matmul (short batch): LDS size");                                       \
        hipLaunchKernelGGL((matmul_short_kernel<CC, SS>), grid, block, lds, s, g, xq, nsb, ncols, rsb);              \
    }
    KC_SHORT(1, false) KC_SHORT(2, false) KC_SHORT(3, false) KC_SHORT(4, false)
    KC_SHORT(1, true) KC_SHORT(2, true) KC_SHORT(3, true) KC_SHORT(4, true)
#undef KC_SHORT
    return fromHip(hipGetLastError(), "matmul (short batch)");
}

}  // namespace kcamd
