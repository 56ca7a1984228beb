// kmatmul_i8.hip -- the prefill matmul of Q6_K weights on the int8 matrix cores (gfx950): Y = W X for 64 or more per-256
// activation columns, read from the slots as they lie (no fp16 form of the activations). The arithmetic is
// kmatmul_mfma.hip's (the exact integer sum of each super-block, the same f32 combine in the same order; reference
// kernels/llm/matmul_q6k_q8kx8.cu, mirror llm/llm_reference.cpp:564-596), so the outputs are bit-identical to it wherever
// its f32 sums are exact (below 2^24), and exact above.
//
// A weight times its sub-block scale, sc (q - 32), takes 14 bits: as two bytes (two 16-bit multiply-adds per four weights)
// it takes two v_mfma_i32_32x32x32_i8 per 32 values, where the fp16 kernel's split of the scale takes four fp16 ops, and
// the int8 activations halve the LDS reads. (Q4_K's product takes two ops either way, so Q4_K stays on the fp16 kernel:
// measured the same, 34-35 us for 8192 x 3072 x 512.)
//
// What bounds it: matrix and vector ops (unpacking ~11, the combine 4 vector ops per matrix op at 64 columns) overlap
// poorly at two wavefronts per SIMD (timing copies, 8192 x 6144 x 512, 82 us: 50 without unpacking, 37 with matrix ops
// and barriers alone). Hence a workgroup of four wavefronts x 32 rows and 64 or 128 columns, two per CU, each wavefront
// unpacking its rows' weights once into registers for all its column blocks, and a block's combine issued between the
// next block's matrix ops. Measured against the fp16 producer-wavefront kernel (us, kernel times of one trace, without that
// kernel's conversion launch of 5): 512 columns, k 3072: 8192 rows 54.0 -> 47.1, 2048 rows 26.1 -> 20.8, 16384 rows 105 -> 71.4;
// 3072 x 8192: 64 columns 51.0 -> 31.7, 200 56.4 -> 35.8, 700 110 -> 102, 2048 231 -> 161; 14336 x 4096, 65 columns 34.0 -> 30.0;
// 128 x 3072, 512 columns 22.6 -> 15.6; 24576 x 4096, 1024 columns 380 -> 257. Faster at all of 181 sizes, 0.73 of the time
// (geometric mean).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "internal.hpp"
#include "kmatmul_mfma.hpp"
#include "kquant.hpp"

namespace kcamd {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* LdsPtr;
typedef __amdgpu_buffer_rsrc_t Rsrc;

constexpr int kWaves = 4;  // wavefronts per workgroup, 32 weight rows each
constexpr int kRows = 32 * kWaves;
// LDS: two stages of a super-block's int8 activations [column][16 chunks of 16 B]; two groups of four super-blocks'
// column scales [column][4] (fetched per super-block they touched a cache line per column each time); zeros as the scales of
// the combine ahead of a range's first super-block (which adds 0: times a column's own scale that is NaN if it is infinite).
template <int NB>
struct Stage {
    static constexpr int kCols = 32 * NB;
    static constexpr int kBytes = kCols * 256;
    static constexpr int kXd = 2 * kBytes;
    static constexpr int kXdGroup = kCols * 16;
    static constexpr int kZero = kXd + 2 * kXdGroup;
    static constexpr int kLds = kZero + 32 * 16;
};

__device__ __forceinline__ Rsrc bufRes(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
// A pointer that every lane holds alike, as scalars (a resource in vector registers costs a loop per load).
template <class T>
__device__ __forceinline__ const T* uniform(const T* p) {
    const uint64_t u = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    return reinterpret_cast<const T*>(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ i32x4 buf4(Rsrc b, uint32_t v, uint32_t s) {
    return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(b, v, s, 0));
}
__device__ __forceinline__ float f16(uint32_t bits) {
    return (float)__builtin_bit_cast(_Float16, (unsigned short)bits);
}
// The same value, opaque: what is derived from it is computed where it is used instead of being kept in registers.
__device__ __forceinline__ int again(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// A super-block of 32 weight rows as loaded by lane (row lane % 32, half h = lane / 32: bytes 16 h .. of every 32).
struct Raw {
    i32x4 sc, ql[2][2], qh[2];
    uint32_t d;
    __device__ __forceinline__ void load(Rsrc w, int s, int lane, uint32_t tileB) {
        const uint32_t vt = (uint32_t)((lane >> 4) & 1) * tileB, v0 = vt + (lane & 15) * 16, vq = v0 + (lane >> 5) * 1024;
        const uint32_t seg = (uint32_t)((s >> 2) * kQ6kSeg), o = seg + (s & 3) * 256;
        sc = buf4(w, v0, o + 12 * 1024);
        d = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(w, vt + (lane & 15) * 2, seg + kQ6kSlabs * 1024 + (s & 3) * 32, 0) &
            0xFFFFu;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
#pragma unroll
            for (int a = 0; a < 2; ++a) ql[n][a] = buf4(w, vq, o + (4 * n + 2 * a) * 1024);
            qh[n] = buf4(w, vq, o + (8 + 2 * n) * 1024);
        }
    }
};
// ... and as matrix-op operands: for each 32-value sub-block the lane's 16 values k = 32 j + 16 h .. times their scale, as
// two bytes: product = 256 hi + lo.
struct Operands {
    i32x4 hi[8], lo[8];
};
// Words 2 half, 2 half + 1 of sub-block j's operands.
__device__ __forceinline__ void unpackHalf(const Raw& r, int h, int j, int half, Operands& o) {
    const int n = j >> 2, t = j & 3;
    // the int8 scale of values 32 j + 16 h ..: byte 2 j + h of the 16
    const int w = r.sc[j >> 1], sc = (w << (24 - 8 * (2 * (j & 1) + h))) >> 24;
    const u16x2 sv = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm((uint32_t)sc, (uint32_t)sc, 0x01000100u));
    const u16x2 c = sv * (unsigned short)(0x10000 - 32) + (unsigned short)128;  // 128 - 32 sc
#pragma unroll
    for (int e = 2 * half; e < 2 * half + 2; ++e) {
        const uint32_t l = (uint32_t)r.ql[n][t & 1][e], g = (uint32_t)r.qh[n][e];
        const uint32_t gb = (t == 0 ? g << 4 : t == 1 ? g << 2 : t == 2 ? g : g >> 2) & 0x30303030u;
        const uint32_t q = ((t >> 1 ? l >> 4 : l) & 0x0F0F0F0Fu) | gb;
        const u16x2 ev = __builtin_bit_cast(u16x2, q & 0x00FF00FFu);
        const u16x2 od = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm(0u, q, 0x0C030C01u));
        // sc (q - 32) + 128 in 16 bits: the high byte is the rounded quotient by 256, the low one the rest + 128
        const uint32_t te = __builtin_bit_cast(uint32_t, (u16x2)(ev * sv + c));
        const uint32_t to = __builtin_bit_cast(uint32_t, (u16x2)(od * sv + c));
        o.hi[j][e] = (int)__builtin_amdgcn_perm(to, te, 0x07030501u);
        o.lo[j][e] = (int)(__builtin_amdgcn_perm(to, te, 0x06020400u) ^ 0x80808080u);
    }
}

// The sums of one 32 x 32 block and super-block: 256 ih + il.
struct Sums {
    i32x16 ih, il;
};
// acc += (d xd) is for elements i and i + 1, in two parts (a matrix op stands between them).
struct Pair {
    float a, b;
};
__device__ __forceinline__ Pair combine1(const Sums& u, int i) {
    return Pair{(float)((u.ih[i] << 8) + u.il[i]), (float)((u.ih[i + 1] << 8) + u.il[i + 1])};
}
__device__ __forceinline__ void combine2(f32x16& acc, Pair p, float d, float2 xd, int i) {
    acc[i] = __builtin_fmaf(d * xd.x, p.a, acc[i]);
    acc[i + 1] = __builtin_fmaf(d * xd.y, p.b, acc[i + 1]);
}

// One workgroup: rows rowTile * 128 .., columns col0 .., super-blocks [sb0, sb1).
template <int NB>
__device__ __forceinline__ void i8Tile(char* lds, const uint8_t* __restrict__ qw, const int* __restrict__ xq,
                                       float* __restrict__ y, int rows, int nsb, int ncols, int rowTile, int col0, int sb0,
                                       int sb1) {
    using G = Stage<NB>;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, l32 = lane & 31;
    const uint32_t slotB = (uint32_t)nsb * 340u;
    const int ngroups = (nsb + kGroupSb - 1) / kGroupSb, tiles = (rows + kTileRows - 1) / kTileRows;
    const int tile0 = (rowTile * kRows + wave * 32) / kTileRows;
    const uint32_t tileB = (uint32_t)ngroups * (uint32_t)kQ6kSeg;
    // (a second tile past the stream and columns past ncols have vector offsets past the buffers' ends and read zeros, a
    // wavefront past the stream reads tile 0: never stored; the scalar offsets stay within one tile or column)
    const int first = tile0 < tiles ? tile0 : 0;
    const Rsrc rw = bufRes(uniform(qw + (size_t)(uint32_t)first * tileB), tiles - first < 2 ? tileB : 2 * tileB);
    const int lcols = ncols - col0 < G::kCols ? ncols - col0 : G::kCols;
    const Rsrc rx = bufRes(uniform(xq + (size_t)(uint32_t)col0 * (uint32_t)(nsb * 85)), (uint32_t)lcols * slotB);
    // super-block s's activations as the t-th of the range: load m of this wavefront holds columns 16 m + 4 wave +
    // lane / 16, piece p at chunk p ^ (column % 16) (the 16 columns an operand read touches: 16 banks' chunks)
    auto stage = [&](int t, int s) {
        const int l = again(tid) & 63, ac = 4 * wave + (l >> 4);
        const uint32_t va = (uint32_t)ac * slotB + (uint32_t)(((l & 15) ^ ac) * 16);
#pragma unroll
        for (int m = 0; m < 2 * NB; ++m)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (LdsPtr)(lds + (t & 1) * G::kBytes + (4 * m + wave) * 1024), 16,
                                                     va + (uint32_t)m * 16u * slotB, (uint32_t)s * 256u, 0, 0);
    };
    // the column scales of super-blocks 4 g ..: by wavefront c for columns 64 c ..
    auto scaleGroup = [&](int g) {
        const int l = again(tid) & 63;
        if (wave < NB / 2)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (LdsPtr)(lds + G::kXd + (g & 1) * G::kXdGroup + wave * 1024), 16,
                                                     (uint32_t)(wave * 64 + l) * slotB, (uint32_t)nsb * 256u + (uint32_t)g * 16u,
                                                     0, 0);
    };
    // the scales of super-block s for columns 4 h + ..
    auto xdOf = [&](int s) {
        return reinterpret_cast<const float*>(lds + G::kXd + ((s >> 2) & 1) * G::kXdGroup) + (4 * h) * 4 + (s & 3);
    };

    Raw raw;
    Operands op;
    Sums u[2];
    f32x16 acc[NB];
#pragma unroll
    for (int cb = 0; cb < NB; ++cb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[cb][i] = 0.0f;
    u[1].ih = i32x16{};
    u[1].il = i32x16{};
    const i32x16 zero = {};
    stage(0, sb0);
    scaleGroup(sb0 >> 2);
    if (tid < 128) reinterpret_cast<float*>(lds + G::kZero)[tid] = 0.0f;
    raw.load(rw, sb0, lane, tileB);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        unpackHalf(raw, h, j, 0, op);
        unpackHalf(raw, h, j, 1, op);
    }
    float d = f16(raw.d), dp = 0.0f;  // this super-block's d and the previous one's
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __syncthreads();
    const int nt = sb1 - sb0;
    const float* xdp = reinterpret_cast<const float*>(lds + G::kZero) + 16 * h - (NB - 1) * 128;  // the previous super-block's
    for (int t = 0; t < nt; ++t) {
        const int s = sb0 + t, sn = t + 1 < nt ? s + 1 : s;  // (past the range: the last one again, unused)
        const char* buf = lds + (t & 1) * G::kBytes;
        const float* xd = xdOf(s);
        stage(t + 1, sn);
        if ((s & 3) == 3) scaleGroup((s >> 2) + 1);
        raw.load(rw, sn, again(tid) & 63, tileB);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
            // block cb's products, the combine of the block before it (the previous super-block's last) and, in the last
            // block, the next super-block's operands as this one's are done with, in between
            Sums& c = u[cb & 1];
            const Sums& pv = u[(cb & 1) ^ 1];
            f32x16& pacc = acc[cb ? cb - 1 : NB - 1];
            const float* px = cb ? xd + (cb - 1) * 128 : xdp + (NB - 1) * 128;
            const float pd = cb ? d : dp;
            const bool last = cb == NB - 1;
            const int al = again(tid) & 31, ax = (h ^ (al & 15)) * 16;
            const char* ab = buf + al * 256 + cb * 8192;
            i32x4 a = *reinterpret_cast<const i32x4*>(ab + ax), an = a;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float* q = px + ((j >> 1) * 8 + (j & 1) * 2) * 4;
                const float2 xv = make_float2(q[0], q[4]);
                if (j + 1 < 8) an = *reinterpret_cast<const i32x4*>(ab + (ax ^ (32 * (j + 1))));
                c.ih = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, op.hi[j], j ? c.ih : zero, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                const Pair pr = combine1(pv, 2 * j);
                if (last && j) unpackHalf(raw, h, j - 1, 0, op);
                __builtin_amdgcn_sched_barrier(0);
                c.il = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, op.lo[j], j ? c.il : zero, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                combine2(pacc, pr, pd, xv, 2 * j);
                if (last && j) unpackHalf(raw, h, j - 1, 1, op);
                __builtin_amdgcn_sched_barrier(0);
                a = an;
            }
        }
        unpackHalf(raw, h, 7, 0, op);
        unpackHalf(raw, h, 7, 1, op);
        dp = d;
        xdp = xd;
        d = f16(raw.d);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();  // this stage read, the next one loaded
    }
    const float* px = xdOf(sb1 - 1) + (NB - 1) * 128;
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
        const float* q = px + ((i >> 2) * 8 + (i & 3)) * 4;
        combine2(acc[NB - 1], combine1(u[(NB - 1) & 1], i), dp, make_float2(q[0], q[4]), i);
    }
    const int row = rowTile * kRows + wave * 32 + l32;
    if (row < rows) {
#pragma unroll
        for (int cb = 0; cb < NB; ++cb)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int c = col0 + cb * 32 + (i >> 2) * 8 + h * 4 + (i & 3);
                if (c < ncols) y[(size_t)c * rows + row] = acc[cb][i];
            }
    }
}

template <int NB>
__global__ __launch_bounds__(64 * kWaves, 2) void matmul_i8_kernel(MfmaGroup g, const int* __restrict__ xq, int nsb,
                                                                   int ncols) {
    extern __shared__ int4 lds4[];
    // (HW_ID's wave slot: of the two wavefronts that share a SIMD one goes first, so that they drift apart: 3%)
    if (__builtin_amdgcn_s_getreg(0x1804) & 1) __builtin_amdgcn_s_setprio(2);
    const int bx = blockIdx.x;
    const int pi = (g.nparts > 2 && bx >= g.p[2].tile0) ? 2 : (g.nparts > 1 && bx >= g.p[1].tile0) ? 1 : 0;
    const MfmaPart& p = g.p[pi];
    const int z = blockIdx.z, sb0 = z * nsb / g.ks, sb1 = (z + 1) * nsb / g.ks;
    i8Tile<NB>(reinterpret_cast<char*>(lds4), p.qw, xq, p.y[z], p.rows, nsb, ncols, bx - p.tile0, blockIdx.y * (32 * NB), sb0,
               sb1);
}

template <int NB>
int launch(const MfmaGroup& g, int tiles, const int* xq, int nsb, int ncols, hipStream_t s) {
    using G = Stage<NB>;
    static const int attr = (int)hipFuncSetAttribute(reinterpret_cast<const void*>(matmul_i8_kernel<NB>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, G::kLds);
    if (attr != 0) return fromHip(attr, "matmul (int8 MFMA): LDS size");
    hipLaunchKernelGGL(matmul_i8_kernel<NB>, dim3(tiles, (ncols + G::kCols - 1) / G::kCols, g.ks), dim3(64 * kWaves), G::kLds,
                       s, g, xq, nsb, ncols);
    return fromHip(hipGetLastError(), "matmul_q6k_q8k (int8 MFMA)");
}

}  // namespace

bool matmulI8Fits(int nsb) { return nsb % 4 == 0 && nsb <= (1 << 16); }

int launchMatmulI8(MfmaGroup g, const int* xq, int nsb, int ncols, hipStream_t s) {
    int tiles = 0;
    for (int i = 0; i < g.nparts; ++i) {
        g.p[i].tile0 = tiles;
        tiles += (g.p[i].rows + kRows - 1) / kRows;
    }
    // 128 columns per workgroup unpack each weight half as often, but pay only where two such workgroups per CU
    // have work (kernel times of one trace, k 3072, 512 columns: 16384 rows 71.4 us against 110 with 64; 2048 rows 25.3 against
    // 20.8; 8192 rows 47 either way) and more than 64 columns (64 columns, half a tile of padding: 128256 x 3072 127 us
    // against 112)
    const long long wgs = (long long)tiles * ((ncols + 127) / 128) * g.ks;
    return ncols > 64 && wgs >= 2LL * cuCount() ? launch<4>(g, tiles, xq, nsb, ncols, s) : launch<2>(g, tiles, xq, nsb, ncols, s);
}

}  // namespace kcamd
