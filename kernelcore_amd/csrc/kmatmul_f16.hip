// kmatmul_f16.hip -- Y = W X for fp16 weights and fp32 activations (gfx950): the matmul_f16 name
// (reference kernels/llm/matmul_f16.cu, mirror llm/llm_reference.cpp:756-764 in
// arasheedu/Kernelcore; the ggml backend sends F16 weights there with the activations as they are,
// integrations/llama.cpp/ggml/src/ggml-kernelcore/ggml-kernelcore.cpp:559-566).
//
// The weights stay in ggml's row-major F16 layout (W[r][k], two values per 32-bit word): a
// wavefront reads whole rows with 16-byte loads, so no load-time interleave is needed (the
// reference's 8-row word interleave, llm_reference.cpp:740-746, serves 8 CPU vector lanes).
// Three kernels, by batch width:
//   * ncols <= 8 (decode): one wavefront per 2 rows; each lane multiplies 8 consecutive values of
//     a row with the same 8 values of every column, the partial sums are reduced across the 64
//     lanes. HBM-bound (2 bytes per weight).
//   * ncols > 8: v_mfma_f32_16x16x32_f16, K split over the wavefronts of a workgroup (a tile
//     per wavefront where the rows are too short for that). The weights
//     are exact fp16 operands; each activation is split into hi = fp16(x) and lo = fp16(x - hi)
//     and every product runs as two MFMAs (f32 accumulation), within about 2^-22 of the fp32
//     product (a single fp16 rounding of x would be 2^-11).
//   * k not a multiple of 8 (the reference allows any even k): one thread per output, the
//     reference's own loop.
// Sums run in a different order than the reference's sequential loop (a tree over the lanes, the
// MFMA's accumulation): within the 1e-3 relative bar, not bit-identical.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "internal.hpp"
#include "kmatmul_mfma.hpp"
#include "launch.hpp"

namespace kcamd {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float h2f(uint32_t bits) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits); }

// Sum over the 64 lanes of a wavefront; every lane gets the total.
__device__ __forceinline__ float waveSum(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// ---- ncols <= 8: two rows per wavefront, NC columns (the launcher rounds ncols up to 1, 2, 4
// or 8; surplus columns reread the last one and are not stored). k % 8 == 0.
template <int NC>
__global__ __launch_bounds__(256) void mmf16_vec_kernel(const uint16_t* __restrict__ w, const float* __restrict__ x,
                                                        float* __restrict__ y, int rows, int k, int ncols) {
    constexpr int R = 2;
    const int lane = threadIdx.x & 63;
    const int r0 = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * R;
    if (r0 >= rows) return;  // rows % 8 == 0: a live wavefront has both rows
    const int nch = k / 8;   // 16-byte chunks per row
    float acc[R][NC];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[r][c] = 0.0f;
    for (int ch = lane; ch < nch; ch += 64) {
        u32x4 wv[R];
#pragma unroll
        for (int r = 0; r < R; ++r)
            wv[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(w + (size_t)(r0 + r) * k) + ch);
        float4 xv[NC][2];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const float4* xp = reinterpret_cast<const float4*>(x + (size_t)min(c, ncols - 1) * k) + 2 * ch;
            xv[c][0] = xp[0];
            xv[c][1] = xp[1];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float wf[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                wf[2 * e] = h2f(wv[r][e] & 0xFFFFu);
                wf[2 * e + 1] = h2f(wv[r][e] >> 16);
            }
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const float xs[8] = {xv[c][0].x, xv[c][0].y, xv[c][0].z, xv[c][0].w,
                                     xv[c][1].x, xv[c][1].y, xv[c][1].z, xv[c][1].w};
                float s = acc[r][c];
#pragma unroll
                for (int e = 0; e < 8; ++e) s += wf[e] * xs[e];
                acc[r][c] = s;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const float t = waveSum(acc[r][c]);
            if (lane == 0 && c < ncols) y[(size_t)c * rows + r0 + r] = t;
        }
}

// ---- ncols > 8, k % 16 == 0: a workgroup of 8 wavefronts covers 16 T rows x 16 C columns; K advances in
// chunks of 256 values, wavefront w taking values 32 w .. 32 w + 31 of each (one v_mfma_f32_16x16x32_f16 per 16 x 16
// block and activation part), and the 8 partial sums meet in LDS at the end. Lane (r = lane % 16, kg = lane / 16)
// holds A = W[row0 + 16 t + r][k + 8 kg .. +8] and B = x[col0 + 16 c + r][k + 8 kg .. +8]; the result's register e is
// row 4 kg + e of column r. Rows and columns past the end reread the last ones and are not stored.
//
// The chunks come by buffer-to-LDS loads of whole row pieces (512 B of a weight row, 1 KiB of a column), S stages
// deep: operand loads straight from memory touch 16 rows' cache lines per instruction, about 54 cycles each,
// and that bound the kernel (1024 x 4096, 77 columns: 16.5 us so, 10 us from LDS; 101 us for one wavefront per
// 32 x 32 block over all of K). A 16-byte piece p of row or column i lies at chunk
// p ^ (i % 16), so the 16 rows an operand read touches lie in different banks.
__device__ __forceinline__ void splitHiLo(const float4& x0, const float4& x1, h8& hi, h8& lo) {
    const float xs[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const _Float16 h = (_Float16)xs[e];
        hi[e] = h;
        lo[e] = (_Float16)(xs[e] - (float)h);
    }
}

typedef __attribute__((address_space(3))) void* LdsPtr;
constexpr int kF16Waves = 8;
template <int T, int C>
constexpr int f16StageBytes() { return T * 16 * 512 + C * 16 * 1024; }

template <int T, int C, int S>
__device__ __forceinline__ void f16Tile(float4* lds4, const uint16_t* __restrict__ w, const float* __restrict__ x,
                                        float* __restrict__ y, int rows, int k, int ncols) {
    constexpr int kStage = f16StageBytes<T, C>(), kLoads = T + 2 * C;  // loads per wavefront and stage
    char* lds = reinterpret_cast<char*>(lds4);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, kg = lane >> 4;
    const int row0 = blockIdx.x * 16 * T, col0 = blockIdx.y * 16 * C;
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(w + (size_t)row0 * k), (short)0, (int)((uint32_t)min(16 * T, rows - row0) * (uint32_t)k * 2u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(x + (size_t)col0 * k), (short)0, (int)((uint32_t)min(16 * C, ncols - col0) * (uint32_t)k * 4u), 0x00020000);
    // this lane's piece of each of its wavefront's loads: weight load 8 i + wave holds rows 2 (8 i + wave), + 1;
    // column load 8 i + wave that column
    uint32_t wo[T], xo[2 * C];  // byte offset of the row
    int wp[T], xp[2 * C];       // piece within the chunk
#pragma unroll
    for (int i = 0; i < T; ++i) {
        const int row = 2 * (8 * i + wave) + (lane >> 5);
        wo[i] = (uint32_t)min(row, rows - row0 - 1) * (uint32_t)k * 2u;
        wp[i] = (lane & 31) ^ (row & 15);
    }
#pragma unroll
    for (int i = 0; i < 2 * C; ++i) {
        const int col = 8 * i + wave;
        xo[i] = (uint32_t)min(col, ncols - col0 - 1) * (uint32_t)k * 4u;
        xp[i] = lane ^ (col & 15);
    }
    const int nch = (k + 255) / 256;
    auto stage = [&](int ch) {  // (chunks past the end: the last one again, unused; pieces past k: the row's first)
        char* buf = lds + (ch % S) * kStage;
        const int k0 = min(ch, nch - 1) * 256;
#pragma unroll
        for (int i = 0; i < T; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (LdsPtr)(buf + (8 * i + wave) * 1024), 16,
                                                     wo[i] + (k0 + 8 * wp[i] < k ? (uint32_t)(k0 * 2 + 16 * wp[i]) : 0u), 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2 * C; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (LdsPtr)(buf + T * 8192 + (8 * i + wave) * 1024), 16,
                                                     xo[i] + (k0 + 4 * xp[i] < k ? (uint32_t)(k0 * 4 + 16 * xp[i]) : 0u), 0, 0, 0);
    };
    f32x4 acc[T][C] = {}, sum[T][C] = {};
#pragma unroll
    for (int i = 0; i < S - 1; ++i) stage(i);
    const int pw = 4 * wave + kg;  // this lane's weight piece
    for (int ch = 0; ch < nch; ++ch) {
        // chunk ch has landed (S - 2 later ones may be in flight), everywhere; chunk ch - 1 has been read
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * kLoads) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        stage(ch + S - 1);
        const char* buf = lds + (ch % S) * kStage;
        h8 hi[C], lo[C], a[T];
#pragma unroll
        for (int t = 0; t < T; ++t) a[t] = *reinterpret_cast<const h8*>(buf + (16 * t + r) * 512 + ((pw ^ r) * 16));
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const char* b = buf + T * 8192 + (16 * c + r) * 1024;
            splitHiLo(*reinterpret_cast<const float4*>(b + ((2 * pw) ^ r) * 16),
                      *reinterpret_cast<const float4*>(b + ((2 * pw + 1) ^ r) * 16), hi[c], lo[c]);
        }
        if (ch == nch - 1 && k % 256) {  // the values past k
            const bool in = ch * 256 + 8 * pw < k;
            const h8 zero = {};
#pragma unroll
            for (int t = 0; t < T; ++t) a[t] = in ? a[t] : zero;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                hi[c] = in ? hi[c] : zero;
                lo[c] = in ? lo[c] : zero;
            }
        }
        // each chunk's products start from zero and are added to the sum while the next chunk's run: the rounding of one
        // long chain of accumulations was most of the error (2.2e-7 at k = 4096, 1.2e-7 so)
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int c = 0; c < C; ++c) {
                sum[t][c] += acc[t][c];
                acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], lo[c], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], hi[c], acc[t][c], 0, 0, 0);
            }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // (the stages past the end)
    __syncthreads();
    float4* part = lds4;  // [wavefront][t][c][lane]
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int c = 0; c < C; ++c) {
            sum[t][c] += acc[t][c];
            part[((wave * T + t) * C + c) * 64 + lane] = make_float4(sum[t][c][0], sum[t][c][1], sum[t][c][2], sum[t][c][3]);
        }
    __syncthreads();
    for (int i = threadIdx.x; i < T * C * 64; i += blockDim.x) {
        f32x4u o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int v = 0; v < kF16Waves; ++v) {
            const float4 q = part[v * T * C * 64 + i];
            o[0] += q.x;
            o[1] += q.y;
            o[2] += q.z;
            o[3] += q.w;
        }
        const int l = i & 63, tc = i >> 6, row = row0 + 16 * (tc / C) + 4 * (l >> 4), col = col0 + 16 * (tc % C) + (l & 15);
        if (row < rows && col < ncols) *reinterpret_cast<f32x4u*>(y + (size_t)col * rows + row) = o;  // rows % 8 == 0
    }
}

template <int T, int C, int S>
__global__ __launch_bounds__(64 * kF16Waves) void mmf16_mfma_kernel(const uint16_t* __restrict__ w,
                                                                    const float* __restrict__ x, float* __restrict__ y,
                                                                    int rows, int k, int ncols) {
    extern __shared__ float4 lds4[];
    f16Tile<T, C, S>(lds4, w, x, y, rows, k, ncols);
}

// ---- ncols > 8, k % 16 == 0, short rows: a workgroup of 4 wavefronts covers 64 rows x 64 columns, each wavefront 32 x 32 of
// them (2 x 2 blocks, the operands and results laid out as above, straight from memory) over the whole row, 32 values at a
// time from zero and added in pairs: 8.5e-8 of the result at k 272 (one chain of accumulations 1.6e-7, the kernel
// above 8.8e-8). Rows
// and columns past the end reread the last ones and are not stored. Bound by the outputs' bytes and the launch where it is used.
__global__ __launch_bounds__(256) void mmf16_tile_kernel(const uint16_t* __restrict__ w, const float* __restrict__ x,
                                                         float* __restrict__ y, int rows, int k, int ncols) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, kg = lane >> 4;
    const int row0 = blockIdx.x * 64 + (wave & 1) * 32, col0 = blockIdx.y * 64 + (wave >> 1) * 32;
    if (row0 >= rows || col0 >= ncols) return;
    const uint16_t* wr[2];
    const float* xr[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        wr[i] = w + (size_t)min(row0 + 16 * i + r, rows - 1) * k;
        xr[i] = x + (size_t)min(col0 + 16 * i + r, ncols - 1) * k;
    }
    f32x4 sum[2][2] = {};
    struct Step {
        h8 a[2];
        float4 xv[2][2];
        __device__ void load(const uint16_t* const (&wr)[2], const float* const (&xr)[2], int at) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[i] = *reinterpret_cast<const h8*>(wr[i] + at);
                const float4* xp = reinterpret_cast<const float4*>(xr[i] + at);
                xv[i][0] = xp[0];
                xv[i][1] = xp[1];
            }
        }
    };
    auto product = [&](const Step& st, bool in, f32x4 (&to)[2][2]) {  // to += (in: this lane's values are in the row)
        const h8 zero = {};
        h8 a[2], hi[2], lo[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            splitHiLo(st.xv[i][0], st.xv[i][1], hi[i], lo[i]);
            a[i] = in ? st.a[i] : zero;
            hi[i] = in ? hi[i] : zero;
            lo[i] = in ? lo[i] : zero;
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                f32x4 p = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], lo[c], f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                to[t][c] += __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], hi[c], p, 0, 0, 0);
            }
    };
    int k0 = 8 * kg;
    Step st[2];
    for (; k0 - 8 * kg + 64 <= k; k0 += 64) {  // two steps' loads together
        st[0].load(wr, xr, k0);
        st[1].load(wr, xr, k0 + 32);
        f32x4 two[2][2] = {};
        product(st[0], true, two);
        product(st[1], true, two);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int c = 0; c < 2; ++c) sum[t][c] += two[t][c];
    }
    for (; k0 - 8 * kg < k; k0 += 32) {  // (past the row: its first values, unused)
        const bool in = k0 < k;
        st[0].load(wr, xr, in ? k0 : 0);
        product(st[0], in, sum);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int row = row0 + 16 * t + 4 * kg, col = col0 + 16 * c + r;
            if (row < rows && col < ncols) *reinterpret_cast<f32x4u*>(y + (size_t)col * rows + row) = sum[t][c];  // rows % 8 == 0
        }
}

// ---- any even k: one thread per (row, column), the reference's loop (llm_reference.cpp:756-764).
__global__ __launch_bounds__(256) void mmf16_simple_kernel(const uint32_t* __restrict__ w, const float* __restrict__ x,
                                                           float* __restrict__ y, int rows, int k, int ncols) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long long)rows * ncols) return;
    const int c = (int)(idx / rows), r = (int)(idx % rows);
    const uint32_t* wr = w + (size_t)r * (k / 2);
    const float* xc = x + (size_t)c * k;
    float a = 0.0f;
    for (int i = 0; i < k / 2; ++i) {
        const uint32_t q = wr[i];
        a += h2f(q & 0xFFFFu) * xc[2 * i] + h2f(q >> 16) * xc[2 * i + 1];
    }
    y[(size_t)c * rows + r] = a;
}

}  // namespace

// Columns of one launch (the grid's second dimension).
constexpr int kMaxCols = 1 << 20;

int launchMatmulF16(const void* w, const float* x, float* y, int rows, int k, int ncols, hipStream_t s) {
    if (rows <= 0 || rows % 8 || k <= 0 || k % 2 || ncols <= 0)
        return fromHip(hipErrorInvalidValue, "matmul_f16: shape");
    const uint16_t* wh = static_cast<const uint16_t*>(w);
    // the vector kernels read 16 bytes at a time: w and x 16-byte aligned (hipMalloc gives 256)
    const bool a16 = ((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(x)) & 15) == 0;
    // a tile's 32-bit byte offsets (past them at most 63 rows and columns)
    const bool wide = (unsigned long long)k * 128 >= (1ull << 32);
    if (a16 && k % 8 == 0 && (ncols <= 8 || k % 16 || wide)) {
        // columns in launches of at most 8
        for (int c0 = 0; c0 < ncols; c0 += 8) {
            const int nc = ncols - c0 < 8 ? ncols - c0 : 8;
            const dim3 grid((rows / 2 + 3) / 4), block(256);
            const float* xc = x + (size_t)c0 * k;
            float* yc = y + (size_t)c0 * rows;
            if (nc == 1) hipLaunchKernelGGL(mmf16_vec_kernel<1>, grid, block, 0, s, wh, xc, yc, rows, k, nc);
            else if (nc == 2) hipLaunchKernelGGL(mmf16_vec_kernel<2>, grid, block, 0, s, wh, xc, yc, rows, k, nc);
            else if (nc <= 4) hipLaunchKernelGGL(mmf16_vec_kernel<4>, grid, block, 0, s, wh, xc, yc, rows, k, nc);
            else hipLaunchKernelGGL(mmf16_vec_kernel<8>, grid, block, 0, s, wh, xc, yc, rows, k, nc);
        }
    } else if (a16 && k % 16 == 0 && ncols > kMaxCols) {
        for (int c0 = 0; c0 < ncols; c0 += kMaxCols)
            if (int e = launchMatmulF16(w, x + (size_t)c0 * k, y + (size_t)c0 * rows, rows, k, std::min(kMaxCols, ncols - c0), s))
                return e;
    } else if (a16 && k % 16 == 0) {
        const auto wgs = [&](int t, int c) { return (long long)((rows + 16 * t - 1) / (16 * t)) * ((ncols + 16 * c - 1) / (16 * c)); };
        const long long cus = cuCount(), n42 = wgs(4, 2);
        // Rows much shorter than the chunk of 256 values leave most of the K split's wavefronts without work, and each
        // workgroup pays for all of them: once per round of workgroups over the GPU (us, K split / tile per wavefront: 4096 rows x
        // 2048 columns, k 64 58.9 / 27.9, 128 58.8 / 36.8; 512 columns, k 128 24.6 / 19.3, 272 28.0 / 21.2; 20480 rows, 12 columns,
        // k 288 19.4 / 17.4), little within one round (16384 rows, 9 columns, k 16: 14.6 / 13.1),
        // nothing where that is not half full (64 rows, 512 columns, k 16: 13.6 / 14.4).
        const bool tile = n42 < cus / 2 ? false
                          : n42 <= cus  ? k <= (ncols <= 16 ? 128 : 64)
                                        : k < 192 || (k < 352 && (k % 32 || (ncols <= 40 && n42 <= 2 * cus)));
        if (tile) {
            hipLaunchKernelGGL(mmf16_tile_kernel, dim3((rows + 63) / 64, (ncols + 63) / 64), dim3(256), 0, s, wh, x, y, rows,
                               k, ncols);
            return fromHip(hipGetLastError(), "matmul_f16");
        }
        // the smallest tile whose workgroups run at once on the CUs (a second round costs more than a larger
        // tile: 1024 x 4096, 77 columns 12.4 us on 16 x 16 (320 workgroups), 9.9 us on 32 x 16 (160), 11.3 us on
        // 64 x 16 (80)), else the largest (512 columns: 18.7 us on 64 x 32, 22.5 us on 64 x 16); three stages where they
        // fit
        const dim3 block(64 * kF16Waves);
#define KC_F16(TT, CC, SS)                                                                                             \
    {                                                                                                                  \
        constexpr int lds = SS * f16StageBytes<TT, CC>();                                                              \
        static_assert(lds >= kF16Waves * TT * CC * 1024, "the partial sums reuse the stages");                         \
        static const int attr = (int)hipFuncSetAttribute(reinterpret_cast<const void*>(mmf16_mfma_kernel<TT, CC, SS>), \
                                                         hipFuncAttributeMaxDynamicSharedMemorySize, lds);             \
        if (attr != 0) return fromHip(attr, "matmul_f16: LDS size");                                                   \
        hipLaunchKernelGGL((mmf16_mfma_kernel<TT, CC, SS>), dim3((rows + 16 * TT - 1) / (16 * TT),                     \
                           (ncols + 16 * CC - 1) / (16 * CC)), block, lds, s, wh, x, y, rows, k, ncols);               \
    }
        if (wgs(1, 1) <= cus) KC_F16(1, 1, 3)
        else if (wgs(2, 1) <= cus) KC_F16(2, 1, 3)
        else if (wgs(4, 1) <= cus) KC_F16(4, 1, 3)
        else KC_F16(4, 2, 2)
#undef KC_F16
    } else {
        const long long n = (long long)rows * ncols;
        hipLaunchKernelGGL(mmf16_simple_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                           static_cast<const uint32_t*>(w), x, y, rows, k, ncols);
    }
    return fromHip(hipGetLastError(), "matmul_f16");
}

}  // namespace kcamd
