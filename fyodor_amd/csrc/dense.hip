// Batch 1..8 products of dense F32 / F16 / BF16 weights with fp32
// activations. Each wavefront owns R rows; its lanes stride over the columns
// (coalesced 4- or 2-byte loads) and the per-lane fp32 sums are reduced
// across the wavefront. These storage types have no block structure; the
// reference decodes them per element (backend/core/llm_quant.c:161-204).
#include "device.h"
#include "formats.h"
#include "kernels.h"
#include "fyodor_hip.h"
#include <float.h>
#include <limits.h>
#include <stdint.h>

namespace fy {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

// F32 / F16 / BF16: lanes stride over the columns of R rows.
template <unsigned T, int N, int R>
__global__ __launch_bounds__(kThreads) void skinny_dense(const uint8_t *__restrict__ w,
    const float *__restrict__ x, float *__restrict__ y, int rows, int cols)
{
    const int lane = threadIdx.x & 63;
    const int row0 = (blockIdx.x * kWaves + (threadIdx.x >> 6)) * R;
    const int nrow = rows - row0 < R ? rows - row0 : R;
    if (nrow <= 0) return;
    float acc[R][N];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int n = 0; n < N; ++n) acc[r][n] = 0.f;
    for (int k = lane; k < cols; k += 64) {
        float xv[N];
#pragma unroll
        for (int n = 0; n < N; ++n) xv[n] = x[(size_t)n * cols + k];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r >= nrow) continue;
            const size_t at = (size_t)(row0 + r) * cols + k;
            float wv;
            if constexpr (T == F32) wv = ((const float *)w)[at];
            else if constexpr (T == F16) wv = f16_to_f32(((const uint16_t *)w)[at]);
            else wv = bf16_to_f32(((const uint16_t *)w)[at]);
#pragma unroll
            for (int n = 0; n < N; ++n) acc[r][n] += wv * xv[n];
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const float v = wave_sum(acc[r][n]);
            if (lane == 0 && r < nrow) y[(size_t)n * rows + row0 + r] = v;
        }
}

template <int N> constexpr int rows_per_wave() { return N <= 2 ? 4 : 2; }

template <unsigned T, int N>
hipError_t launch_n(const uint8_t *w, const float *x, float *y, int rows, int cols, hipStream_t stream)
{
    constexpr int R = rows_per_wave<N>();
    const int rows_per_block = kWaves * R;
    const dim3 grid((unsigned)((rows + rows_per_block - 1) / rows_per_block));
    hipLaunchKernelGGL((skinny_dense<T, N, R>), grid, dim3(kThreads), 0, stream, w, x, y, rows, cols);
    return hipGetLastError();
}

template <unsigned T>
hipError_t launch_type(const uint8_t *w, const float *x, float *y, int rows, int cols, int batch, hipStream_t s)
{
    switch (batch) {
    case 1: return launch_n<T, 1>(w, x, y, rows, cols, s);
    case 2: return launch_n<T, 2>(w, x, y, rows, cols, s);
    case 3: return launch_n<T, 3>(w, x, y, rows, cols, s);
    case 4: return launch_n<T, 4>(w, x, y, rows, cols, s);
    case 5: return launch_n<T, 5>(w, x, y, rows, cols, s);
    case 6: return launch_n<T, 6>(w, x, y, rows, cols, s);
    case 7: return launch_n<T, 7>(w, x, y, rows, cols, s);
    case 8: return launch_n<T, 8>(w, x, y, rows, cols, s);
    default: return hipErrorInvalidValue;
    }
}

// ---- batches above 8: a GEMM on the bf16 matrix cores ----------------------
//
// Y [batch][rows] = X [batch][cols] W^T with fp32 products and accumulation,
// as the reference's CUDA GEMM (CUDA/gemm.cu:53-96), on
// v_mfma_f32_32x32x16_bf16: an fp32 value is exactly the sum of three bf16
// ones (each the rounded rest of the ones before), an F16 weight of two, a BF16
// weight is one. Products of bf16 pairs are exact in the MFMA, so
//   BF16  w x = w x1 + w x2 + w x3                               (3 MFMAs)
//   F16   w x = w1 x1 + (w1 x2 + w2 x1) + (w1 x3 + w2 x2) + e    (5)
//   F32   w x = the same + w3 x1 + e                             (6)
// with |e| below 2^-24 |w x|: the error of one fp32 product. The leading
// products have an accumulator of their own, so the others round at 2^-8 of
// its scale. 32 x 32 x 16 takes 96, 160 or 192 cycles where the fp32 matrix
// cores take 512 (153 TFLOP/s measured for a library fp32 product).
//
// The matrix cores read bf16 subnormals as zeros, so that a product loses up
// to about 2^-125 (|w| + |x|), and a non-finite value, or one that rounds to
// infinity, leaves NaN or infinity in its outputs. Outputs small enough for the
// first to show (against the largest operand that the workgroup met) or not
// finite are computed again as plain fp32 dots, or with their tile on the fp32
// matrix cores, unless what their operands hold says that they stand.
//
// Work split. A workgroup of eight wavefronts owns 64 tokens x 128 rows;
// wavefront (wr, ks) computes the 64 tokens of rows 32 wr .. 32 wr + 31 over
// the ks-th half of the columns (two wavefronts per SIMD, and sums half as
// long), 64 columns per step. The weights go from memory to their operand
// registers and are split there; the tokens' pieces are made once per
// workgroup half and read from LDS by its four wavefronts, double-buffered
// with one barrier per step; 16-byte chunk c of token t at place c ^ (t / 2 % 8).
// Tokens past the batch and rows past the matrix read zeros (buffer range
// checks).
//
// 4096 x 4096, us before (fp32 matrix cores) and now: see launch_gemm.
constexpr int kGemmTokens = 64, kGemmRows = 128, kGemmK = 64;
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

template <unsigned T> constexpr int kElem = T == F32 ? 4 : 2;
// A buffer offset past every range (at most 2^31 - 1 bytes), also 16 bytes on.
constexpr int kOutside = INT_MIN;
template <unsigned T> constexpr int kPieces = T == F32 ? 3 : T == F16 ? 2 : 1;   // of a weight
constexpr int kPlaneBytes = kGemmTokens * kGemmK * 2;   // one piece of a step's tokens

template <unsigned T>
__device__ __forceinline__ float widen(uint32_t bits)
{
    if constexpr (T == F16) return f16_to_f32(bits & 0xFFFFu);
    else return bf16_to_f32(bits & 0xFFFFu);
}

// N bf16 pieces of each of 2 P values, packed in pairs.
template <int N, int P>
__device__ __forceinline__ void split(const float (&v)[2 * P], uint32_t (&out)[N][P])
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < P; ++i) {
        float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
        for (int p = 0; p < N; ++p) {
            out[p][i] = __builtin_bit_cast(uint32_t, (bf16x2){(__bf16)a, (__bf16)b});
            if (p + 1 < N) {
                a = a - __builtin_bit_cast(float, out[p][i] << 16);
                b = b - __builtin_bit_cast(float, out[p][i] & 0xFFFF0000u);
            }
        }
    }
}

// This lane's weights of a step as loaded: slice s (of four) holds columns
// 16 s + 8 h .. + 7 of its row (the two lanes of a row read 32 or 64
// consecutive bytes per slice). ALIGN: bytes that every row's start is a
// multiple of, 16, 4 or 2 (one load each). Columns past the row's end hold
// whatever follows (the buffer range bounds it): their activations are zeros,
// and where a product of zero is no number the output is computed again. Whole
// steps past the wavefront's columns [.., kend) are read too with 16-byte loads
// (a select per slice costs more); the narrow loads skip them, as offsets outside
// the range.
template <unsigned T>
struct GemmWeights {
    u32x4 w[T == F32 ? 8 : 4];
};

// Slice s of the step at column kc.
template <unsigned T, int ALIGN>
__device__ __forceinline__ void load_slice(GemmWeights<T> &st, __amdgpu_buffer_rsrc_t wb, int cols, int row, int kc, int s,
    int kend)
{
    constexpr int kPer = T == F32 ? 2 : 1;   // 16-byte words per slice
    const int h = (int)((threadIdx.x >> 5) & 1);
    const int at = ALIGN == 16 || kc < kend
                       ? (int)(((uint32_t)row * (uint32_t)cols + (uint32_t)(kc + 16 * s + 8 * h)) * kElem<T>) : kOutside;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        if constexpr (ALIGN == 16) {
            st.w[kPer * s + q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wb, at + 16 * q, 0, 0));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int off = at + 16 * q + 4 * e;
                st.w[kPer * s + q][e] = ALIGN == 4 ? __builtin_amdgcn_raw_buffer_load_b32(wb, off, 0, 0)
                                                   : (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(wb, off, 0, 0) |
                                                       (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(wb, off + 2, 0, 0) << 16;
            }
        }
    }
}

// This thread's sixteen activations of a step: columns 4 (l % 16) .. + 3 of
// tokens 16 (wave % 4) + 4 q + l / 16, q = 0..3 (a load covers 256 consecutive
// bytes of four tokens).
struct Tokens {
    int first, col;   // the first token (of the workgroup's 64), the column within a step
};

__device__ __forceinline__ Tokens tokens_of()
{
    const int t = threadIdx.x & 255;
    return {16 * (t >> 6) + ((t & 63) >> 4), 4 * (t & 15)};
}

template <int ALIGN>
__device__ __forceinline__ void load_tokens(float (&x)[16], __amdgpu_buffer_rsrc_t xb, int cols, int t0, int kc, int kend)
{
    const Tokens t = tokens_of();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int at = ALIGN == 16 || kc < kend
                           ? (int)(((uint32_t)(t0 + t.first + 4 * q) * (uint32_t)cols + (uint32_t)(kc + t.col)) * 4u)
                           : kOutside;
        if constexpr (ALIGN == 16) {
            const float4 v = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(xb, at, 0, 0));
            x[4 * q] = v.x, x[4 * q + 1] = v.y, x[4 * q + 2] = v.z, x[4 * q + 3] = v.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                x[4 * q + e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xb, at + 4 * e, 0, 0));
        }
    }
}

// Zeros for the columns from kend on (a uniform test: whole steps skip it).
__device__ __forceinline__ void cut_tokens(float (&x)[16], int kc, int kend)
{
    if (kc + kGemmK <= kend) return;
    const int col = kc + tokens_of().col;
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = col + i % 4 < kend ? x[i] : 0.f;
}

__device__ __forceinline__ float larger(float m, float a, float b)
{
    return __builtin_fmaxf(m, __builtin_fmaxf(__builtin_fabsf(a), __builtin_fabsf(b)));
}

// The pieces of two of its tokens (half 0 or 1) into LDS: plane p at
// p kPlaneBytes, token t's 128 bytes at 128 t.
__device__ __forceinline__ void store_tokens(const float (&x)[16], int half, uint8_t *lds, float &big)
{
    const Tokens t = tokens_of();
#pragma unroll
    for (int q = 2 * half; q < 2 * half + 2; ++q) {
        const float v[4] = {x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
        big = larger(larger(big, v[0], v[1]), v[2], v[3]);
        uint32_t p[3][2];
        split<3, 2>(v, p);
        const int token = t.first + 4 * q, at = 128 * token + 16 * ((t.col >> 3) ^ ((token >> 1) & 7)) + 2 * (t.col & 4);
#pragma unroll
        for (int k = 0; k < 3; ++k) *(uint2 *)(lds + k * kPlaneBytes + at) = make_uint2(p[k][0], p[k][1]);
    }
}

// Slice s in pieces; big becomes the largest magnitude met (a BF16 pair's
// second value is taken with the first one's bits below it; F16 stays below
// the 2^16 that big starts from), seen the bits of all weights together.
template <unsigned T>
__device__ __forceinline__ void weight_pieces(const GemmWeights<T> &st, int s, bf16x8 (&out)[kPieces<T>], float &big,
    uint32_t &seen)
{
    constexpr int kWords = T == F32 ? 2 : 1;
#pragma unroll
    for (int q = 0; q < kWords; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) seen |= st.w[kWords * s + q][i];
    if constexpr (T == BF16) {
        out[0] = __builtin_bit_cast(bf16x8, st.w[s]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t word = st.w[s][i];
            big = larger(big, __builtin_bit_cast(float, word << 16), __builtin_bit_cast(float, word));
        }
    } else {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            // A copy first: a bit cast of the vector's element reads element 0.
            const uint32_t word = T == F32 ? st.w[(2 * s + i / 4) % (T == F32 ? 8 : 4)][i % 4] : st.w[s][i / 2];
            if constexpr (T == F32) v[i] = __builtin_bit_cast(float, word);
            else v[i] = widen<T>(word >> (16 * (i & 1)));
        }
        if constexpr (T == F32) {
#pragma unroll
            for (int i = 0; i < 8; i += 2) big = larger(big, v[i], v[i + 1]);
        }
        uint32_t p[kPieces<T>][4];
        split<kPieces<T>, 4>(v, p);
#pragma unroll
        for (int k = 0; k < kPieces<T>; ++k)
            out[k] = __builtin_bit_cast(bf16x8, (u32x4){p[k][0], p[k][1], p[k][2], p[k][3]});
    }
}

template <unsigned T>
__device__ __forceinline__ float weight_at(const uint8_t *w, size_t at)
{
    if constexpr (T == F32) return ((const float *)w)[at];
    else return widen<T>(((const uint16_t *)w)[at]);
}

// One output as a plain fp32 dot over columns [k0, k1), by the wavefront.
template <unsigned T>
__device__ float plain_dot(const uint8_t *w, const float *x, int cols, int row, int token, int k0, int k1)
{
    const float *xr = x + (size_t)token * cols;
    float s = 0.f;
#pragma unroll 8
    for (int k = k0 + (int)(threadIdx.x & 63); k < k1; k += 64) s += weight_at<T>(w, (size_t)row * cols + k) * xr[k];
    return wave_sum(s);
}

// ---- the fp32 matrix cores -------------------------------------------------
//
// A tile of 64 tokens x 128 rows on v_mfma_f32_32x32x2_f32, by four wavefronts:
// wavefront wr computes the 64 tokens of rows 32 wr .. 32 wr + 31 as two 32 x 32
// tiles, each in two accumulator chains (even and odd chunks) added at the end.
// K advances 32 columns per chunk: the tokens' 64 x 32 and the rows' 128 x 32
// values go through LDS as fp32 (rows padded to 36 floats: conflict-free 16-byte
// reads), the next chunk's through registers while the matrix cores work. MFMA
// step s takes column 16 h + s in lane half h, for both operands alike.
constexpr int kChunk = 32, kPitch = 36;
constexpr int kChunkFloats = (kGemmRows + kGemmTokens) * kPitch;   // of LDS

// Thread t (of 256): W row t / 2, columns 16 (t % 2) .. + 15; X token t / 4,
// columns 8 (t % 4) .. + 7.
struct Chunk {
    float w[16], x[8];
};

// The chunk at column kc of [.., kend): zeros past it. Rows and tokens past the
// last read zeros or stay unused (buffer ranges).
template <unsigned T>
__device__ __forceinline__ void load_chunk(Chunk &c, __amdgpu_buffer_rsrc_t wb, __amdgpu_buffer_rsrc_t xb, int cols,
    int r0, int t0, int kc, int kend, int t)
{
    const int row = r0 + (t >> 1), wcol = kc + 16 * (t & 1);
    const int tok = t0 + (t >> 2), xcol = kc + 8 * (t & 3);
    if ((size_t)cols * kElem<T> % 16 == 0 && kc + kChunk <= kend) {
        const int wo = (int)(((uint32_t)row * (uint32_t)cols + (uint32_t)wcol) * kElem<T>);
#pragma unroll
        for (int q = 0; q < (T == F32 ? 4 : 2); ++q) {
            const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wb, wo + 16 * q, 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t u = v[e];
                if constexpr (T == F32) c.w[4 * q + e] = __builtin_bit_cast(float, u);
                else c.w[8 * q + 2 * e] = widen<T>(u), c.w[8 * q + 2 * e + 1] = widen<T>(u >> 16);
            }
        }
        const int xo = (int)(((uint32_t)tok * (uint32_t)cols + (uint32_t)xcol) * 4u);
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float4 v = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(xb, xo + 16 * q, 0, 0));
            c.x[4 * q] = v.x, c.x[4 * q + 1] = v.y, c.x[4 * q + 2] = v.z, c.x[4 * q + 3] = v.w;
        }
        return;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int k = wcol + e;
        const int off = k < kend ? (int)(((uint32_t)row * (uint32_t)cols + (uint32_t)k) * kElem<T>) : kOutside;
        if constexpr (T == F32) c.w[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wb, off, 0, 0));
        else c.w[e] = widen<T>(__builtin_amdgcn_raw_buffer_load_b16(wb, off, 0, 0));
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int k = xcol + e;
        const int off = k < kend ? (int)(((uint32_t)tok * (uint32_t)cols + (uint32_t)k) * 4u) : kOutside;
        c.x[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xb, off, 0, 0));
    }
}

__device__ __forceinline__ void store_chunk(const Chunk &c, float *sw, int t)
{
    float *w = sw + (t >> 1) * kPitch + 16 * (t & 1), *x = sw + (kGemmRows + (t >> 2)) * kPitch + 8 * (t & 3);
#pragma unroll
    for (int q = 0; q < 4; ++q)
        *(float4 *)(w + 4 * q) = make_float4(c.w[4 * q], c.w[4 * q + 1], c.w[4 * q + 2], c.w[4 * q + 3]);
#pragma unroll
    for (int q = 0; q < 2; ++q)
        *(float4 *)(x + 4 * q) = make_float4(c.x[4 * q], c.x[4 * q + 1], c.x[4 * q + 2], c.x[4 * q + 3]);
}

// The tile's sums over `chunks` chunks of columns [k0, kend), in sw (kChunkFloats
// of LDS of these four wavefronts). Every wavefront of the workgroup calls it with
// the same number of chunks: it meets them at barriers.
template <unsigned T>
__device__ __forceinline__ void fp32_tile(f32x16 (&acc)[2][2], __amdgpu_buffer_rsrc_t wb, __amdgpu_buffer_rsrc_t xb,
    int cols, int r0, int t0, int k0, int kend, int chunks, int wr, float *sw)
{
    // Opaque: a caller's registers hold none of this before it gets here.
    int t = threadIdx.x & 255;
    asm("" : "+v"(t));
    const int lane = t & 63, h = lane >> 5;
    Chunk c;
    load_chunk<T>(c, wb, xb, cols, r0, t0, k0, kend, t);
    auto step = [&](int i, int chain) {
        __syncthreads();   // the operand reads of the chunk before are done
        store_chunk(c, sw, t);
        __syncthreads();
        if (i + 1 < chunks) load_chunk<T>(c, wb, xb, cols, r0, t0, k0 + kChunk * (i + 1), kend, t);
        const float *pw = sw + (32 * wr + (lane & 31)) * kPitch + 16 * h;
        const float *px = sw + (kGemmRows + (lane & 31)) * kPitch + 16 * h;
        float b[16], a0[16], a1[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 w = *(const float4 *)(pw + 4 * q), v0 = *(const float4 *)(px + 4 * q),
                         v1 = *(const float4 *)(px + 32 * kPitch + 4 * q);
            b[4 * q] = w.x, b[4 * q + 1] = w.y, b[4 * q + 2] = w.z, b[4 * q + 3] = w.w;
            a0[4 * q] = v0.x, a0[4 * q + 1] = v0.y, a0[4 * q + 2] = v0.z, a0[4 * q + 3] = v0.w;
            a1[4 * q] = v1.x, a1[4 * q + 1] = v1.y, a1[4 * q + 2] = v1.z, a1[4 * q + 3] = v1.w;
        }
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            acc[0][chain] = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[s], b[s], acc[0][chain], 0, 0, 0);
            acc[1][chain] = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[s], b[s], acc[1][chain], 0, 0, 0);
        }
    };
    int i = 0;
    for (; i + 1 < chunks; i += 2) step(i, 0), step(i + 1, 1);
    if (i < chunks) step(i, 0);
}

// Short rows: four wavefronts and 27 KiB of LDS per tile, several workgroups on a
// CU, where the kernel above spends most of its one workgroup's time on filling
// its pipeline and on meeting. launch_dense_gemm says where the line lies.
template <unsigned T>
__global__ __launch_bounds__(256) void dense_gemm(const uint8_t *__restrict__ w, const float *__restrict__ x,
    float *__restrict__ y, int rows, int cols, int batch)
{
    __shared__ __align__(16) float sw[kChunkFloats];
    const int lane = threadIdx.x & 63, h = lane >> 5, wr = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = blockIdx.x * kGemmRows, t0 = blockIdx.y * kGemmTokens;
    const __amdgpu_buffer_rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(w), (short)0, (int)((size_t)rows * cols * kElem<T>), 0x00020000);
    const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(x), (short)0, (int)((size_t)batch * cols * 4), 0x00020000);
    f32x16 acc[2][2] = {};
    fp32_tile<T>(acc, wb, xb, cols, r0, t0, 0, cols, (cols + kChunk - 1) / kChunk, wr, sw);
    // D[token][row]: register i of lane l holds token 8 (i / 4) + 4 h + i % 4 of
    // its 32, row l % 32.
    const int row = r0 + 32 * wr + (lane & 31);
    if (row >= rows) return;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        const int token = t0 + 32 * (i >> 4) + 8 * ((i >> 2) & 3) + 4 * h + (i & 3);
        if (token < batch) y[(size_t)token * rows + row] = acc[i >> 4][0][i & 15] + acc[i >> 4][1][i & 15];
    }
}

// ---- outputs that the pieces may have missed ---------------------------------
//
// Flagged outputs of a wavefront that are computed again one by one (about 3 us
// each over 4096 columns) before their operands are looked at (25 us for 64
// tokens), and that are afterwards, before the whole tile runs again (210 us).
// us, 4096 x 4096 F16 by 333 tokens, 80 without: every token NaN 107, one token with
// an infinity 210, three 308, all 314 (the fp32 cores alone: 220 whatever the
// input; every flagged output as a dot: 4100 to 4600), one of 1e30 114, half the
// products zero by disjoint columns 94 (1250), a diagonal matrix 101 (2130).
constexpr int kFew = 8, kMany = 64;

struct Review {
    int votes[3][4];          // [round][row group]: outputs left
    uint32_t rows[3][4];      // their rows
    uint32_t tokens[4][2];    // [row group][lane half]: of the first round, bit i as output i of a lane
    uint2 token[64], row[128];
};

// The bits of the largest magnitude among columns [k0, k1) of the row at `at`, and
// of the least that is not zero, minus 1 (all ones: every one is zero). By the
// wavefront.
template <unsigned T>
__device__ uint2 range_of(const uint8_t *v, size_t at, int k0, int k1)
{
    uint32_t most = 0, least = ~0u;
#pragma unroll 16
    for (int k = k0 + (int)(threadIdx.x & 63); k < k1; k += 64) {
        const uint32_t b = __builtin_bit_cast(uint32_t, weight_at<T>(v, at + k)) & 0x7FFFFFFFu;
        most = most > b ? most : b;
        least = least < b - 1 ? least : b - 1;
    }
    for (int o = 32; o; o >>= 1) {
        const uint32_t m = (uint32_t)__shfl_xor((int)most, o, 64), l = (uint32_t)__shfl_xor((int)least, o, 64);
        most = most > m ? most : m;
        least = least < l ? least : l;
    }
    return make_uint2(most, least);
}

// Whether output v of a token and a row of these ranges is what plain sums give:
// not a number because an operand is none; or finite (so no operand was infinite
// or rounded to infinity), and zero for want of operands, or of operands whose
// pieces and products are all above the subnormals, or large against what
// subnormals of this token and row can have lost.
__device__ __forceinline__ bool stands(uint2 t, uint2 w, float v, float cols)
{
    if (t.x > 0x7F800000u || w.x > 0x7F800000u) return true;
    if (!(__builtin_fabsf(v) <= FLT_MAX)) return false;
    if (t.y == ~0u || w.y == ~0u) return true;
    const float tm = __builtin_bit_cast(float, t.y + 1), wm = __builtin_bit_cast(float, w.y + 1);
    if (tm >= 0x1p-100f && wm >= 0x1p-100f && tm * wm >= 0x1p-98f) return true;
    return __builtin_fabsf(v) >=
           cols * 0x1p-99f * __builtin_fmaxf(__builtin_bit_cast(float, t.x), __builtin_bit_cast(float, w.x));
}

// Shares out what is left of the four row groups in this round; the most that one
// of them has, the same in every wavefront.
__device__ __forceinline__ int review_votes(Review &rv, uint32_t again, int wr, int ks, int round)
{
    if (ks == 0) {
        const uint64_t lanes = __ballot(again != 0);
        int n = __popc(again);
        uint32_t m = again;
        for (int o = 1; o < 64; o *= 2) {
            n += __shfl_xor(n, o, 64);
            if (o < 32) m |= (uint32_t)__shfl_xor((int)m, o, 64);
        }
        if ((threadIdx.x & 31) == 0) {
            if (round == 0) rv.tokens[wr][(threadIdx.x >> 5) & 1] = m;
            rv.votes[round][wr] = n;
            rv.rows[round][wr] = (uint32_t)lanes | (uint32_t)(lanes >> 32);
        }
    }
    __syncthreads();
    int most = 0;
    for (int i = 0; i < 4; ++i) most = most > rv.votes[round][i] ? most : rv.votes[round][i];
    return __builtin_amdgcn_readfirstlane(most);
}

// Workgroup (row tile, token tile, split z) covers the 64-column steps
// [z per, (z + 1) per) of the split count gridDim.z; with one split it
// writes Y, else its partial sums to part[z][token][row] for dense_combine.
template <unsigned T, int ALIGN>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void dense_gemm(
    const uint8_t *__restrict__ w, const float *__restrict__ x, float *__restrict__ y, int rows, int cols, int batch,
    int per, float *__restrict__ part)
{
    constexpr int kBuf = 3 * kPlaneBytes;
    __shared__ __align__(16) uint8_t sx[2][2][kBuf];   // [half of the columns][buffer]
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wave & 3, ks = wave >> 2;
    const int r0 = blockIdx.x * kGemmRows, t0 = blockIdx.y * kGemmTokens;
    const __amdgpu_buffer_rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(w), (short)0, (int)((size_t)rows * cols * kElem<T>), 0x00020000);
    const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(x), (short)0, (int)((size_t)batch * cols * 4), 0x00020000);
    const int k0 = blockIdx.z * per * kGemmK, k1 = k0 + per * kGemmK < cols ? k0 + per * kGemmK : cols;
    // Both halves walk as many steps (the barriers are the workgroup's); past
    // its columns the second one's loads are zeros.
    const int steps = k0 < k1 ? ((k1 - k0 + kGemmK - 1) / kGemmK + 1) / 2 : 0;
    const int first = k0 + ks * steps * kGemmK, mid = k0 + steps * kGemmK, kend = ks || k1 < mid ? k1 : mid;
    const int row = r0 + 32 * wr + (lane & 31);
    // Leading products and the rest, per token tile.
    f32x16 acc[2][2] = {};
    // Step i takes each slice's weights out of their registers and requests
    // step i + 2's into them; meanwhile the tokens of step i + 1, requested in
    // step i - 1, are split into the other buffer, and those of step i + 2
    // requested.
    float big = T == F16 ? 0x1p16f : 0.f;   // the largest |w| and |x| met
    uint32_t seen = 0;                      // the bits of this lane's weights
    GemmWeights<T> w0, w1;
    float x0[16], x1[16];
    auto at = [&](int i) { return first + i * kGemmK; };
    auto step = [&](int i, int odd, GemmWeights<T> &cur, float (&xs)[16], float (&xn)[16]) {
        // (Past the last step nobody computes on what is requested.)
        load_tokens<ALIGN>(xn, xb, cols, t0, at(i + 2), kend);
        __builtin_amdgcn_sched_barrier(0);
        cut_tokens(xs, at(i + 1), kend);
        const uint8_t *buf = sx[ks][odd];
        bf16x8 a[2][2][3], b[2][kPieces<T>];
        auto fetch = [&](int s, bf16x8 (&x8)[2][3], bf16x8 (&w8)[kPieces<T>]) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    x8[t][p] = *(const bf16x8 *)(buf + p * kPlaneBytes + 128 * (32 * t + (lane & 31)) +
                                                 16 * ((2 * s + h) ^ ((lane >> 1) & 7)));
            weight_pieces<T>(cur, s, w8, big, seen);
        };
        // A slice's operands are made among the MFMAs of the one before, but
        // for F32, whose second set would not fit the registers.
        constexpr bool kAhead = T != F32;
        if (kAhead) fetch(0, a[0], b[0]);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (!kAhead) fetch(s, a[s & 1], b[s & 1]);
            else if (s < 3) fetch(s + 1, a[(s + 1) & 1], b[(s + 1) & 1]);
            if (s < 2) store_tokens(xs, s, sx[ks][1 - odd], big);
            // The two token tiles in turn.
            auto mul = [&](int which, int pa, int pb) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    acc[t][which] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s & 1][t][pa], b[s & 1][pb], acc[t][which],
                                                                            0, 0, 0);
            };
            mul(1, 2, 0);
            mul(0, 0, 0);
            mul(1, 1, 0);
            if constexpr (kPieces<T> > 1) {
                mul(1, 1, 1);
                mul(1, 0, 1);
            }
            if constexpr (kPieces<T> > 2) mul(1, 0, 2);
            load_slice<T, ALIGN>(cur, wb, cols, row, at(i + 2), s, kend);
            constexpr int kMfma = 2 * (kPieces<T> == 1 ? 3 : kPieces<T> == 2 ? 5 : 6);
#pragma unroll
            for (int q = 0; q < kMfma; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);   // VALU
                if (q < 6) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
            }
            __builtin_amdgcn_sched_group_barrier(0x020, T == F32 ? 2 : 1, 0);   // the slice's load
        }
        __syncthreads();
    };
    if (steps) {
        load_tokens<ALIGN>(x0, xb, cols, t0, at(0), kend);
#pragma unroll
        for (int s = 0; s < 4; ++s) load_slice<T, ALIGN>(w0, wb, cols, row, at(0), s, kend);
#pragma unroll
        for (int s = 0; s < 4; ++s) load_slice<T, ALIGN>(w1, wb, cols, row, at(1), s, kend);
        cut_tokens(x0, at(0), kend);
        store_tokens(x0, 0, sx[ks][0], big);
        store_tokens(x0, 1, sx[ks][0], big);
        load_tokens<ALIGN>(x0, xb, cols, t0, at(1), kend);
    }
    __syncthreads();
    // Two steps per pass: the registers of one take the loads of the next
    // without copies (a copy would wait for them).
    for (int i = 0; i + 1 < steps; i += 2) {
        step(i, 0, w0, x0, x1);
        step(i + 1, 1, w1, x1, x0);
    }
    if (steps & 1) step(steps - 1, 0, w0, x0, x1);
    // (Formed anew: nothing of it lives in registers through the loop.)
    int end_lane = threadIdx.x & 63;
    asm("" : "+v"(end_lane));
    const int end_h = end_lane >> 5, end_row = r0 + 32 * wr + (end_lane & 31);
    // The halves meet in LDS. D[token][row]: register i of lane l holds token
    // 8 (i / 4) + 4 h + i % 4 of its token tile, row l % 32.
    float *meet = (float *)&sx[0][0][0] + 2048 * wr + end_lane, *most = (float *)&sx[0][0][0] + 8192;
    uint32_t *bits = (uint32_t *)most + 8 + 64 * wr + end_lane;
    for (int o = 32; o; o >>= 1) big = __builtin_fmaxf(big, __shfl_xor(big, o, 64));
    if (end_lane == 0) most[wave] = big;
    if (ks == 1) {
        *bits = seen;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) meet[64 * (16 * t + i)] = acc[t][0][i] + acc[t][1][i];
    }
    __syncthreads();
    // Outputs to look at again, by output i of the lane (its row, 32 tokens).
    uint32_t again = 0;
    float *out = gridDim.z == 1 ? y : part + (size_t)blockIdx.z * batch * rows;
    auto token = [&](int i) { return t0 + 32 * (i >> 4) + 8 * ((i >> 2) & 3) + 4 * end_h + (i & 3); };
    if (ks == 0) {
        for (int i = 0; i < 8; ++i) big = __builtin_fmaxf(big, most[i]);
        // cols 2^-125 2 big is lost at most; it may weigh 2^-25.
        const float least = (float)cols * 0x1p-99f * big;
        uint32_t zero = 0;
#pragma unroll
        for (int i = 0; i < 32; ++i) {
            const float v = (acc[i >> 4][0][i & 15] + acc[i >> 4][1][i & 15]) + meet[64 * i];
            if (end_row < rows && token(i) < batch) {
                const float m = __builtin_fabsf(v);
                if (!(m >= least && m <= FLT_MAX)) again |= 1u << i;
                if (m == 0.f) zero |= 1u << i;
                out[(size_t)token(i) * rows + end_row] = v;
            }
        }
        // The zeros of a row of zeros stand.
        seen |= *bits;
        seen |= (uint32_t)__shfl_xor((int)seen, 32, 64);
        if ((seen & (T == F32 ? 0x7FFFFFFFu : 0x7FFF7FFFu)) == 0) again &= ~zero;
    }
    // Few of them: plain dots. More: what their tokens hold settles most, then
    // what their rows hold; of what is left, few are dots again, else the tile is
    // computed again on the fp32 matrix cores.
    Review &rv = *(Review *)((float *)&sx[0][0][0] + 8192 + 8 + 256);
    int left = review_votes(rv, again, wr, ks, 0);
    if (left == 0) return;
    for (int stage = 0; stage < 2 && left > kFew; ++stage) {
        int n = 0;   // the stage's tokens or rows, dealt to the eight wavefronts
        if (stage == 0) {
            for (int f = 0; f < 2; ++f) {
                uint32_t m = rv.tokens[0][f] | rv.tokens[1][f] | rv.tokens[2][f] | rv.tokens[3][f];
                for (m = __builtin_amdgcn_readfirstlane(m); m; m &= m - 1) {
                    const int i = __ffs(m) - 1, at = t0 + 32 * (i >> 4) + 8 * ((i >> 2) & 3) + 4 * f + (i & 3);
                    if ((n++ & 7) != wave) continue;
                    const uint2 r = range_of<F32>((const uint8_t *)x, (size_t)at * cols, k0, k1);
                    if (end_lane == 0) rv.token[32 * f + i] = r;
                }
            }
        } else {
            for (int f = 0; f < 4; ++f)
                for (uint32_t m = __builtin_amdgcn_readfirstlane(rv.rows[1][f]); m; m &= m - 1) {
                    const int i = __ffs(m) - 1;
                    if ((n++ & 7) != wave) continue;
                    const uint2 r = range_of<T>(w, (size_t)(r0 + 32 * f + i) * cols, k0, k1);
                    if (end_lane == 0) rv.row[32 * f + i] = r;
                }
        }
        __syncthreads();
        // Before the rows are looked at: anything, but that F16 is in its range.
        const uint2 any = T == F16 ? make_uint2(0x477FE000u, 0x33800000u - 1) : make_uint2(0x7F7FFFFFu, 0u);
        uint32_t keep = again;
        for (uint32_t m = again; m; m &= m - 1) {
            const int i = __ffs(m) - 1;
            const float v = out[(size_t)token(i) * rows + end_row];
            if (stands(rv.token[32 * end_h + i], stage ? rv.row[32 * wr + (end_lane & 31)] : any, v, (float)cols)) keep &= ~(1u << i);
        }
        again = keep;
        left = review_votes(rv, again, wr, ks, stage + 1);
    }
    if (left > kMany) {
        f32x16 sum[2][2] = {};
        static_assert(2 * kChunkFloats * 4 <= (int)sizeof(sx), "both halves' chunks");
        fp32_tile<T>(sum, wb, xb, cols, r0, t0, first, kend, 2 * steps, wr, (float *)&sx[0][0][0] + ks * kChunkFloats);
        __syncthreads();
        if (ks == 1) {
#pragma unroll
            for (int i = 0; i < 32; ++i) meet[64 * i] = sum[i >> 4][0][i & 15] + sum[i >> 4][1][i & 15];
        }
        __syncthreads();
        if (ks == 1) return;
#pragma unroll
        for (int i = 0; i < 32; ++i)
            if (end_row < rows && token(i) < batch)
                out[(size_t)token(i) * rows + end_row] = (sum[i >> 4][0][i & 15] + sum[i >> 4][1][i & 15]) + meet[64 * i];
        return;
    }
    if (ks == 1) return;
    for (int i = 0; i < 32; ++i)
        for (uint64_t need = __ballot(again >> i & 1); need; need &= need - 1) {
            const int l = __ffsll((unsigned long long)need) - 1;
            const int at = __builtin_amdgcn_readlane(end_row, l), tok = __builtin_amdgcn_readlane(token(i), l);
            const float v = plain_dot<T>(w, x, cols, at, tok, k0, k1);
            if (end_lane == l) out[(size_t)tok * rows + at] = v;
        }
}

// y = the splits' partial sums added in split order.
__global__ __launch_bounds__(256) void dense_combine(const float *__restrict__ part, float *__restrict__ y,
    size_t n, int splits)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        float s = part[i];
        for (int z = 1; z < splits; ++z) s += part[(size_t)z * n + i];
        y[i] = s;
    }
}

// us before (one fp32 MFMA chain, 64 x 64 tiles) and now, 4096 x 4096 by
// tokens, alone on the stream:
//          16          333          512          2048
//   F16    38 -> 19    219 -> 73    235 -> 85    690 -> 345
//   BF16   38 -> 18    243 -> 68    241 -> 71
//   F32    34 -> 28    208 -> 105   213 -> 115
// (of which the largest magnitude and the rows' bits cost 3 to 5 us at 512.)
// At 512 tokens that is 1010 (F16), 730 (BF16) and 900 (F32) TFLOP/s issued
// of the 1406 a large bf16 product reaches here: what bounds it now. Rows of
// a multiple of 16 bytes load 16 bytes per lane, of 4 bytes 4 (F16 1000 x 1002,
// 700 tokens: 55 with the fp32 cores, 57 in loads of 2, 30 in loads of 4), the
// others element by element (F16 1000 x 1001 the same: 55, 60 with the steps past
// the end loaded too, 47 without).
template <unsigned T>
hipError_t launch_gemm(const uint8_t *w, const float *x, float *y, int rows, int cols, int batch, int splits,
    float *part, hipStream_t s)
{
    const int steps = (cols + kGemmK - 1) / kGemmK, per = (steps + splits - 1) / splits;
    const dim3 grid((unsigned)((rows + kGemmRows - 1) / kGemmRows), (unsigned)((batch + kGemmTokens - 1) / kGemmTokens),
                    (unsigned)splits);
    if ((size_t)cols * kElem<T> % 16 == 0)
        hipLaunchKernelGGL((dense_gemm<T, 16>), grid, dim3(512), 0, s, w, x, y, rows, cols, batch, per, part);
    else if ((size_t)cols * kElem<T> % 4 == 0)
        hipLaunchKernelGGL((dense_gemm<T, 4>), grid, dim3(512), 0, s, w, x, y, rows, cols, batch, per, part);
    else if constexpr (T != F32)
        hipLaunchKernelGGL((dense_gemm<T, 2>), grid, dim3(512), 0, s, w, x, y, rows, cols, batch, per, part);
    if (splits > 1) {
        const size_t n = (size_t)batch * rows;
        const size_t blocks = (n + 255) / 256;
        hipLaunchKernelGGL(dense_combine, dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(256), 0, s, part, y, n,
                           splits);
    }
    return hipGetLastError();
}

}  // namespace

// Column splits of the dense GEMM: where the row and token tiles leave most
// of the 256 CUs idle (small batches of matrices up to a few thousand rows),
// the columns are split over up to 8 workgroups (at least 8 chunks of 32
// columns each), whose partial sums a second launch adds in order.
int dense_gemm_splits(int rows, int cols, int batch)
{
    const long tiles = (long)((rows + kGemmRows - 1) / kGemmRows) * ((batch + kGemmTokens - 1) / kGemmTokens);
    int splits = 1;
    while (splits < 8 && tiles * splits < 192 && (cols + 31) / 32 >= 16 * splits) splits *= 2;
    return splits;
}

size_t dense_gemm_workspace(int rows, int cols, int batch)
{
    const int splits = dense_gemm_splits(rows, cols, batch);
    return splits > 1 ? (size_t)splits * batch * rows * sizeof(float) : 0;
}

// The whole batch in one GEMM launch (batch > 8). The buffer ranges are
// 32-bit: W, X and Y each below 2 GiB.
bool dense_gemm_supported(unsigned type, int rows, int cols, int batch)
{
    if (type != F32 && type != F16 && type != BF16) return false;
    const size_t esize = type == F32 ? 4 : 2;
    return batch > 8 && rows > 0 && cols > 0 && batch <= 65535 * kGemmTokens &&
           (size_t)rows * cols * esize <= (size_t)INT32_MAX && (size_t)batch * cols * 4 <= (size_t)INT32_MAX &&
           (size_t)batch * rows <= (size_t)INT32_MAX;
}

// Rows short enough for the fp32 matrix cores (no column splits there). us, bf16 /
// fp32 cores, 4096 rows by 333 and 2048 tokens (192 and 1024 tiles):
//   columns   64             128            160            192            256            320
//   F16     10.0/6.7      9.9/9.0       12.2/10.4      12.5/11.9      12.6/14.9      15.0/17.7
//           35.7/18.5    35.5/27.1      44.0/32.4      45.5/38.3      45.7/47.9      55.4/56.9
//   F32     11.9/6.6     12.3/8.3       15.8/9.6       15.8/11.1      15.8/13.7      18.7/16.4
//           43.0/19.3    44.6/27.5      57.4/33.5      57.5/38.5      58.1/48.8      71.5/61.2
// (F32, 384: 18.7/18.7 and 73.5/70.3; BF16 as F16). Rows that are not multiples of
// 16 bytes, whose loads the fp32 tile does one by one: F16 66 columns 9.7/10.4 and
// 34.4/28.4, 98 9.7/13.6 and 34.3/37.8; 155 (2-byte loads on both sides) 18.1/16.7
// and 66.2/44.0, 193 20.1/21.3 and 74.3/57.8; F32 82 11.0/10.3 and 39.3/29.1, 155
// 14.2/15.9 and 51.9/43.8.
static bool dense_gemm_short(unsigned type, int rows, int cols, int batch)
{
    const long tiles = (long)((rows + kGemmRows - 1) / kGemmRows) * ((batch + kGemmTokens - 1) / kGemmTokens);
    const bool many = tiles > 256;   // more than one workgroup per CU
    if (type == F32) return cols <= (cols % 4 == 0 ? (many ? 448 : 320) : many ? 160 : 88);
    return cols <= (cols % 8 == 0 ? (many ? 192 : 160) : cols % 2 == 0 ? (many ? 80 : 64) : many ? 224 : 160);
}

hipError_t launch_dense_gemm(unsigned type, const uint8_t *w, const float *x, float *y, int rows, int cols,
    int batch, void *workspace, size_t workspace_bytes, hipStream_t s)
{
    if (!dense_gemm_supported(type, rows, cols, batch)) return hipErrorInvalidValue;
    // Without room for the partial sums, one workgroup per tile covers all
    // columns.
    const size_t need = dense_gemm_workspace(rows, cols, batch);
    const int splits = need && workspace && workspace_bytes >= need ? dense_gemm_splits(rows, cols, batch) : 1;
    float *part = (float *)workspace;
    if (dense_gemm_short(type, rows, cols, batch)) {
        const dim3 grid((unsigned)((rows + kGemmRows - 1) / kGemmRows), (unsigned)((batch + kGemmTokens - 1) / kGemmTokens));
        if (type == F32) hipLaunchKernelGGL(dense_gemm<F32>, grid, dim3(256), 0, s, w, x, y, rows, cols, batch);
        else if (type == F16) hipLaunchKernelGGL(dense_gemm<F16>, grid, dim3(256), 0, s, w, x, y, rows, cols, batch);
        else hipLaunchKernelGGL(dense_gemm<BF16>, grid, dim3(256), 0, s, w, x, y, rows, cols, batch);
        return hipGetLastError();
    }
    if (type == F32) return launch_gemm<F32>(w, x, y, rows, cols, batch, splits, part, s);
    if (type == F16) return launch_gemm<F16>(w, x, y, rows, cols, batch, splits, part, s);
    return launch_gemm<BF16>(w, x, y, rows, cols, batch, splits, part, s);
}

hipError_t launch_dense(unsigned type, const uint8_t *w, const float *x, float *y,
    int rows, int cols, int batch, hipStream_t s)
{
    switch (type) {
    case F32: return launch_type<F32>(w, x, y, rows, cols, batch, s);
    case F16: return launch_type<F16>(w, x, y, rows, cols, batch, s);
    case BF16: return launch_type<BF16>(w, x, y, rows, cols, batch, s);
    default: return hipErrorInvalidValue;
    }
}

namespace {
__global__ __launch_bounds__(256) void copy16(uint4 *__restrict__ dst, const uint4 *__restrict__ src, size_t count)
{
    for (size_t i = blockIdx.x * 256u + threadIdx.x; i < count; i += (size_t)gridDim.x * 256u) dst[i] = src[i];
}
}  // namespace

hipError_t launch_copy(uint4 *dst, const uint4 *src, size_t count, hipStream_t stream)
{
    const size_t blocks = (count + 255) / 256;
    hipLaunchKernelGGL(copy16, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, stream, dst, src, count);
    return hipGetLastError();
}

namespace {
// Plain streaming read of `bytes` (a multiple of 16): one workgroup of four
// wavefronts per CU over a contiguous share; each wavefront issues 32
// non-temporal 16-byte loads per lane per pass (1 KiB per load, wavefronts
// interleaved per KiB), the fastest plain read of a 33 MB matrix measured
// among 2..16 wavefronts and 8..64 loads in flight. Loads past the share
// read zeros (buffer range check); they stay live through an xor that is
// stored only if it equals a constant.
constexpr int kReadWaves = 4, kReadDepth = 32;
__global__ __launch_bounds__(64 * kReadWaves) void read16(const uint8_t *__restrict__ src, size_t bytes, size_t share,
    unsigned *__restrict__ sink)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t begin = (size_t)blockIdx.x * share;
    const size_t n = begin < bytes ? (bytes - begin < share ? bytes - begin : share) : 0;
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(src + begin), (short)0, (int)n, 0x00020000);
    u32x4 acc = {0u, 0u, 0u, 0u};
    for (size_t pass = 0; pass < n; pass += (size_t)1024 * kReadWaves * kReadDepth) {
        u32x4 v[kReadDepth];
#pragma unroll
        for (int u = 0; u < kReadDepth; ++u)
            v[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       r, (int)(pass + 1024 * (u * kReadWaves + wave)) + 16 * lane, 0, 2));
#pragma unroll
        for (int u = 0; u < kReadDepth; ++u) acc ^= v[u];
    }
    const unsigned x = acc.x ^ acc.y ^ acc.z ^ acc.w;
    if (x == 0x9E3779B9u) sink[blockIdx.x] = x;
}
}  // namespace

hipError_t launch_read(const uint4 *src, size_t count, unsigned *sink, hipStream_t stream)
{
    const int cus = device_cu_count();
    const unsigned blocks = (unsigned)(cus < kReadSinkWords ? cus : kReadSinkWords);
    const size_t bytes = count * 16;
    // Shares are whole KiB, and below 2 GiB for the 32-bit buffer range.
    const size_t share = (bytes + (size_t)1024 * blocks - 1) / ((size_t)1024 * blocks) * 1024;
    if (share > (size_t)INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(read16, dim3(blocks), dim3(64 * kReadWaves), 0, stream, (const uint8_t *)src, bytes, share,
                       sink);
    return hipGetLastError();
}

namespace {
// The same streaming read in other shapes, to find the fastest plain read of
// a given size: W wavefronts per workgroup, D 16-byte loads in flight per
// lane per pass, and the loads either into registers (MODE 0 non-temporal,
// MODE 1 the default cache policy) or straight into LDS (MODE 2,
// buffer_load_dwordx4 ... lds: wavefront w's D KiB at LDS offset w D KiB,
// waited for before the next pass reuses it); MODE 3 is MODE 0 followed by
// an output store of 56 words per workgroup, as a matvec's y. A workgroup reads one
// contiguous share; past it the buffer range check returns zeros.
template <int W, int D, int MODE>
__global__ __launch_bounds__(64 * W) void read_shaped(const uint8_t *__restrict__ src, size_t bytes, size_t share,
    unsigned *__restrict__ sink)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t begin = (size_t)blockIdx.x * share;
    const size_t n = begin < bytes ? (bytes - begin < share ? bytes - begin : share) : 0;
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(src + begin), (short)0, (int)n, 0x00020000);
    u32x4 acc = {0u, 0u, 0u, 0u};
    if constexpr (MODE == 2) {
        extern __shared__ __align__(16) uint8_t lds[];
        for (size_t pass = 0; pass < n; pass += (size_t)1024 * W * D) {
#pragma unroll
            for (int u = 0; u < D; ++u)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    r, (__attribute__((address_space(3))) void *)(lds + 1024 * (wave * D + u)), 16, 16 * lane,
                    (int)(pass + 1024 * (u * W + wave)), 0, 0);
            // The copies land before the next pass overwrites the same LDS.
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        acc = *(const u32x4 *)(lds + 1024 * wave * D + 16 * lane);
    } else {
        for (size_t pass = 0; pass < n; pass += (size_t)1024 * W * D) {
            u32x4 v[D];
#pragma unroll
            for (int u = 0; u < D; ++u)
                v[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                           r, (int)(pass + 1024 * (u * W + wave)) + 16 * lane, 0, MODE == 1 ? 0 : 2));
#pragma unroll
            for (int u = 0; u < D; ++u) acc ^= v[u];
        }
    }
    const unsigned x = acc.x ^ acc.y ^ acc.z ^ acc.w;
    if (MODE == 3) {
        // An output every real kernel has: wavefront 0 stores 56 words per
        // workgroup (a 14336-row matvec's y share), unconditionally.
        if (wave == 0 && lane < 56) sink[(size_t)blockIdx.x * 64 + lane] = x;
    } else if (x == 0x9E3779B9u) {
        sink[blockIdx.x % kReadSinkWords] = x;
    }
}

template <int W, int D, int MODE>
hipError_t launch_shaped(const uint8_t *src, size_t bytes, size_t share, unsigned blocks, unsigned *sink,
    hipStream_t stream)
{
    const size_t lds = MODE == 2 ? (size_t)1024 * W * D : 0;
    hipLaunchKernelGGL((read_shaped<W, D, MODE>), dim3(blocks), dim3(64 * W), lds, stream, src, bytes, share, sink);
    return hipGetLastError();
}
}  // namespace

// (waves, depth) pairs: 4 x 32, 4 x 16, 8 x 16, 8 x 8, 16 x 8, 16 x 4, all
// at most 128 KiB in flight per workgroup (the LDS form holds them all).
hipError_t launch_read_shaped(const uint4 *src, size_t count, unsigned *sink, int waves, int depth, int per_cu,
    int mode, hipStream_t stream)
{
    if (mode < 0 || mode > 3 || per_cu < 1 || per_cu > 4) return hipErrorInvalidValue;
    const unsigned blocks = (unsigned)(device_cu_count() * per_cu);
    const size_t bytes = count * 16;
    const size_t share = (bytes + (size_t)1024 * blocks - 1) / ((size_t)1024 * blocks) * 1024;
    if (share > (size_t)INT32_MAX) return hipErrorInvalidValue;
    if (mode == 3 && (size_t)blocks * 256 > NYA_HIP_READ_STORE_SINK_BYTES) return hipErrorInvalidValue;
    const uint8_t *s = (const uint8_t *)src;
#define FY_SHAPE(w, d)                                                                                            \
    if (waves == w && depth == d) {                                                                               \
        if (mode == 0) return launch_shaped<w, d, 0>(s, bytes, share, blocks, sink, stream);                     \
        if (mode == 1) return launch_shaped<w, d, 1>(s, bytes, share, blocks, sink, stream);                     \
        if (mode == 2) return launch_shaped<w, d, 2>(s, bytes, share, blocks, sink, stream);                     \
        return launch_shaped<w, d, 3>(s, bytes, share, blocks, sink, stream);                                    \
    }
    FY_SHAPE(4, 32)
    FY_SHAPE(4, 16)
    FY_SHAPE(8, 16)
    FY_SHAPE(8, 8)
    FY_SHAPE(16, 8)
    FY_SHAPE(16, 4)
#undef FY_SHAPE
    return hipErrorInvalidValue;
}

}  // namespace fy
