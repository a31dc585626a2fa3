// Causal attention of a run of prompt tokens over the KV cache on the fp32
// matrix cores (v_mfma_f32_32x32x2_f32): head widths 64, 128 and 256. Each
// output restates the engine's step (backend/core/llm_cpu.c:491-511) with the
// softmax taken online over key tiles; everything stays fp32.
//
// Bound. Per (query row, key) 4 W flops and nothing to re-read but K and V:
// the matrix cores. The per-head kernel (resident.hip, attention_w) streams a
// head's whole history for every token instead. 512 tokens at positions
// 3584..4095: 32/8 heads of 128 took 2720 us there (12 TFLOP/s), 365 here (88,
// 58 % of what an fp32 library product reaches on this card); 32/4 heads of
// 64 1336 -> 199 us; 16/8 heads of 256 3408 -> 870 us. What is left is the
// softmax's expf and the barriers between the two products.
//
// Work split. The query heads that share a KV head are extra query rows: row
// r of KV head k is token r / G, head k G + r % G (G = heads / kv_heads), so
// one 32-row tile shares every K and V tile it reads whatever G is. A
// workgroup holds RG row tiles and splits the keys KS ways: each step covers
// KS key tiles of 32, wavefront (rg, ks) computes row tile rg against key
// tile ks, and the KS partial softmaxes meet in LDS at the end. With one
// wavefront per row tile a 512-token chunk of 32 heads would fill half the
// SIMDs; KS = 4 gives every SIMD two wavefronts (one's softmax runs under the
// other's MFMAs). Workgroups of one KV head share blockIdx % kv_heads, so at 8
// KV heads each XCD's L2 holds one head's cache.
//
// Layout. Both products are formed transposed: S^T = K Q^T leaves lane l the
// scores of query row l % 32 against the keys 8 (i / 4) + 4 (l / 32) + i % 4
// (register i), which is also the operand O^T = V^T P^T wants from lane l at
// MFMA step i (K slot l / 32). Scores become probabilities and feed the second
// product in place; maximum, sum and rescaling are one value per lane.
// Q stays in registers; K tiles lie in LDS in 16-byte chunks permuted by
// chunk ^ row (one ds_read_b128 of every lane feeds four MFMA steps without
// bank conflicts), V tiles as they are. Both arrive by buffer_load ... lds:
// V(t) lands under the scores of step t, K(t + 1) under its softmax and
// second product; two barriers per step.
//
// Sums. Score dots start two chains of 8 MFMAs every 32 columns; each key tile's P V starts
// from zero and is added to the running output as O = O alpha + T, so a chain
// never exceeds 16 MFMAs and the rescale costs nothing extra.
#include <math.h>

#include "device.h"
#include "kernels.h"

#pragma clang fp contract(off)

namespace fy {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) uint8_t lds_u8;

constexpr int kKeys = 32;   // keys per tile

__device__ __forceinline__ void barrier_all()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0);   // this wavefront's copies have landed, its LDS reads are done
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The wavefront's query row in lane l % 32 and what it attends: positions
// [first, last] (last < first: nothing); lowest / highest over the wavefront.
struct QueryRow {
    int first, last, lowest, highest;
};

// This wavefront's share (1 KiB copies rg, rg + RG, ...) of key tile ks of a
// step: rows [key0, key0 + 32) of one KV head, at `base` (row `key0`), `rows`
// of them inside the cache (copies past them read zeros). SWIZZLE: 16-byte
// chunk c of row r goes to place c ^ (r % min(32, chunks)).
template <int W, int RG, bool SWIZZLE>
__device__ __forceinline__ void copy_tile(lds_u8 *dst, const float *base, int rows, uint32_t stride, int rg)
{
    constexpr int kChunks = W / 4, kRowsPerCopy = 64 / kChunks, kCopies = kKeys / kRowsPerCopy;
    constexpr int kMask = kChunks < 32 ? kChunks - 1 : 31;
    // Opaque: the addresses are formed where they are used instead of living
    // in registers throughout the kernel.
    int lane = threadIdx.x & 63;
    asm("" : "+v"(lane));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(base), (short)0, (int)((uint32_t)(rows < 0 ? 0 : rows < kKeys ? rows : kKeys) * stride),
        0x00020000);
#pragma unroll
    for (int k = 0; k < kCopies / RG; ++k) {
        const int j = rg + RG * k;
        const int row = kRowsPerCopy * j + lane / kChunks, place = lane % kChunks;
        const int chunk = SWIZZLE ? place ^ (row & kMask) : place;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void *)(dst + 1024 * j), 16,
                                                 (int)((uint32_t)row * stride) + 16 * chunk, 0, 0, 0);
    }
}

// Step, first half: V's copies go out, the scores of this wavefront's tile
// come in (kt: its K tile).
template <int W, int RG>
__device__ __forceinline__ void score_step(const lds_u8 *__restrict__ kt, lds_u8 *__restrict__ vt,
    const float *vbase, int rows, uint32_t stride, int rg, const float4 (&qv)[W / 8], bool active, f32x16 &S)
{
    constexpr int kChunks = W / 4, kMask = kChunks < 32 ? kChunks - 1 : 31;
    int lane = threadIdx.x & 63;
    asm("" : "+v"(lane));   // as in copy_tile
    const int key = lane & 31, h = lane >> 5;
    copy_tile<W, RG, false>(vt, vbase, rows, stride, rg);
    if (active) {
        const lds_u8 *row = kt + 4 * W * key;
        // Four chunks' MFMAs run while the next four are read; every 32
        // columns start two new chains.
        constexpr int kAhead = 4, kParts = W / 8 / kAhead;
        float4 k[2][kAhead];
        auto read = [&](int part, float4 (&dst)[kAhead]) {
#pragma unroll
            for (int c = 0; c < kAhead; ++c)
                dst[c] = *(const float4 *)(row + 16 * ((2 * (kAhead * part + c) + h) ^ (key & kMask)));
        };
        read(0, k[0]);
#pragma unroll
        for (int part = 0; part < kParts; ++part) {
            if (part + 1 < kParts) read(part + 1, k[(part + 1) & 1]);
            f32x16 s0 = {}, s1 = {};
#pragma unroll
            for (int c = 0; c < kAhead; ++c) {
                const float4 a = k[part & 1][c], b = qv[kAhead * part + c];
                s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, s1, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, s1, 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) S[i] = part ? S[i] + (s0[i] + s1[i]) : s0[i] + s1[i];
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    barrier_all();
}

__device__ __forceinline__ bool finite_bits(float v)
{
    return (__builtin_bit_cast(uint32_t, v) & 0x7F800000u) != 0x7F800000u;
}

// Step, second half: the next step's K copies go out; online softmax of S
// over keys key0 + 8 (i / 4) + 4 h + i % 4, then O = O alpha + V^T P^T.
// BOUNDARY: some row does not see all of the tile. Unseen keys get
// probability 0, and since 0 times a non-finite value would still reach
// every row, V's non-finite elements enter the product as 0 and are added
// afterwards to the rows that do see them.
template <int W, bool BOUNDARY>
__device__ __forceinline__ void output_tile(const lds_u8 *vt, const QueryRow &qr, int key0, float scale,
    f32x16 &S, float &m, float &l, f32x16 (&O)[W / 32])
{
    const int lane = threadIdx.x & 63, h = lane >> 5;
    // Key i of this lane is seen iff (unsigned)(from + 8 (i / 4) + i % 4) < span.
    const unsigned from = (unsigned)(key0 + 4 * h - qr.first), span = (unsigned)(qr.last - qr.first + 1);
    float top = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        S[i] = S[i] * scale;
        if constexpr (BOUNDARY) {
            if (from + (unsigned)(8 * (i >> 2) + (i & 3)) >= span) S[i] = -INFINITY;
        }
        top = fmaxf(top, S[i]);
    }
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    const float next = fmaxf(m, top);
    const float alpha = next == m ? 1.f : expf(m - next);
    m = next;
    // Scores of minus infinity have probability 0 also where the row has seen
    // nothing else yet (a row that never does ends in 0 / 0).
    const float top_seen = next == -INFINITY ? 0.f : next;
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        float e = expf(S[i] - top_seen);
        if constexpr (BOUNDARY) {
            if (from + (unsigned)(8 * (i >> 2) + (i & 3)) >= span) e = 0.f;
        }
        S[i] = e;
        sum[i & 3] += e;
    }
    l = l * alpha + ((sum[0] + sum[1]) + (sum[2] + sum[3]));
    // 64 columns at a time: row 2 x + e of V's 32 x 64 part in tile e.
    const lds_u8 *col = vt + 4 * W * 4 * h + 8 * (lane & 31);
#pragma unroll
    for (int part = 0; part < W / 64; ++part) {
        f32x16 t0 = {}, t1 = {};
        bool odd = false;
        constexpr int kAhead = 4;
        float2 v[2][kAhead];
        auto read = [&](int four, float2 (&dst)[kAhead]) {
#pragma unroll
            for (int i = 0; i < kAhead; ++i)
                dst[i] = *(const float2 *)(col + 4 * W * (8 * four + i) + 256 * part);
        };
        read(0, v[0]);
#pragma unroll
        for (int four = 0; four < 4; ++four) {
            if (four < 3) read(four + 1, v[(four + 1) & 1]);
#pragma unroll
            for (int i = 0; i < kAhead; ++i) {
                float2 a = v[four & 1][i];
                if constexpr (BOUNDARY) {
                    if (!finite_bits(a.x)) a.x = 0.f, odd = true;
                    if (!finite_bits(a.y)) a.y = 0.f, odd = true;
                }
                t0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, S[4 * four + i], t0, 0, 0, 0);
                t1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, S[4 * four + i], t1, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (BOUNDARY) {
            if (__builtin_amdgcn_ballot_w64(odd)) {
                // Rare: this lane's columns 64 part + 2 x + e, x = 8 (i / 4) + 4 h + i % 4.
                // `none`: the row's keys of probability 0.
                uint32_t none = 0;
#pragma unroll
                for (int i = 0; i < 16; ++i) none |= (S[i] == 0.f ? 1u : 0u) << (8 * (i >> 2) + 4 * h + (i & 3));
                none |= (uint32_t)__shfl_xor((int)none, 32, 64);
#pragma unroll 1
                for (int t = 0; t < kKeys; ++t) {
                    const bool seen = key0 + t >= qr.first && key0 + t <= qr.last;
                    const float p = none >> t & 1 ? 0.f : 1.f;   // (not finite times more than 0: itself)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const float2 v = *(const float2 *)(vt + 4 * W * t + 256 * part +
                                                           8 * (8 * (i >> 2) + 4 * h + (i & 3)));
                        if (seen && !finite_bits(v.x)) t0[i] += v.x * p;
                        if (seen && !finite_bits(v.y)) t1[i] += v.y * p;
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            O[2 * part][i] = __builtin_fmaf(O[2 * part][i], alpha, t0[i]);
            O[2 * part + 1][i] = __builtin_fmaf(O[2 * part + 1][i], alpha, t1[i]);
        }
    }
}

template <int W, int RG>
__device__ __forceinline__ void output_step(lds_u8 *__restrict__ kt, const lds_u8 *__restrict__ vt,
    const float *kbase, int rows, uint32_t stride, int rg, const QueryRow &qr, int key0, float scale, bool active,
    f32x16 &S, float &m, float &l, f32x16 (&O)[W / 32])
{
    copy_tile<W, RG, true>(kt, kbase, rows, stride, rg);
    if (active) {
        const bool whole = qr.first <= key0 && qr.last >= key0 + kKeys - 1;
        if (__builtin_amdgcn_ballot_w64(whole) == ~0ull)
            output_tile<W, false>(vt, qr, key0, scale, S, m, l, O);
        else
            output_tile<W, true>(vt, qr, key0, scale, S, m, l, O);
    }
    barrier_all();
}

// Wavefronts per SIMD: two (eight-wavefront workgroups, or two workgroups per
// CU at width 64); one for the four-wavefront shapes of width 128 and 256,
// whose tiles fill the LDS.
template <int W, int RG, int KS> constexpr int kPerSimd = W == 64 ? 2 : RG * KS / 4;

// Workgroups of a shape that fits a CU twice, on the whole chip.
template <int W, int RG> constexpr int kAtOnce = W == 64 && RG == 1 ? 512 : 0;

template <int W, int RG, int KS>
__global__ __launch_bounds__(64 * RG * KS)
__attribute__((amdgpu_waves_per_eu(kPerSimd<W, RG, KS>, kPerSimd<W, RG, KS>))) void attention_tile(
    const float *q, int q_stride, const float *__restrict__ keys, const float *__restrict__ values, float *out,
    const int *__restrict__ positions, int count, int heads, int kv_heads, int max_length, int window, float scale)
{
    constexpr int kTileBytes = 4 * W * kKeys;
    __shared__ __align__(16) uint8_t smem_k[KS * kTileBytes], smem_v[KS * kTileBytes];
    __shared__ float2 smem_ml[RG * KS][32];
    __shared__ int smem_range[2][RG * KS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rg = wave / KS, ks = wave % KS, h = lane >> 5;
    const int group = heads / kv_heads, rows = count * group;
    const int blocks = (rows + 32 * RG - 1) / (32 * RG);
    // Later tokens see more: their workgroups start first. Where all of them
    // run at once, two to a CU, the second half of the grid goes from the first
    // tokens on instead, so that a CU's two see about as many keys together.
    const int kvh = blockIdx.x % kv_heads, b = (int)(blockIdx.x / kv_heads);
    const int block = kAtOnce<W, RG> && (int)gridDim.x <= kAtOnce<W, RG> && 2 * b >= blocks ? b - (blocks + 1) / 2
                                                                                          : blocks - 1 - b;
    const int row_raw = 32 * (RG * block + rg) + (lane & 31);
    const int row = row_raw < rows ? row_raw : rows - 1;
    const int token = row / group, head = kvh * group + row % group;
    QueryRow qr;
    {
        const int p = positions[token];
        const int end = p < 0 ? -1 : p >= max_length ? max_length - 1 : p;
        qr.first = window > 0 && end >= window ? end - window + 1 : 0;
        qr.last = end;
    }
    // [lowest, highest] of the wavefront, then of the workgroup.
    int lo = qr.last < 0 ? max_length : qr.first, hi = qr.last;
#pragma unroll
    for (int o = 16; o >= 1; o >>= 1) {
        lo = min(lo, __shfl_xor(lo, o, 64));
        hi = max(hi, __shfl_xor(hi, o, 64));
    }
    qr.lowest = __builtin_amdgcn_readfirstlane(lo);
    qr.highest = __builtin_amdgcn_readfirstlane(hi);
    if (lane == 0) {
        smem_range[0][wave] = qr.lowest;
        smem_range[1][wave] = qr.highest;
    }
    float4 qv[W / 8];
    const float4 *q4 = (const float4 *)(q + (size_t)token * q_stride + (size_t)head * W);
#pragma unroll
    for (int c = 0; c < W / 8; ++c) qv[c] = q4[2 * c + h];
    __syncthreads();
    int begin = max_length, end = -1;
#pragma unroll
    for (int w = 0; w < RG * KS; ++w) {
        begin = min(begin, smem_range[0][w]);
        end = max(end, smem_range[1][w]);
    }
    begin = __builtin_amdgcn_readfirstlane(begin);
    end = __builtin_amdgcn_readfirstlane(end);

    const uint32_t stride = 4u * W * (uint32_t)kv_heads;
    const float *kh = keys + (size_t)kvh * W, *vh = values + (size_t)kvh * W;
    const size_t row_floats = (size_t)kv_heads * W;
    lds_u8 *const kt = (lds_u8 *)smem_k + ks * kTileBytes, *const vt = (lds_u8 *)smem_v + ks * kTileBytes;
    f32x16 O[W / 32];
#pragma unroll
    for (int d = 0; d < W / 32; ++d) O[d] = (f32x16){};
    float m = -INFINITY, l = 0.f;
    int key0 = begin + kKeys * ks;
    copy_tile<W, RG, true>(kt, kh + (size_t)(key0 < max_length ? key0 : 0) * row_floats,
                           key0 < max_length ? max_length - key0 : 0, stride, rg);
    barrier_all();
    for (int at = begin; at <= end; at += kKeys * KS, key0 += kKeys * KS) {
        const bool active = key0 <= qr.highest && key0 + kKeys - 1 >= qr.lowest;
        const int here = key0 < max_length ? key0 : 0, left = key0 < max_length ? max_length - key0 : 0;
        f32x16 S;
        score_step<W, RG>(kt, vt, vh + (size_t)here * row_floats, left, stride, rg, qv, active, S);
        const int nk = key0 + kKeys * KS, next = nk < max_length ? nk : 0, nleft = nk < max_length ? max_length - nk : 0;
        output_step<W, RG>(kt, vt, kh + (size_t)next * row_floats, nleft, stride, rg, qr, key0, scale, active, S, m, l,
                           O);
    }

    // The KS partial softmaxes of each row tile: each wavefront leaves its
    // output rows (float2 f of row r at place f ^ (r % 32)) and (m, l); then
    // out = sum_k O_k e^(m_k - M) / sum_k l_k e^(m_k - M).
    l += __shfl_xor(l, 32, 64);
    lds_u8 *const part = rg == 0 ? kt : vt;
    static_assert(RG <= 2, "one LDS region per row tile");
#pragma unroll
    for (int p = 0; p < W / 64; ++p)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int f = 32 * p + 8 * (i >> 2) + 4 * h + (i & 3);
            *(float2 *)(part + 4 * W * (lane & 31) + 8 * (f ^ (lane & 31))) = make_float2(O[2 * p][i], O[2 * p + 1][i]);
        }
    if (h == 0) smem_ml[wave][lane] = make_float2(m, l);
    __syncthreads();
    const uint8_t *const parts = rg == 0 ? smem_k : smem_v;
    for (int i = ks * 64 + lane; i < 32 * (W / 2); i += 64 * KS) {
        const int r = i / (W / 2), f = i % (W / 2);
        const int rr = 32 * (RG * block + rg) + r;
        if (rr >= rows) continue;
        const int tok = rr / group;
        if (positions[tok] < 0) continue;
        float top = -INFINITY;
#pragma unroll
        for (int k = 0; k < KS; ++k) top = fmaxf(top, smem_ml[rg * KS + k][r].x);
        float total = 0.f;
        float2 o = make_float2(0.f, 0.f);
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const float2 ml = smem_ml[rg * KS + k][r];
            const float w = ml.x == -INFINITY ? 0.f : expf(ml.x - top);
            const float2 v = *(const float2 *)(parts + k * kTileBytes + 4 * W * r + 8 * (f ^ (r & 31)));
            total += ml.y * w;
            o.x += v.x * w;
            o.y += v.y * w;
        }
        *(float2 *)(out + ((size_t)tok * heads + kvh * group + rr % group) * W + 2 * f) =
            make_float2(o.x / total, o.y / total);
    }
}

template <int W, int RG, int KS>
hipError_t launch_tile(const float *q, int q_stride, const float *keys, const float *values, float *out,
    const int *positions, int count, int heads, int kv_heads, int max_length, int window, float scale, hipStream_t s)
{
    const long rows = (long)count * (heads / kv_heads), blocks = (rows + 32 * RG - 1) / (32 * RG);
    hipLaunchKernelGGL((attention_tile<W, RG, KS>), dim3((unsigned)(blocks * kv_heads)), dim3(64 * RG * KS), 0, s, q,
                       q_stride, keys, values, out, positions, count, heads, kv_heads, max_length, window, scale);
    return hipGetLastError();
}

}  // namespace

// The runs this kernel takes from the per-head kernel, which fills the chip
// with one workgroup per (token, head) and so wins on few of them and on short
// ranges: its time grows with tokens x heads x range, this kernel's stays that of
// one workgroup's key steps (17 us with one, 7.6 more for each, at width 128) until
// the chip is full. The positions are on the device: what is known of the ranges
// is that none exceeds max_length or the window. us, per-head / this kernel:
//   tokens x heads     window 64      128        512     run's end 512   4096
//    64 x 32 of 128    12.3/17.1  15.3/24.6   44.4/45.0   42.7/36.8    340/221
//    96 x 32 of 128    16.5/17.2  20.9/24.8   63.2/45.2   64.5/43.9    502/222
//   128 x 32 of 128    20.5/17.4  27.1/25.1   82.5/45.3   86.0/44.0    657/221
//    64 x 32 of  64     9.2/10.5  10.0/14.7   25.7/26.5   24.8/22.2    172/140
//   256 x 16 of 256    25.5/47.3  43.1/60.3    148/140     119/125    1653/862
//   512 x 16 of 256    48.0/48.3  81.0/61.2    289/141     166/126    3395/872
//   200 x 48 of 256    58.0/92.6  99.0/119     402/285     441/269    9108/1700
// and of runs from position 0: 64, 96 and 128 x 32 of 128 12.7/17.3, 17.1/17.2,
// 22.7/17.4; of 64 8.9/10.3, 11.8/10.4, 14.9/10.4; 256 and 512 x 16 of 256 48/72,
// 166/126; 512 x 8 of 256 79/125; 200 x 48 of 256 94/78. So, in (token, head)
// pairs, at width 64 and 128: 4096, 3072 unless a window below 512 keeps the ranges
// short, 2048 where they may reach 512 (a window 1024); at width 256: 24576, 8192
// unless a window is below 256, 4096 where they may reach 512 in a run that may
// reach 1024. Fewer pairs that see little of a longer cache lose what the
// figures show; a caller that knows its run's end passes it as max_length.
bool attention_tile_supported(int count, int heads, int kv_heads, int width, int max_length, int window)
{
    if (width != 64 && width != 128 && width != 256) return false;
    const bool windowed = window > 0 && window < max_length;
    const int range = windowed ? window : max_length;
    const long pairs = (long)count * heads;
    if (width <= 128 ? pairs < (windowed && range < 512 ? 4096 : range < (windowed ? 1024 : 512) ? 3072 : 2048)
                     : pairs < (windowed && range < 256 ? 24576 : range < 512 || max_length < 1024 ? 8192 : 4096))
        return false;
    const long rows = (long)count * (heads / kv_heads);
    // 32-bit row counts, grid and per-tile buffer offsets.
    return rows <= (long)1 << 30 && (rows / 32 + 1) * kv_heads <= (long)1 << 30 &&
           (long)kv_heads * width <= (long)1 << 23;
}

hipError_t launch_attention_tile(const float *q, int q_stride, const float *keys, const float *values, float *out,
    const int *positions, int count, int heads, int kv_heads, int width, int max_length, int window, float scale,
    hipStream_t s)
{
    const long rows = (long)count * (heads / kv_heads);
    // Two row tiles per workgroup (a K and V tile read once for both) where
    // those workgroups fill the 256 CUs, else one (twice the
    // workgroups): 32 heads of 128 over 4096 positions, 256 tokens with one
    // take 229 us, 512 tokens with two 368. At width 64 two workgroups of one
    // tile fit a CU: until those fill the chip, which the order of the grid
    // balances (32/4 heads, 512 tokens from position 0: 33.5 us with two tiles,
    // 26.7 with one; 16/16, 1024 tokens: 54 and 41; at positions 3584..4095 of
    // 32/8 heads, where all see as much: 194 and 198; past one round the pairs
    // win, 32/4 heads, 1024 tokens: 73 and 79).
    const bool pairs = width == 64 ? (rows + 31) / 32 * kv_heads > kAtOnce<64, 1> : (rows + 63) / 64 * kv_heads >= 256;
#define FY_TILE(WW, RGG, KSS) \
    launch_tile<WW, RGG, KSS>(q, q_stride, keys, values, out, positions, count, heads, kv_heads, max_length, window, scale, s)
    if (width == 64) return pairs ? FY_TILE(64, 2, 4) : FY_TILE(64, 1, 4);
    if (width == 128) return pairs ? FY_TILE(128, 2, 4) : FY_TILE(128, 1, 4);
    return pairs ? FY_TILE(256, 2, 2) : FY_TILE(256, 1, 2);
#undef FY_TILE
}

}  // namespace fy
