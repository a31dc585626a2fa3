// Products of 9..64 tokens with quantized weights that need no workspace: the
// weights are read once for the whole batch, where 8-token launches read and
// decode them again for every eight.
//
// Y[n][row] = sum_k W[row][k] X[n][k] on v_mfma_f32_16x16x4_f32: weights
// decoded to fp32 as the reference decodes them
// (backend/core/llm_quant.c:70-142), activations as they are, fp32 sums.
//
// Work split. A workgroup of eight wavefronts owns 16 rows (half a tile of
// formats.h) and all tokens; wavefront w takes the 256-column groups w, w + 8,
// ... and the shares meet in LDS at the end, in wavefront order. Within a group
// lane l holds row l % 16 and of every 16 columns its four 4 (l / 16) .. + 3:
// a 4-byte load of packed weights, and one 16-byte load of x per 16 tokens
// (token l % 16), feed four MFMAs per token tile, MFMA j taking the lanes' j-th
// columns. D[token][row]: register i of lane l is token 4 (l / 16) + i, row
// l % 16. Up to four tokens past the whole tiles are summed by fp32 FMAs
// instead (16 cycles of a token's step against 128 of a tile's, full or not).
// A group's sums start from zero and join the running ones afterwards: chains
// of 64 MFMAs at most, and a third of the 8-token launches' error against 64 bits
// (3e-7, 1e-6: their activations are rounded to 22-bit integers per group).
//
// x goes through LDS (copied there without registers, eight tokens' 128 bytes
// per copy, one to three stages of 32 columns ahead): loaded straight into the
// MFMA's lane order, sixteen tokens at a time, every lane is a memory access
// of its own, and the L1's return path bounds the kernel (48 tokens of Q6_K
// 4096 x 14336: 93 us, 60 through LDS). A group's packed weights come into the
// registers of the group before as soon as those have been used.
//
// us, 8-token launches and here:            9    16    17    32    33    48    56 tokens
//   Q6_K 4096 x 14336                      37    53    65   107   117   160   187
//                                          27    30    33    45    53    61    75
//   Q4_K 4096 x 4096                       12    14          26
//                                           9.9   9.8        14.4
// The tokens past the whole tiles as FMAs, Q6_K 4096 x 14336: 17 tokens 31.5, 20
// 35.4, 24 (two tiles) 39.7; 33 46.0, 36 53.2, 48 59.6; 49 61.7, 52 68.1, 64 73.5.
// What bounds it now: from 32 tokens on the fp32 matrix cores (61 % busy at 48
// tokens, 48 % at 33; one wavefront's decoding and waits are covered by one other)
// and the return path of x, which every workgroup reads whole; below that latency.
#include "blockdot.h"
#include "kernels.h"
#include <limits.h>
#include <type_traits>

namespace fy {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint8_t lds_u8;
constexpr int kWaves = 8, kRows = 16;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *p, size_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ uint32_t load4(__amdgpu_buffer_rsrc_t r, int v, int s)
{
    return __builtin_amdgcn_raw_buffer_load_b32(r, v, s, 0);
}
__device__ __forceinline__ u32x4 load16b(__amdgpu_buffer_rsrc_t r, int v, int s)
{
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0));
}

// Waits until at most VM vector memory operations of this wavefront are in
// flight (they complete in order) and its LDS reads are done. The pointers to
// weights and x are not restrict, so that no load crosses this.
template <int VM>
__device__ __forceinline__ void wait_loads()
{
    static_assert(VM < 64, "vmcnt");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4) << 14 | 7 << 4);
    asm volatile("" ::: "memory");
}

// Where a lane reads its row: the tile's first byte is in v4 and v16 (the
// row's 16-byte fields, at the lane's four bytes of one and at its start); R
// rows in the tile.
struct Place {
    int v4, v16, vd, R, groups;
};

// The packed weights of one group, this lane's share. load(i) requests the
// i-th quarter of the quants, scales() the rest; step(s) decodes columns 16 s
// + 4 (l / 16) .. + 3 (s constant).
template <unsigned T> struct Packed;

template <> struct Packed<Q6_K> {
    static constexpr int kScaleLoads = 2, kQuarterLoads = 3;
    uint32_t a[4], b[4], h[4];
    u32x4 sc, own;
    uint32_t d;
    float df;
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t w, const Place &p, int g, int i)
    {
        const int s = p.R * (208 * g + 48 * i);
        a[i] = load4(w, p.v4, s), b[i] = load4(w, p.v4, s + 16 * p.R), h[i] = load4(w, p.v4, s + 32 * p.R);
    }
    __device__ __forceinline__ void scales(__amdgpu_buffer_rsrc_t w, const Place &p, int g)
    {
        sc = load16b(w, p.v16, p.R * (208 * g + 192));
        d = __builtin_amdgcn_raw_buffer_load_b16(w, p.vd, p.R * (208 * p.groups + 2 * g), 0);
    }
    __device__ __forceinline__ void begin() { own = sc, df = f16_to_f32(d); }
    // Quarters (units of formats.h) that step s is the last to use.
    static constexpr int done(int s) { return s == 6 ? 0 : s == 7 ? 1 : s == 14 ? 2 : s == 15 ? 3 : -1; }
    __device__ __forceinline__ void step(int s, float (&v)[4]) const
    {
        const int p = 2 * (s >> 3) + (s & 1), q = (s >> 1) & 3;
        const uint32_t six = (((q & 1 ? b[p] : a[p]) >> (4 * (q >> 1))) & 0x0F0F0F0Fu) |
                             ((q < 2 ? h[p] << (4 - 2 * q) : h[p] >> (2 * q - 4)) & 0x30303030u);
        const float t = df * (float)(int8_t)(own[p] >> (8 * q));   // exact
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = __builtin_fmaf((float)((six >> (8 * j)) & 255u), t, -32.f * t);
    }
};

// Q4_K and Q4_0: nibbles of four units of 64 columns.
template <unsigned T> struct Nibbles {
    static constexpr int kScaleLoads = 1, kQuarterLoads = 2;
    uint32_t a[4], b[4];
    u32x4 sc, own;
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t w, const Place &p, int g, int i)
    {
        const int s = p.R * (144 * g + 32 * i);
        a[i] = load4(w, p.v4, s), b[i] = load4(w, p.v4, s + 16 * p.R);
    }
    __device__ __forceinline__ void scales(__amdgpu_buffer_rsrc_t w, const Place &p, int g)
    {
        sc = load16b(w, p.v16, p.R * (144 * g + 128));
    }
    static constexpr int done(int s) { return s % 4 == 3 ? s / 4 : -1; }
    __device__ __forceinline__ uint32_t quants(int s) const
    {
        return ((s & 1 ? b[s >> 2] : a[s >> 2]) >> (4 * ((s >> 1) & 1))) & 0x0F0F0F0Fu;
    }
};

template <> struct Packed<Q4_K> : Nibbles<Q4_K> {
    float d, dmin;
    __device__ __forceinline__ void begin()
    {
        own = sc;
        const uint32_t dd = (own.x >> 24) | ((own.y >> 24) << 8) | ((own.z >> 24) << 16) | ((own.w >> 24) << 24);
        d = f16_to_f32(dd & 0xFFFFu), dmin = f16_to_f32(dd >> 16);
    }
    __device__ __forceinline__ void step(int s, float (&v)[4]) const
    {
        const uint32_t q = quants(s), f = own[s >> 2] >> (12 * ((s >> 1) & 1));
        const float t = d * (float)(f & 63u), m = -(dmin * (float)((f >> 6) & 63u));   // exact
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = __builtin_fmaf((float)((q >> (8 * j)) & 255u), t, m);
    }
};

template <> struct Packed<Q4_0> : Nibbles<Q4_0> {
    __device__ __forceinline__ void begin() { own = sc; }
    __device__ __forceinline__ void step(int s, float (&v)[4]) const
    {
        const uint32_t q = quants(s);
        const float t = f16_to_f32((own[s >> 2] >> (16 * ((s >> 1) & 1))) & 0xFFFFu);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = __builtin_fmaf((float)((q >> (8 * j)) & 255u), t, -8.f * t);
    }
};

template <> struct Packed<Q8_0> {
    static constexpr int kScaleLoads = 1, kQuarterLoads = 4;
    uint32_t q[16];
    u32x4 sc, own;
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t w, const Place &p, int g, int i)
    {
#pragma unroll
        for (int k = 4 * i; k < 4 * i + 4; ++k) q[k] = load4(w, p.v4, p.R * (272 * g + 16 * k));
    }
    __device__ __forceinline__ void scales(__amdgpu_buffer_rsrc_t w, const Place &p, int g)
    {
        sc = load16b(w, p.v16, p.R * (272 * g + 256));
    }
    __device__ __forceinline__ void begin() { own = sc; }
    static constexpr int done(int s) { return s % 4 == 3 ? s / 4 : -1; }
    __device__ __forceinline__ void step(int s, float (&v)[4]) const
    {
        const float t = f16_to_f32((own[s >> 2] >> (16 * ((s >> 1) & 1))) & 0xFFFFu);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (float)(int8_t)(q[s] >> (8 * j)) * t;
    }
};

// One wavefront's x of a stage (32 columns) in LDS: token t's 128 bytes at 128
// t, 16-byte chunk c at place c ^ (t / 2 % 8), so that the sixteen tokens of an
// operand read meet every bank once.
constexpr int kStages = 8;   // per group
// Buffers of a wavefront: x is requested kBuffers - 1 stages ahead.
template <int COPIES> constexpr int kBuffers = COPIES <= 4 ? 4 : COPIES <= 6 ? 3 : 2;
// Packed loads of stage i (0..7), which follow its copies.
template <unsigned T> constexpr int weight_loads(int i)
{
    return (i == 0 ? Packed<T>::kScaleLoads : 0) + (Packed<T>::done(2 * i) >= 0 ? Packed<T>::kQuarterLoads : 0) +
           (Packed<T>::done(2 * i + 1) >= 0 ? Packed<T>::kQuarterLoads : 0);
}
// Vector memory operations younger than the copies that stage i + 1 reads, at
// the end of stage i: the copies requested since, and the packed loads of the
// stages from the one that requested them on.
template <unsigned T, int COPIES> constexpr int younger(int i)
{
    int n = COPIES * (kBuffers<COPIES> - 2);
    for (int k = 0; k < kBuffers<COPIES> - 1; ++k) n += weight_loads<T>((i - k + kStages) % kStages);
    return n;
}

// Copies of a stage's tokens into LDS, eight tokens each: voff is this lane's
// chunk of its token (tokens past n repeat the last one: nobody stores them).
template <int COPIES, int EXTRA>
__device__ __forceinline__ void copy_x(lds_u8 *buf, __amdgpu_buffer_rsrc_t xb, const int *voff, int soff)
{
#pragma unroll
    for (int c = 0; c < COPIES; ++c)
        if (c + 1 < COPIES || EXTRA == 0 || (int)(threadIdx.x & 63) < 8 * EXTRA)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xb, (__attribute__((address_space(3))) void *)(buf + 1024 * c), 16,
                                                 voff[c], soff, 0, 0);
}

template <int TILES, int EXTRA>
struct Sums {
    f32x4 tile[TILES];
    float more[EXTRA ? EXTRA : 1];
};

// Stage I of a group: the x of a later stage (column offset soff) requested
// into nbuf, this one's products from buf, packed weights of group `next` requested as theirs are
// done with. Restrict pointers: the compiler sees that the copies do not touch
// what is read.
template <unsigned T, int TILES, int EXTRA, int I>
__device__ __forceinline__ void stage(Sums<TILES, EXTRA> &part, Packed<T> &pk, const lds_u8 *__restrict__ buf,
    lds_u8 *__restrict__ nbuf, const Place &at, __amdgpu_buffer_rsrc_t wb, __amdgpu_buffer_rsrc_t xb,
    const int *voff, int soff, int next, int lane_at)
{
    constexpr int kCopies = (16 * TILES + EXTRA + 7) / 8;
    copy_x<kCopies, EXTRA>(nbuf, xb, voff, soff);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (I == 0) pk.scales(wb, at, next);
    __builtin_amdgcn_sched_barrier(0);
    const int kq = (int)((threadIdx.x >> 4) & 3);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int s = 2 * I + h;
        f32x4 px[TILES], pe[EXTRA ? EXTRA : 1];
#pragma unroll
        for (int t = 0; t < TILES; ++t)
            px[t] = *(const __attribute__((address_space(3))) f32x4 *)(buf + 2048 * t + (lane_at ^ (64 * h)));
#pragma unroll
        for (int e = 0; e < EXTRA; ++e)
            pe[e] = *(const __attribute__((address_space(3))) f32x4 *)(buf + 128 * (16 * TILES + e) +
                                                                        16 * ((4 * h + kq) ^ (e >> 1)));
        float v[4];
        pk.step(s, v);
        if (Packed<T>::done(s) >= 0) pk.load(wb, at, next, Packed<T>::done(s));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                part.tile[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(px[t][j], v[j], part.tile[t], 0, 0, 0);
#pragma unroll
            for (int e = 0; e < EXTRA; ++e) part.more[e] = __builtin_fmaf(pe[e][j], v[j], part.more[e]);
        }
        // Holds this step's sums (and so their operands) to this step.
#pragma unroll
        for (int e = 0; e < EXTRA; ++e) asm volatile("" : "+v"(part.more[e]));
    }
    __builtin_amdgcn_sched_barrier(0);
    wait_loads<younger<T, kCopies>(I)>();   // the next stage's copies have landed
}

// TILES whole tiles of 16 tokens and EXTRA tokens after them. cols in whole
// 256-column groups.
template <unsigned T, int TILES, int EXTRA>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2))) void rows_tokens(
    const uint8_t *w, const float *x, float *__restrict__ y, int rows, int cols, int n)
{
    constexpr int kCopies = (16 * TILES + EXTRA + 7) / 8, kBuf = 1024 * kCopies, kBufs = kBuffers<kCopies>,
                  kAcc = 4 * TILES + EXTRA;
    static_assert(kAcc * 64 * 4 <= kBufs * kBuf, "the shares reuse the x buffers");
    __shared__ __align__(16) uint8_t lds[kWaves * kBufs * kBuf];
    const int lane = threadIdx.x & 63, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = kRows * blockIdx.x, tile = row0 / kTileRows, last = rows - kTileRows * tile;
    const size_t row_bytes = tiled_row_bytes<T>(cols);
    Place at;
    at.R = last < kTileRows ? last : kTileRows;
    at.groups = cols / kGroupCols;
    int r = row0 % kTileRows + (lane & 15);
    r = r < at.R ? r : at.R - 1;
    at.v16 = (int)(kTileRows * tile * row_bytes) + 16 * r;
    at.v4 = at.v16 + 4 * kq;
    at.vd = at.v16 - 14 * r;
    const __amdgpu_buffer_rsrc_t wb = buffer_of(w, (size_t)rows * row_bytes), xb = buffer_of(x, (size_t)n * cols * 4);
    int voff[kCopies];
#pragma unroll
    for (int c = 0; c < kCopies; ++c) {
        const int t = 8 * c + (lane >> 3);
        voff[c] = 4 * cols * (t < n ? t : n - 1) + 16 * ((lane & 7) ^ ((t >> 1) & 7));
    }
    const int lane_at = 128 * (lane & 15) + 16 * (kq ^ ((lane >> 1) & 7));
    lds_u8 *const bufs = (lds_u8 *)lds + kBufs * kBuf * wave;

    const int ns = wave < at.groups ? (at.groups - wave + kWaves - 1) / kWaves : 0;
    // Past the wavefront's last group the loads repeat it.
    auto group_of = [&](int k) { return wave + kWaves * (k < ns ? k : ns - 1); };
    Sums<TILES, EXTRA> acc = {};
    if (ns > 0) {
        Packed<T> pk;
#pragma unroll
        for (int i = 0; i < kBufs - 1; ++i) copy_x<kCopies, EXTRA>(bufs + kBuf * i, xb, voff, 1024 * wave + 128 * i);
        pk.scales(wb, at, wave);
#pragma unroll
        for (int i = 0; i < 4; ++i) pk.load(wb, at, wave, i);
        wait_loads<0>();
        int from = 0, to = kBuf * (kBufs - 1);   // the buffers read and filled
        for (int k = 0; k < ns; ++k) {
            const int g = group_of(k), next = group_of(k + 1);
            pk.begin();
            Sums<TILES, EXTRA> part = {};
            auto run = [&](auto I) {
                constexpr int i = decltype(I)::value, ahead = i + kBufs - 1;
                stage<T, TILES, EXTRA, i>(part, pk, bufs + from, bufs + to, at, wb, xb, voff,
                                          1024 * (ahead < kStages ? g : next) + 128 * (ahead % kStages), next, lane_at);
                to = from;
                from = from + kBuf < kBufs * kBuf ? from + kBuf : 0;
            };
            run(std::integral_constant<int, 0>{});
            run(std::integral_constant<int, 1>{});
            run(std::integral_constant<int, 2>{});
            run(std::integral_constant<int, 3>{});
            run(std::integral_constant<int, 4>{});
            run(std::integral_constant<int, 5>{});
            run(std::integral_constant<int, 6>{});
            run(std::integral_constant<int, 7>{});
#pragma unroll
            for (int t = 0; t < TILES; ++t) acc.tile[t] += part.tile[t];
#pragma unroll
            for (int e = 0; e < EXTRA; ++e) acc.more[e] += part.more[e];
        }
        // Copies requested ahead are still in flight into these buffers, which
        // past the barrier hold other wavefronts' sums.
        wait_loads<0>();
    }
    __syncthreads();
    float *const red = (float *)lds;   // [wave][share][lane]
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[(kAcc * wave + 4 * t + i) * 64 + lane] = acc.tile[t][i];
#pragma unroll
    for (int e = 0; e < EXTRA; ++e) red[(kAcc * wave + 4 * TILES + e) * 64 + lane] = acc.more[e];
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * (16 * TILES + EXTRA); i += 64 * kWaves) {
        const int token = i >> 4, row = row0 + (i & 15);
        float s = 0.f;
        if (token < 16 * TILES) {
            const int slot = 4 * (token >> 4) + (token & 3), l = 16 * ((token >> 2) & 3) + (i & 15);
#pragma unroll
            for (int q = 0; q < kWaves; ++q) s += red[(kAcc * q + slot) * 64 + l];
        } else {
            // An extra token's lanes of a row hold a quarter of the columns each.
#pragma unroll
            for (int q = 0; q < kWaves; ++q) {
                const float *p = red + (kAcc * q + 4 * TILES + token - 16 * TILES) * 64 + (i & 15);
                s += (p[0] + p[16]) + (p[32] + p[48]);
            }
        }
        if (token < n && row < rows) y[(size_t)token * rows + row] = s;
    }
}

template <unsigned T, int TILES, int EXTRA>
hipError_t launch(const uint8_t *w, const float *x, float *y, int rows, int cols, int n, hipStream_t s)
{
    hipLaunchKernelGGL((rows_tokens<T, TILES, EXTRA>), dim3((unsigned)((rows + kRows - 1) / kRows)), dim3(64 * kWaves), 0,
                       s, w, x, y, rows, cols, n);
    return hipGetLastError();
}

template <unsigned T>
hipError_t launch_type(const uint8_t *w, const float *x, float *y, int rows, int cols, int n, hipStream_t s)
{
    if (n <= 16) return launch<T, 1, 0>(w, x, y, rows, cols, n, s);
    if (n <= 17) return launch<T, 1, 1>(w, x, y, rows, cols, n, s);
    if (n <= 20) return launch<T, 1, 4>(w, x, y, rows, cols, n, s);
    if (n <= 32) return launch<T, 2, 0>(w, x, y, rows, cols, n, s);
    if (n <= 33) return launch<T, 2, 1>(w, x, y, rows, cols, n, s);
    if (n <= 36) return launch<T, 2, 4>(w, x, y, rows, cols, n, s);
    if (n <= 48) return launch<T, 3, 0>(w, x, y, rows, cols, n, s);
    if (n <= 49) return launch<T, 3, 1>(w, x, y, rows, cols, n, s);
    if (n <= 52) return launch<T, 3, 4>(w, x, y, rows, cols, n, s);
    return launch<T, 4, 0>(w, x, y, rows, cols, n, s);
}

}  // namespace

// Up to 4096 rows: a workgroup per CU. Beyond, where a CU reads x several times
// over, 8-token launches win (Q4_K 14336 x 4096, 16 tokens: 20 us, 30 here; 6144
// x 4096: 13.8, 15.9; Q8_0 5120 x 4096: 13.6, 18.4) but on short rows, and on
// those of up to 2048 columns from 25 tokens on, a launch more. us, 8-token
// launches / here, 5632 rows by 9, 16, 24 and 28 tokens:
//   Q4_K  1024 columns   7.0/6.0   7.7/6.1  11.5/10.3  14.7/10.3
//         1536           7.4/8.8   8.9/9.0  13.2/14.8  16.8/14.8
//         2048           7.9/9.4   9.4/9.6  14.1/15.8  17.7/15.8
//   Q4_0  1024           6.5/5.9   7.1/6.0  10.7/10.3  13.6/10.3
//   Q8_0   512           7.0/5.7   7.1/5.7  10.5/9.6   13.4/9.5
//         1024 (6144)    6.4/7.1   7.3/7.1  10.9/11.2  14.0/11.2
// Q6_K, whose 8-token launches decode longest, from 17 tokens on (8192 x 14336: 16
// tokens 55, 54 here; 33 tokens 133, 104; 6144 x 8192: 33 tokens 77, 57), but for
// three whole launches of the tallest (8192 x 14336, 24 tokens 81.5, 86; 8192 x
// 4608 32.9, 33.9; 6144 x 8192 51.5, 49.1). Nine tokens of wide rows are one
// launch of eight and a matvec up to 4096 rows (Q4_K 4096 x 14336: 25.3, 26.4 here).
bool rows_tokens_supported(unsigned type, int rows, int cols, int batch)
{
    if (type != Q4_K && type != Q4_0 && type != Q8_0 && type != Q6_K) return false;
    if (rows <= 0 || cols <= 0 || cols % kGroupCols || batch <= 8 || batch > kRowsTokens) return false;
    // x within a 32-bit buffer range.
    if ((size_t)kRowsTokens * cols * 4 > (size_t)INT32_MAX) return false;
    if (type == Q6_K)
        return rows <= 4096 || (rows <= 8192 && batch > 16 && (rows <= 6144 || batch <= 20 || batch > 24));
    if (rows <= 4096) return batch > 9 || cols <= 4096;
    return rows <= 6144 && cols <= (batch > 24 ? 2048 : type == Q8_0 ? 512 : 1024);
}

hipError_t launch_rows_tokens(unsigned type, const uint8_t *w, const float *x, float *y, int rows, int cols,
    int batch, hipStream_t s)
{
    if (!rows_tokens_supported(type, rows, cols, batch)) return hipErrorInvalidValue;
    if (type == Q4_K) return launch_type<Q4_K>(w, x, y, rows, cols, batch, s);
    if (type == Q4_0) return launch_type<Q4_0>(w, x, y, rows, cols, batch, s);
    if (type == Q6_K) return launch_type<Q6_K>(w, x, y, rows, cols, batch, s);
    return launch_type<Q8_0>(w, x, y, rows, cols, batch, s);
}

}  // namespace fy
