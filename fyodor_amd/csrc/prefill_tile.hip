// Prefill GEMM Y[m][row] = sum_k W[row][k] X[m][k] for batches above 8 of
// whole 256-column groups: Q4_K, Q8_0, Q4_0 (prefill_f16) and Q6_K
// (prefill_mfma), on v_mfma_f32_32x32x16_f16 with the activation pieces of
// pieces.h.
//
// Numbers. Q4_K (sc q), Q8_0 and Q4_0 weights are exact fp16 integers, so a
// block dot is sum w (hi + lo) with fp32 accumulation error only; d and dmin
// (or the fp16 block scale) are applied in fp32. Q6_K's sc (q - 32) reaches
// 4096, one bit past fp16's integers: w1 = fp16(sc (q - 32)) and the exact
// remainder w2 (at most 1 in magnitude, non-zero only above 2048) enter as
// hi w1 + lo w1 + hi w2; the dropped lo w2 is below 2^-23 |w x|. Error against
// 64 bits at 4096 x 14336: 1.9e-7 (three int8 digits per activation: 3.6e-7).
//
// Bound. Every operand that a wavefront reads from LDS feeds kR MFMAs (its row
// tiles). With one row tile per wavefront the LDS reads alone need all 128
// bytes per cycle of the CU at the matrix cores' full rate; two row tiles
// halve that, and the weights are still unpacked once per 64 tokens. Large
// batches run against the card's power: Q4_K 14336 x 4096 x 2048 keeps the
// matrix cores busy 65 % of the cycles at a clock that has fallen to 1.67 GHz
// (1107 issued TFLOP/s; a library fp16 product reaches 1495).
//
// Wide workgroups: four wavefronts, 256 rows x 64 tokens (Q8_0 and Q4_0 also x
// 32, where that evens the CUs out). The accumulators (128 registers with a
// K-quant's running group) leave two wavefronts per SIMD: two workgroups per CU,
// each other's cover at the barriers. K advances 128 columns per step; copies
// for the next step go out at a step's start. Narrow workgroups split the
// columns four ways (below).
//
// The pieces go global -> LDS directly (buffer_load ... lds). 16-byte chunk c
// of token t lies at place c ^ (t % 16) of the token's 256 bytes (the
// permutation is in the copies' source addresses), so the lanes of one read
// hit distinct banks. In memory the pieces are tiled: a copy reads 1 KiB in
// one run. Weights are requested two 64-column units ahead and waited for by
// count, never for all loads.
//
// Blocks are renumbered so that the token blocks of one row block run on one
// XCD (the dispatcher deals block b to XCD b % 8) and its weights enter one L2.
#include "blockdot.h"
#include "kernels.h"
#include "pieces.h"

namespace fy {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) uint8_t lds_u8;

constexpr int kR = 2;              // row tiles per wavefront
constexpr int kSumTile = 1024;     // Q4_K block sums of one group: 32 tokens x 2 halves x 16 bytes

template <unsigned T> constexpr bool kSuper = T == Q4_K || T == Q6_K;   // scales per 256 columns (else per 32)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void *p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t r, int voff, int soff)
{
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// A 64-column unit of one row tile (formats.h: unit p of a 256-column group;
// Q8_0: blocks 2p, 2p + 1), and the group's scales.
template <unsigned T> struct Unit { u32x4 a; };
template <> struct Unit<Q6_K> { u32x4 a, b; };   // ql, qh
template <> struct Unit<Q8_0> { u32x4 a, b; };   // blocks 2p, 2p + 1
template <unsigned T> struct Scales { u32x4 s; };
template <> struct Scales<Q6_K> { u32x4 s; uint32_t d; };

// One row tile of the wavefront: R rows, lane l holding row l % 32 (clamped)
// and the column half l / 32.
struct Tile {
    __amdgpu_buffer_rsrc_t rs;
    int R, voff, voff_row;   // 16 R h + 16 r, 16 r
};

template <unsigned T> constexpr int kGroupRow = T == Q4_K ? 144 : T == Q6_K ? 208 : T == Q8_0 ? 272 : 144;

template <unsigned T>
__device__ __forceinline__ void load_unit(Unit<T> &u, const Tile &t, int g, int p)
{
    const int b = kGroupRow<T> * t.R * g;
    if constexpr (T == Q6_K) {
        u.a = load16(t.rs, t.voff, b + 48 * t.R * p);
        u.b = load16(t.rs, t.voff_row, b + 48 * t.R * p + 32 * t.R);
    } else if constexpr (T == Q8_0) {
        u.a = load16(t.rs, t.voff, b + 64 * t.R * p);
        u.b = load16(t.rs, t.voff, b + 64 * t.R * p + 32 * t.R);
    } else {
        u.a = load16(t.rs, t.voff, b + 32 * t.R * p);
    }
}

template <unsigned T>
__device__ __forceinline__ void load_scales(Scales<T> &s, const Tile &t, int g, int groups)
{
    const int b = kGroupRow<T> * t.R * g;
    if constexpr (T == Q6_K) {
        s.s = load16(t.rs, t.voff_row, b + 192 * t.R);
        s.d = __builtin_amdgcn_raw_buffer_load_b16(t.rs, t.voff_row >> 3, 208 * t.R * groups + 2 * t.R * g, 0);
    } else {
        s.s = load16(t.rs, t.voff_row, b + (T == Q8_0 ? 256 : 128) * t.R);
    }
}

__device__ __forceinline__ uint32_t as_u32(h2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
// fp16 pairs 1024 + (byte 0, byte 2) and 1024 + (byte 1, byte 3) of v.
__device__ __forceinline__ h2 pair02(uint32_t v) { return as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04020400u)); }
__device__ __forceinline__ h2 pair13(uint32_t v) { return as_h2(__builtin_amdgcn_perm(0x64646464u, v, 0x04030401u)); }
__device__ __forceinline__ h2 both(float f)
{
    const _Float16 v = (_Float16)f;
    return (h2){v, v};
}

// B operand `o` of a unit (o = 2 n + kappa: its n-th 32-column block — for
// Q6_K blocks 2 n + h of the unit's 128 columns — and 8-column slice kappa),
// in the pieces' column order; B[1] is Q6_K's remainder. sw: the unit's word
// of the group's scales.
template <unsigned T>
__device__ __forceinline__ void operand(const Unit<T> &u, uint32_t sw, int o, int h, h8 (&B)[T == Q6_K ? 2 : 1])
{
    const int n = o >> 1, kappa = o & 1;
    uint32_t v[4], r[4] = {};
    if constexpr (T == Q4_K) {
        const float sc = (float)((sw >> (12 * n)) & 63u);
        const h2 sc2 = both(sc), nsc2 = both(-1024.f * sc);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t nib = (n ? u.a[2 * kappa + i] >> 4 : u.a[2 * kappa + i]) & 0x0F0F0F0Fu;
            v[2 * i] = as_u32(__builtin_elementwise_fma(pair02(nib), sc2, nsc2));
            v[2 * i + 1] = as_u32(__builtin_elementwise_fma(pair13(nib), sc2, nsc2));
        }
    } else if constexpr (T == Q6_K) {
        const h2 sc2 = both((float)(int8_t)(sw >> (16 * n + 8 * h)));
        const h2 off = {(_Float16)1056, (_Float16)1056};   // 1024 + 32
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t lo = u.a[2 * kappa + i] >> (4 * n), hi = u.b[2 * kappa + i] >> (4 * n + 2 * h);
            const uint32_t q = (lo & 0x0F0F0F0Fu) | ((hi & 0x03030303u) << 4);
            const h2 a = pair02(q) - off, b = pair13(q) - off;
            const h2 wa = a * sc2, wb = b * sc2;
            v[2 * i] = as_u32(wa);
            v[2 * i + 1] = as_u32(wb);
            r[2 * i] = as_u32(__builtin_elementwise_fma(a, sc2, -wa));
            r[2 * i + 1] = as_u32(__builtin_elementwise_fma(b, sc2, -wb));
        }
        B[1] = __builtin_bit_cast(h8, (u32x4){r[0], r[1], r[2], r[3]});
    } else if constexpr (T == Q8_0) {
        const h2 off = {(_Float16)1152, (_Float16)1152};   // 1024 + 128
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t q = (n ? u.b[2 * kappa + i] : u.a[2 * kappa + i]) ^ 0x80808080u;
            v[2 * i] = as_u32(pair02(q) - off);
            v[2 * i + 1] = as_u32(pair13(q) - off);
        }
    } else {
        const h2 off = {(_Float16)1032, (_Float16)1032};   // 1024 + 8
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t nib = (u.a[2 * kappa + i] >> (4 * n)) & 0x0F0F0F0Fu;
            v[2 * i] = as_u32(pair02(nib) - off);
            v[2 * i + 1] = as_u32(pair13(nib) - off);
        }
    }
    B[0] = __builtin_bit_cast(h8, (u32x4){v[0], v[1], v[2], v[3]});
}

// What a wavefront's copies need: the pieces' planes, the workgroup's tokens,
// and the wavefront's part of the four.
struct Copies {
    Pieces p;
    int cols, np, m0, part;
    int voff;   // this lane's bytes within the 1 KiB of one copy
};

// The copies of one step: COLS columns of both pieces of 32 TT tokens. One
// copy takes 1 KiB, four tokens of a 32-token x 128-column block of the tiled
// pieces; lane l's 16 bytes are chunk (l % 16) ^ (token % 16) of the copy's
// token l / 16, so that in LDS chunk c of token t lies at place c ^ (t % 16).
// Of the W wavefronts (4 or 8) each takes every W-th copy: token % 16 is
// 4 (part % 4) + l / 16 in all of them.
template <int W, int TT, int COLS> constexpr int kStepCopies = 16 * TT * (COLS / 128) / W;   // per wavefront

__device__ __forceinline__ int copy_voff(int part)
{
    const int lane = threadIdx.x & 63, row = lane >> 4;
    return 256 * row + 16 * ((lane & 15) ^ (4 * (part & 3) + row));
}

// This wavefront's copies of step s (columns COLS s ..) into buf: 8 KiB per
// block, [128-column half][piece][token tile]. Tiles past the np padded
// tokens read zeros.
template <int W, int TT, int COLS>
__device__ __forceinline__ void copy_step(lds_u8 *buf, const Copies &c, int s)
{
    constexpr int kHalves = COLS / 128;
#pragma unroll
    for (int b = 0; b < kHalves * 2 * TT; ++b) {
        const int half = b / (2 * TT), piece = b / TT % 2, m = c.m0 + 32 * (b % TT);
        const __amdgpu_buffer_rsrc_t rs =
            rsrc_of(tiled_block(piece ? c.p.lo : c.p.hi, c.cols, m, kHalves * s + half), m < c.np ? 8192u : 0u);
#pragma unroll
        for (int k = 0; k < 8 / W; ++k)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rs, (__attribute__((address_space(3))) void *)(buf + 8192 * b + 1024 * (W * k + c.part)), 16, c.voff,
                1024 * (W * k + c.part), 0, 0);
    }
}

// Q4_K: group g's block sums of token tile part % TT.
template <int TT>
__device__ __forceinline__ void copy_sums(lds_u8 *sums, const Copies &c, int g)
{
    const int lane = threadIdx.x & 63, t = c.part % TT, m = c.m0 + 32 * t;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_of(tiled_sums(c.p.bsum, c.cols, m, g), m < c.np ? 1024u : 0u),
                                             (__attribute__((address_space(3))) void *)(sums + kSumTile * t), 16,
                                             16 * lane, 0, 0, 0);
}

// The accumulators of a wavefront, and its row tiles.
template <unsigned T, int TT>
struct State {
    f32x16 acc[kR][TT];
    f32x16 C[kSuper<T> ? kR : 1][kSuper<T> ? TT : 1];   // the running 256-column group
    Tile tile[kR];
};

// Vector memory operations one wavefront issues for a unit's weights and a
// group's scales.
template <unsigned T> constexpr int kUnitLoads = kR * (T == Q6_K || T == Q8_0 ? 2 : 1);
template <unsigned T> constexpr int kScaleLoads = kR * (T == Q6_K ? 2 : 1);

// Keeps the vector memory operations around it in order (the waits count
// them); the weights are not a restrict pointer for the same reason.
__device__ __forceinline__ void in_order()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// Waits until at most `vm` vector memory operations of this wavefront are in
// flight (they complete in order) and its LDS reads are done.
template <int VM>
__device__ __forceinline__ void wait_loads()
{
    static_assert(VM < 64, "vmcnt field");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4));
    asm volatile("" ::: "memory");
}

template <int VM>
__device__ __forceinline__ void meet()
{
    wait_loads<VM>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <unsigned T, int TT>
__device__ __forceinline__ void request_unit(Unit<T> (&u)[kR], const State<T, TT> &st, int g, int p)
{
    in_order();
#pragma unroll
    for (int r = 0; r < kR; ++r) load_unit<T>(u[r], st.tile[r], g, p);
    in_order();
}

template <unsigned T, int TT>
__device__ __forceinline__ void request_scales(Scales<T> (&s)[kR], const State<T, TT> &st, int g, int groups)
{
    in_order();
#pragma unroll
    for (int r = 0; r < kR; ++r) load_scales<T>(s[r], st.tile[r], g, groups);
    in_order();
}

// One unit (64 columns of each row; its pieces at buf + a_off): C += W X, or
// for block scales acc += d W X. FRESH starts the group's C. sw: the unit's
// word of each row tile's scales.
template <unsigned T, int TT, bool FRESH>
__device__ __forceinline__ void unit_step(State<T, TT> &st, const Unit<T> (&u)[kR], const uint32_t (&sw)[kR],
    const lds_u8 *buf, int a_off, int h)
{
    constexpr int kB = T == Q6_K ? 2 : 1;
    // Operands of slice o + 1 are read and unpacked among slice o's MFMAs.
    h8 a[2][TT][2], b[2][kR][kB];
    auto fetch = [&](int o, h8 (&x)[TT][2], h8 (&w)[kR][kB]) {
        // Chunk within the unit: 32-column block (Q6_K: 2 n + h) and slice;
        // the lane half and the unit are in a_off.
        const int at = (T == Q6_K ? 128 : 64) * (o >> 1) + 16 * (o & 1);
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int pc = 0; pc < 2; ++pc)
                x[t][pc] = *(const h8 *)(buf + (a_off ^ at) + 8192 * (TT * pc + t));
#pragma unroll
        for (int r = 0; r < kR; ++r) operand<T>(u[r], sw[r], o, h, w[r]);
    };
    f32x16 blk[kSuper<T> ? 1 : kR][kSuper<T> ? 1 : TT];
    fetch(0, a[0], b[0]);
#pragma unroll
    for (int o = 0; o < 4; ++o) {
        if (o < 3) fetch(o + 1, a[(o + 1) & 1], b[(o + 1) & 1]);
        auto mfma = [&](int pc, int k) {
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int r = 0; r < kR; ++r) {
                    f32x16 &c = kSuper<T> ? st.C[r % (kSuper<T> ? kR : 1)][t % (kSuper<T> ? TT : 1)]
                                          : blk[r % (kSuper<T> ? 1 : kR)][t % (kSuper<T> ? 1 : TT)];
                    const bool fresh = k == 0 && pc == 0 && (kSuper<T> ? FRESH && o == 0 : (o & 1) == 0);
                    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[o & 1][t][pc], b[o & 1][r][k], fresh ? (f32x16){} : c,
                                                               0, 0, 0);
                }
        };
        mfma(0, 0);
        mfma(1, 0);
        if constexpr (T == Q6_K) mfma(0, 1);
        if constexpr (!kSuper<T>) {
            if (o & 1) {
                // The block's scale: two fp16 per word.
#pragma unroll
                for (int r = 0; r < kR; ++r) {
                    const float d = f16_to_f32((sw[r] >> (16 * (o >> 1))) & 0xFFFFu);
#pragma unroll
                    for (int t = 0; t < TT; ++t)
#pragma unroll
                        for (int i = 0; i < 16; ++i) st.acc[r][t][i] = __builtin_fmaf(d, blk[r][t][i], st.acc[r][t][i]);
                }
            }
        }
        constexpr int kMfma = kR * TT * (T == Q6_K ? 3 : 2);
#pragma unroll
        for (int q = 0; q < kMfma; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, T == Q6_K ? 5 : kSuper<T> ? 4 : 6, 0);   // VALU
            if (q < 2 * TT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
        }
    }
}

// The end of a K-quant's group: acc += d C, and for Q4_K the minimums on one more MFMA
// per tile: M = sum_j m_j 2^-5 (sum of x s over block j), exact products (lane
// half h of A holds piece h of the eight sums), acc -= 32 dmin M.
template <unsigned T, int TT>
__device__ __forceinline__ void close_group(State<T, TT> &st, const Scales<T> (&sc)[kR], const lds_u8 *sums, int lane)
{
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        if constexpr (T == Q4_K) {
            const u32x4 s = sc[r].s;
            const uint32_t dd = (s.x >> 24) | ((s.y >> 24) << 8) | ((s.z >> 24) << 16) | ((s.w >> 24) << 24);
            const float d = f16_to_f32(dd & 0xFFFFu), ndmin = -32.f * f16_to_f32(dd >> 16);
            h8 bm;
#pragma unroll
            for (int j = 0; j < 8; ++j) bm[j] = (_Float16)(int)((s[j >> 1] >> (12 * (j & 1) + 6)) & 63u);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const h8 ys = *(const h8 *)(sums + kSumTile * t + 16 * lane);
                const f32x16 M = __builtin_amdgcn_mfma_f32_32x32x16_f16(ys, bm, (f32x16){}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    st.acc[r][t][i] = __builtin_fmaf(d, st.C[r][t][i], __builtin_fmaf(ndmin, M[i], st.acc[r][t][i]));
            }
        } else if constexpr (T == Q6_K) {
            const float d = f16_to_f32(sc[r].d);
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int i = 0; i < 16; ++i) st.acc[r][t][i] = __builtin_fmaf(d, st.C[r][t][i], st.acc[r][t][i]);
        }
    }
}

// ---- wide: four wavefronts of distinct rows, two step buffers --------------

template <unsigned T, int TT>
struct Wide : State<T, TT> {
    Unit<T> unit[4][kR];   // by unit of the group: the current one, the next, and the one after in flight
    Scales<T> scales[kR], next[kR];
};

// Columns 128 HALF .. of group g from buf, the next step's pieces into nbuf.
// The two buffers are restrict pointers so that the compiler sees that the
// LDS reads do not depend on the copies in flight.
template <unsigned T, int TT, int HALF>
__device__ __forceinline__ void wide_step(Wide<T, TT> &st, const lds_u8 *__restrict__ buf, lds_u8 *__restrict__ nbuf,
    lds_u8 *__restrict__ sums, const Copies &c, int a_off, int g, int groups)
{
    constexpr int kCols = 128, P = 2 * HALF;
    constexpr int kSecond = T == Q6_K ? 32 : 128;   // the second unit's first chunk
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const int gn = g + 1 < groups ? g + 1 : g;   // past the end the last group again
    const int next = HALF == 0 ? 2 * g + 1 : 2 * gn;
    request_unit<T, TT>(st.unit[(P + 2) & 3], st, HALF ? gn : g, (P + 2) & 3);
    if constexpr (HALF == 1) request_scales<T, TT>(st.next, st, gn, groups);
    copy_step<4, TT, kCols>(nbuf, c, next);
    // The group's block sums, read at the group's end past the next barrier.
    if constexpr (T == Q4_K && HALF == 0) copy_sums<TT>(sums, c, g);
    in_order();
    uint32_t sw[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) sw[r] = st.scales[r].s[P];
    unit_step<T, TT, HALF == 0>(st, st.unit[P], sw, buf, a_off, h);
    // The second unit's weights were requested before everything above.
    wait_loads<kUnitLoads<T> + (HALF == 1 ? kScaleLoads<T> : 0) + kStepCopies<4, TT, kCols> +
               (T == Q4_K && HALF == 0 ? 1 : 0)>();
    request_unit<T, TT>(st.unit[(P + 3) & 3], st, HALF ? gn : g, (P + 3) & 3);
#pragma unroll
    for (int r = 0; r < kR; ++r) sw[r] = st.scales[r].s[P + 1];
    unit_step<T, TT, false>(st, st.unit[P + 1], sw, buf, a_off ^ kSecond, h);
    if constexpr (HALF == 1) close_group<T, TT>(st, st.scales, sums, lane);
    // All but the last request: the copies have landed, past the barrier
    // every wavefront's.
    meet<kUnitLoads<T>>();
    if constexpr (HALF == 1) {
#pragma unroll
        for (int r = 0; r < kR; ++r) st.scales[r] = st.next[r];
    }
}

// ---- narrow: four wavefronts share a row block's columns -------------------
//
// Where wide workgroups would leave CUs idle: 64 WR rows per workgroup of 4 WR
// wavefronts. A step covers a whole 256-column group, wavefront (wr, ks) takes
// its unit ks. NBUF step buffers: copies go out NBUF - 1 steps ahead, weights
// three steps ahead (two with two buffers).

// The scales a wavefront needs of a group: its unit's word (and Q6_K's d).
struct Share { uint32_t w, d; };
template <unsigned T> constexpr int kShareLoads = kR * (T == Q6_K ? 2 : 1);

template <unsigned T, int TT>
struct Narrow : State<T, TT> {
    Unit<T> unit[4][kR];     // by step % 4
    Share scales[4][kR];
};

template <unsigned T, int TT>
__device__ __forceinline__ void request_share(Unit<T> (&u)[kR], Share (&s)[kR], const State<T, TT> &st, int g, int ks,
    int groups)
{
    in_order();
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const Tile &t = st.tile[r];
        const int b = kGroupRow<T> * t.R * g;
        s[r].w = __builtin_amdgcn_raw_buffer_load_b32(t.rs, t.voff_row + 4 * ks,
                                                      b + (T == Q6_K ? 192 : T == Q8_0 ? 256 : 128) * t.R, 0);
        if constexpr (T == Q6_K)
            s[r].d = __builtin_amdgcn_raw_buffer_load_b16(t.rs, t.voff_row >> 3, 208 * t.R * groups + 2 * t.R * g, 0);
    }
#pragma unroll
    for (int r = 0; r < kR; ++r) load_unit<T>(u[r], st.tile[r], g, ks);
    in_order();
}

// Group `at`, at % 4 == I, from buf; nbuf: the buffer of group at + NBUF - 1.
template <unsigned T, int TT, int WR, int NBUF, int I>
__device__ __forceinline__ void narrow_step(Narrow<T, TT> &st, const lds_u8 *__restrict__ buf,
    lds_u8 *__restrict__ nbuf, const Copies &c, int a_off, int at, int groups, int ks)
{
    constexpr int kCopied = kStepCopies<4 * WR, TT, 256>;
    constexpr int kAsked = kUnitLoads<T> + kShareLoads<T>, kAhead = NBUF == 2 ? 2 : 3;
    const int lane = threadIdx.x & 63, h = lane >> 5;
    // Past the end the last group again.
    const int copied = at + NBUF - 1 < groups ? at + NBUF - 1 : groups - 1;
    const int asked = at + kAhead < groups ? at + kAhead : groups - 1;
    copy_step<4 * WR, TT, 256>(nbuf, c, copied);
    request_share<T, TT>(st.unit[(I + kAhead) & 3], st.scales[(I + kAhead) & 3], st, asked, ks, groups);
    uint32_t sw[kR];
    Scales<T> sc[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        sw[r] = st.scales[I][r].w;
        if constexpr (T == Q6_K) sc[r].d = st.scales[I][r].d;
    }
    unit_step<T, TT, true>(st, st.unit[I], sw, buf, a_off, h);
    if constexpr (T == Q6_K) close_group<T, TT>(st, sc, nullptr, lane);
    // Two buffers: left in flight is what was asked for after the copies.
    // Four: what this step and the one before issued.
    if constexpr (NBUF == 2) meet<kAsked>();
    else meet<2 * (kCopied + kAsked)>();
}

// The rows of wavefront row group `wr` of workgroup row block bx.
template <unsigned T, int TT, int WR>
__device__ __forceinline__ void place(State<T, TT> &st, int (&tile_of)[kR], const uint8_t *w, int rows, int cols, int bx,
    int wr)
{
    const int lane = threadIdx.x & 63, tiles = (rows + kTileRows - 1) / kTileRows;
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        tile_of[r] = kR * (WR * bx + wr) + r;
        const int t = tile_of[r] < tiles ? tile_of[r] : tiles - 1;
        const int R = rows - kTileRows * t < kTileRows ? rows - kTileRows * t : kTileRows;
        const int row = (lane & 31) < R ? (lane & 31) : R - 1;
        st.tile[r].rs = rsrc_of(w + (size_t)kTileRows * t * tiled_row_bytes<T>(cols),
                                (uint32_t)((size_t)R * tiled_row_bytes<T>(cols)));
        st.tile[r].R = R;
        st.tile[r].voff_row = 16 * row;
        st.tile[r].voff = 16 * R * (lane >> 5) + 16 * row;
#pragma unroll
        for (int t2 = 0; t2 < TT; ++t2) st.acc[r][t2] = (f32x16){};
    }
}

// Consecutive work items on each XCD: one eighth of the grid each.
__device__ __forceinline__ int work_item()
{
    const int n = gridDim.x, xcd = blockIdx.x % 8, per = n / 8, extra = n % 8;
    return xcd * per + (xcd < extra ? xcd : extra) + (int)(blockIdx.x / 8);
}

template <unsigned T, int TT>
__device__ __forceinline__ void store_tile(const State<T, TT> &st, const int (&tile_of)[kR], const Pieces &p,
    float *__restrict__ y, int rows, int batch, int np, int m0)
{
    const int lane = threadIdx.x & 63, h = lane >> 5, tiles = (rows + kTileRows - 1) / kTileRows;
    // Register i of lane l holds token 8 (i / 4) + 4 (l / 32) + i % 4 of its
    // token tile, row l % 32 of its row tile. Every 1 / s is requested before
    // the first store.
    float4 inv[TT][4];
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            inv[t][q] = *(const float4 *)(p.inv + (m0 + 32 * t < np ? m0 + 32 * t : m0) + 8 * q + 4 * h);
#pragma unroll
    for (int r = 0; r < kR; ++r) {
        const int row = kTileRows * tile_of[r] + (lane & 31);
        if (tile_of[r] >= tiles || row >= rows) continue;
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int token = m0 + 32 * t + 8 * (i >> 2) + 4 * h + (i & 3);
                const float4 v = inv[t][i >> 2];
                const float scale = (i & 3) == 0 ? v.x : (i & 3) == 1 ? v.y : (i & 3) == 2 ? v.z : v.w;
                if (token < batch) y[(size_t)token * rows + row] = st.acc[r][t][i] * scale;
            }
    }
}

template <unsigned T, int TT>
__device__ __forceinline__ void wide_gemm(const uint8_t *w, const Pieces &p, float *__restrict__ y, int rows, int cols,
    int batch, int np, int token_blocks, lds_u8 *b0, lds_u8 *b1, lds_u8 *sums)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int id = work_item(), m0 = 32 * TT * (id % token_blocks), groups = cols / kGroupCols;
    Wide<T, TT> st;
    int tile_of[kR];
    place<T, TT, 4>(st, tile_of, w, rows, cols, id / token_blocks, wave);
    const Copies c{p, cols, np, m0, wave, copy_voff(wave)};
    copy_step<4, TT, 128>(b0, c, 0);
    request_unit<T, TT>(st.unit[0], st, 0, 0);
    request_unit<T, TT>(st.unit[1], st, 0, 1);
    request_scales<T, TT>(st.scales, st, 0, groups);
    meet<0>();
    // Token l % 32 of a token tile: its row, the permuted place of the lane
    // half's first chunk (the other chunks of a step are xors of it).
    const int a_off = 256 * (lane & 31) + 16 * (((T == Q6_K ? 4 : 2) * (lane >> 5)) ^ (lane & 15));
    for (int g = 0; g < groups; ++g) {
        wide_step<T, TT, 0>(st, b0, b1, sums, c, a_off, g, groups);
        wide_step<T, TT, 1>(st, b1, b0, sums, c, a_off, g, groups);
    }
    wait_loads<0>();   // the last requests
    store_tile<T, TT>(st, tile_of, p, y, rows, batch, np, m0);
}

template <unsigned T, int TT, int WR, int NBUF>
__device__ __forceinline__ void narrow_gemm(const uint8_t *w, const Pieces &p, float *__restrict__ y, int rows,
    int cols, int batch, int np, int token_blocks, lds_u8 *b0, lds_u8 *b1, lds_u8 *b2, lds_u8 *b3)
{
    constexpr int kAhead = NBUF == 2 ? 2 : 3;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave % WR, ks = wave / WR;
    const int id = work_item(), m0 = 32 * TT * (id % token_blocks), groups = cols / kGroupCols;
    Narrow<T, TT> st;
    int tile_of[kR];
    place<T, TT, WR>(st, tile_of, w, rows, cols, id / token_blocks, wr);
    const Copies c{p, cols, np, m0, wave, copy_voff(wave)};
    lds_u8 *const b[4] = {b0, b1, b2, b3};
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
        if (i && i >= groups) break;   // (Q6_K 1024 x 256 x64: 9.9 us with the last group again, 9.0)
        if (i < NBUF - 1) copy_step<4 * WR, TT, 256>(b[i], c, i);
        request_share<T, TT>(st.unit[i], st.scales[i], st, i, ks, groups);
    }
    meet<0>();
    const int base = 256 * (lane & 31) + 16 * (((T == Q6_K ? 4 : 2) * (lane >> 5)) ^ (lane & 15));
    // The wavefront's unit of the step: 64 columns of its 128-column half
    // ks / 2, for Q6_K 16-column halves ks % 2 of that half's blocks.
    const int a_off = (base ^ ((T == Q6_K ? 32 : 128) * (ks & 1))) + 2 * TT * 8192 * (ks >> 1);
#define FY_NARROW(I, CUR, NEXT)                                                           \
    narrow_step<T, TT, WR, NBUF, I>(st, CUR, NEXT, c, a_off, at + I, groups, ks);         \
    if (at + I + 1 >= groups) break
    for (int at = 0;; at += 4) {
        if constexpr (NBUF == 4) {
            FY_NARROW(0, b0, b3);
            FY_NARROW(1, b1, b0);
            FY_NARROW(2, b2, b1);
            FY_NARROW(3, b3, b2);
        } else {
            FY_NARROW(0, b0, b1);
            FY_NARROW(1, b1, b0);
            FY_NARROW(2, b0, b1);
            FY_NARROW(3, b1, b0);
        }
    }
#undef FY_NARROW
    wait_loads<0>();
    __syncthreads();   // every wavefront's copies and reads are done

    // The shares meet in LDS: wavefronts ks > 0 leave their sums in the step
    // buffers (8 TT KiB each), the first adds them in order.
    constexpr int kFloats = kR * TT * 16, kPart = kFloats * 64 * 4;
    static_assert(3 * WR * kPart <= NBUF * 32768 * TT && (NBUF == 4 || 2 * WR * kPart <= 32768 * TT), "the sums fit");
    auto part_of = [&](int k) {   // share k = 1, 2, 3
        lds_u8 *q = NBUF == 4 ? b[k - 1] : k < 3 ? b0 + (k - 1) * WR * kPart : b1;
        return (float *)(q + wr * kPart) + lane;
    };
    if (ks > 0) {
        float *part = part_of(ks);
#pragma unroll
        for (int i = 0; i < kFloats; ++i) part[64 * i] = st.acc[i / (16 * TT)][i / 16 % TT][i % 16];
    }
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int k = 1; k < 4; ++k) {
        const float *part = part_of(k);
#pragma unroll
        for (int i = 0; i < kFloats; ++i) {
            st.acc[i / (16 * TT)][i / 16 % TT][i % 16] += part[64 * i];
            if (i % 16 == 15) __builtin_amdgcn_sched_barrier(0);   // 16 reads in registers at a time
        }
    }
    store_tile<T, TT>(st, tile_of, p, y, rows, batch, np, m0);
}

// Wide: 256 rows x 32 TT tokens, 32 TT KiB of step buffers, two workgroups per CU.
// Narrow: 64 WR rows x 32 TT tokens, 128 KiB, one workgroup per CU.
template <unsigned T, int TT>
__device__ __forceinline__ void wide_kernel(const uint8_t *w, const Pieces &p, float *__restrict__ y, int rows, int cols,
    int batch, int np, int token_blocks)
{
    __shared__ __align__(16) uint8_t s0[16384 * TT], s1[16384 * TT];
    __shared__ __align__(16) uint8_t sums[T == Q4_K ? TT * kSumTile : 16];
    wide_gemm<T, TT>(w, p, y, rows, cols, batch, np, token_blocks, (lds_u8 *)s0, (lds_u8 *)s1, (lds_u8 *)sums);
}

template <unsigned T, int TT, int WR>
__device__ __forceinline__ void narrow_kernel(const uint8_t *w, const Pieces &p, float *__restrict__ y, int rows,
    int cols, int batch, int np, int token_blocks)
{
    __shared__ __align__(16) uint8_t s0[32768 * TT], s1[32768 * TT];
    if constexpr (TT == 1) {
        __shared__ __align__(16) uint8_t s2[32768], s3[32768];
        narrow_gemm<T, TT, WR, 4>(w, p, y, rows, cols, batch, np, token_blocks, (lds_u8 *)s0, (lds_u8 *)s1,
                                  (lds_u8 *)s2, (lds_u8 *)s3);
    } else {
        narrow_gemm<T, TT, WR, 2>(w, p, y, rows, cols, batch, np, token_blocks, (lds_u8 *)s0, (lds_u8 *)s1,
                                  (lds_u8 *)s0, (lds_u8 *)s1);
    }
}

// Q4_K (wide only), Q8_0 and Q4_0; prefill_mfma: Q6_K (three products per
// operand pair). WR = 0: wide.
template <unsigned T, int TT, int WR>
__global__ __launch_bounds__(WR == 2 ? 512 : 256) __attribute__((amdgpu_waves_per_eu(WR == 1 ? 1 : 2, WR == 1 ? 1 : 2))) void prefill_f16(
    const uint8_t *w, Pieces p, float *__restrict__ y, int rows, int cols, int batch, int np, int token_blocks)
{
    if constexpr (WR == 0) wide_kernel<T, TT>(w, p, y, rows, cols, batch, np, token_blocks);
    else narrow_kernel<T, TT, WR>(w, p, y, rows, cols, batch, np, token_blocks);
}

template <int TT, int WR>
__global__ __launch_bounds__(WR == 2 ? 512 : 256) __attribute__((amdgpu_waves_per_eu(WR == 1 ? 1 : 2, WR == 1 ? 1 : 2))) void prefill_mfma(
    const uint8_t *w, Pieces p, float *__restrict__ y, int rows, int cols, int batch, int np, int token_blocks)
{
    if constexpr (WR == 0) wide_kernel<Q6_K, TT>(w, p, y, rows, cols, batch, np, token_blocks);
    else narrow_kernel<Q6_K, TT, WR>(w, p, y, rows, cols, batch, np, token_blocks);
}

#define FY_ARGS w, p, y, rows, cols, batch, np, token_blocks
template <int TT, int WR>
hipError_t launch_blocks(unsigned type, const uint8_t *w, const Pieces &p, float *y, int rows, int cols, int batch,
    int np, hipStream_t s)
{
    const int token_blocks = (batch + 32 * TT - 1) / (32 * TT), per = kTileRows * kR * WR;
    const dim3 grid((unsigned)(((long)rows + per - 1) / per * token_blocks)), block(256 * WR);
    if (type == Q8_0) hipLaunchKernelGGL((prefill_f16<Q8_0, TT, WR>), grid, block, 0, s, FY_ARGS);
    else if (type == Q4_0) hipLaunchKernelGGL((prefill_f16<Q4_0, TT, WR>), grid, block, 0, s, FY_ARGS);
    else if (type == Q6_K) hipLaunchKernelGGL((prefill_mfma<TT, WR>), grid, block, 0, s, FY_ARGS);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_wide(unsigned type, const uint8_t *w, const Pieces &p, float *y, int rows, int cols, int batch, int np,
    hipStream_t s)
{
    const int token_blocks = (batch + 63) / 64, per = 4 * kTileRows * kR;
    const dim3 grid((unsigned)(((long)rows + per - 1) / per * token_blocks)), block(256);
    if (type == Q4_K) hipLaunchKernelGGL((prefill_f16<Q4_K, 2, 0>), grid, block, 0, s, FY_ARGS);
    else if (type == Q8_0) hipLaunchKernelGGL((prefill_f16<Q8_0, 2, 0>), grid, block, 0, s, FY_ARGS);
    else if (type == Q4_0) hipLaunchKernelGGL((prefill_f16<Q4_0, 2, 0>), grid, block, 0, s, FY_ARGS);
    else if (type == Q6_K) hipLaunchKernelGGL((prefill_mfma<2, 0>), grid, block, 0, s, FY_ARGS);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// 256 rows x 32 tokens (Q8_0 and Q4_0).
hipError_t launch_half(unsigned type, const uint8_t *w, const Pieces &p, float *y, int rows, int cols, int batch, int np,
    hipStream_t s)
{
    const int token_blocks = (batch + 31) / 32, per = 4 * kTileRows * kR;
    const dim3 grid((unsigned)(((long)rows + per - 1) / per * token_blocks)), block(256);
    if (type == Q8_0) hipLaunchKernelGGL((prefill_f16<Q8_0, 1, 0>), grid, block, 0, s, FY_ARGS);
    else if (type == Q4_0) hipLaunchKernelGGL((prefill_f16<Q4_0, 1, 0>), grid, block, 0, s, FY_ARGS);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
#undef FY_ARGS

}  // namespace

// The workgroup shape with the fewest idle CUs, smallest first: up to 256
// workgroups (one per CU) of 64 rows x 32 tokens, then 128 x 32, then 128 x 64;
// past that 256 x 64 wide. Q4_K's narrow shapes close a group (its minimums
// and scales) every 64 columns of a wavefront and lose to the 32-token
// workgroups of prefill_f16.hip, which keep every batch that would not give some
// CU two of 256 x 64 (with just one for each, the older form of that shape is
// faster: 8192 x 4096 x512 76.8 us there, 84.3 here; 4096 x 4096 x1024 79.4, 85.3).
// Measured, us (64x32 / 128x32 / 128x64 / 256x64; the int8 kernel before for Q6_K,
// prefill_f16.hip for the others):
//   Q6_K 4096x14336 x128     82 / 105 / 136 / 249   218
//   Q6_K 4096x14336 x256    148 / 115 / 140 / 251   275
//   Q6_K 4096x14336 x512    288 / 220 / 171 / 256   502
//   Q6_K 4096x4096  x512    102 /  74 /  62 /  83   161
//   Q4_K 14336x4096 x512    331 / 220 / 218 / 123   136
//   Q4_K 11264x2048 x256     88 /  60 /  73 /  41    42
//   Q4_K 4096x4096  x512    105 /  69 /  65 /  70    48
// Tall Q6_K matrices are bound by their weights on few tokens: 128256 x 4096, 9
// tokens 157 (the int8 kernel's 16-token workgroups: 182).
//
// Q8_0 and Q4_0: where that shape leaves its last round of the CUs nearly empty,
// 256 x 32, or for rows of up to eight groups prefill_f16.hip (128 x 32, two to
// a CU, no shares to add), if its time by the model below is less. us: the kernels
// before this file's, the shape by the workgroups alone, now:
//   Q8_0 42240x5632 x22    80 / 107 /  66    Q4_0 16896x14336 x89   152 / 217 / 138
//   Q8_0 7104x8192 x283   112 / 156 / 100    Q4_0 7872x256 x182      12 /  17 /  11
//   Q8_0 6432x512 x305     18 /  21 /  17    Q4_0 992x1024 x994      18 /  20 /  16
enum Shape { kRows64, kRows128, kRows128Wide, kRows256, kRows256Half, kElsewhere };

// A shape's time in 10 ns, for Q8_0 (Q4_0's are the same to a few percent):
// `pair` and `single` per 256-column group of two workgroups on a CU and of one
// (narrow ones come one at a time), `round` per such workgroup, `once`, and
// per 1000 tokens and group, and 1000 tokens, the split. Fitted to 1600 shapes
// (256 to 80000 rows, 256 to 14336 columns, 21 to 2048 tokens): half of a form's
// times within 4 to 6 %, nine of ten within 9 to 13; what the rule takes is within
// 2 % of the faster of both kernels before it on all but 12, 0.4 to 4 us off there.
struct ShapeTime {
    long pair, single, round, once, split_group, split;
};
constexpr ShapeTime kTimes[] = {{172, 86, 405, 419, 57, 229},  {228, 114, 638, 207, 41, 239},
                                {418, 209, 1273, 0, 24, 645},  {680, 413, 278, 613, 35, 214},
                                {400, 240, 174, 546, 37, 193}, {256, 188, 138, 497, 30, 174}};

static long time_of(Shape shape, long workgroups, long groups, long tokens)
{
    const ShapeTime &t = kTimes[shape];
    const long k = (workgroups + 255) / 256;   // of the fullest CU
    return (k / 2 * t.pair + k % 2 * t.single) * groups + k * t.round + t.once +
           tokens * (groups * t.split_group + t.split) / 1000;
}

static Shape shape_of(unsigned type, int rows, int cols, int whole)
{
    const long t32 = ((long)whole + 31) / 32, t64 = ((long)whole + 63) / 64;
    auto blocks = [&](int per) { return ((long)rows + per - 1) / per; };
    if (type == Q4_K) return blocks(256) * t64 > 256 ? kRows256 : kElsewhere;
    const long workgroups[] = {blocks(64) * t32,  blocks(128) * t32, blocks(128) * t64,
                               blocks(256) * t64, blocks(256) * t32, blocks(128) * t32};
    int shape = kRows64;
    while (shape < kRows256 && workgroups[shape] > 256) ++shape;
    if (type == Q6_K) return (Shape)shape;
    const long groups = cols / kGroupCols;
    long least = time_of((Shape)shape, workgroups[shape], groups, whole);
    // (From 256 workgroups of 256 x 64 on, prefill_f16.hip has another shape.)
    const int last = groups <= 8 && workgroups[kRows256] < 256 ? kElsewhere : kRows256Half;
    for (int s = kRows256Half; s <= last; ++s) {
        const long time = time_of((Shape)s, workgroups[s], groups, whole);
        if (time < least) least = time, shape = s;
    }
    return (Shape)shape;
}

bool prefill_tile_supported(unsigned type, int rows, int cols, int whole)
{
    return cols % kGroupCols == 0 && shape_of(type, rows, cols, whole) != kElsewhere;
}

hipError_t launch_prefill_tile(unsigned type, const uint8_t *w, const float *x, float *y, int rows, int cols, int batch,
    int whole, void *workspace, int np, hipStream_t s)
{
    const Pieces p = pieces_of(workspace, cols, np);
    const hipError_t e = launch_split_x(x, batch, cols, p, true, s);
    if (e != hipSuccess) return e;
    switch (shape_of(type, rows, cols, whole)) {
    case kRows64: return launch_blocks<1, 1>(type, w, p, y, rows, cols, batch, np, s);
    case kRows128: return launch_blocks<1, 2>(type, w, p, y, rows, cols, batch, np, s);
    case kRows128Wide: return launch_blocks<2, 2>(type, w, p, y, rows, cols, batch, np, s);
    case kRows256Half: return launch_half(type, w, p, y, rows, cols, batch, np, s);
    case kRows256: return launch_wide(type, w, p, y, rows, cols, batch, np, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace fy
