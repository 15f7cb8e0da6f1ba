// Decode attention of one layer over an f16 KV cache, bit-identical to the
// reference's x86 path: attn_head (reference engine.c:90-147) with its AVX2
// f16 dot (kernels_avx2.c:118-148), softmax (kernels.c:855-885) and the
// softmax's exp polynomial (kernels.c:820-850).
//
// Up to about a thousand positions (the host's rule) one launch,
// attn_fused_kernel: a workgroup per query head and a few blocks of 16 value
// rows scores every position itself. Beyond, three launches on one stream:
//   attn_scores_kernel   s[h][j] = dot(K[hk][j], f16(q_h)) * kq_scale, and the
//                        maximum of each block of positions
//   attn_exp_kernel      e[h][j] = exp(s[h][j] - max), and each block's total
//   attn_pv_kernel       out[h][c] = dot(V[hk][c][0..n), f16(e[h] / total))
//
// The f16 dot is evaluated in the reference's order. Its 32 f32
// accumulators (accumulator a takes elements i with i % 32 == a, by FMA in
// increasing i) are reduced as registers r0+r2, r1+r3 (8 accumulators
// each), then their sum, then elements l and l+4, then two pairwise rounds;
// elements past the last multiple of 32 are added to the double total one
// by one. Each accumulator is one chain of n / 32 dependent FMAs over the
// whole context, so the value contraction cannot be split along the
// positions without changing the result: the parallelism is over rows,
// heads and accumulators.
//
// The softmax sums its 8-element group totals in double in a tree rather
// than in the reference's sequential order. The two double totals differ
// by at most n * 2^-53 relative, which changes the float 1/total only when
// that lies within that distance of a float rounding boundary (about 1e-6
// of heads at n = 4096). Tail elements (n % 8) use expf in the reference
// (libm): here exp in double rounded to float, which differs from glibc's
// expf in about 0.07% of arguments by one float ulp, and such a difference
// survives the f16 rounding of its probability only rarely.
#pragma once

#include <type_traits>

#include "quant.h"

namespace sihip {

constexpr int kAttnMaxHd = 512;
constexpr int64_t kAttnMaxN = (int64_t)1 << 29;  // positions, so that indexes stay ints
constexpr int kAttnHeads = 4;  // query heads per workgroup of the scores launch
constexpr int64_t kAttnWsBlock = 4096;  // positions that workspace rows are a multiple of

struct AttnArgs {
    const float *q;        // [n_head * hd]
    const uint16_t *k;     // [n_head_kv][n_ctx][hd]
    const uint16_t *v;     // [n_head_kv][hd][n_ctx]
    float *out;            // [n_head * hd]
    float *sc;             // [n_head][ld] scaled scores (caller's, optional)
    uint16_t *p16;         // [n_head][ld] f16 probabilities (caller's, optional)
    float *sw;             // [n_head][lw] scores, then exponentials (workspace)
    float *pm;             // [n_head][nbs] maxima of the score blocks (workspace)
    double *ps;            // [n_head][nbe] totals of the exponential blocks (workspace)
    int64_t n_ctx, ld, lw;
    int n, hd, gqa, n_kv;
    int nbs, nbe;
    union {
        int gx;            // blocks per row of the grid (attn_block)
        int rb;            // 16-row blocks of values per workgroup of the single launch
    };
    float kq_scale;
};

// The scores and exponential launches have a block per piece of a head's
// positions, which can be more than one grid dimension takes (2^32 work items:
// 32 heads over 1 KV head at 2^27 positions): past kAttnGridX blocks the grid
// has further rows, the last one with blocks to spare.
constexpr int64_t kAttnGridX = (int64_t)1 << 22;
__device__ inline int attn_block(const AttnArgs &A) { return (int)blockIdx.y * A.gx + (int)blockIdx.x; }

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));

__device__ inline float f16_at(const uint16_t *p, int64_t i) { return f16_bits_to_f32(p[i]); }

// f32_to_f16_bits by the hardware's conversion (RNE, subnormals kept; the
// bits of a NaN as f32_to_f16_bits makes them). The empty asm keeps a
// product in f from being folded into the conversion (v_fma_mixlo_f16), which
// would round once where the reference rounds to f32 first.
__device__ inline uint32_t f32_to_f16_hw(float f) {
    asm("" : "+v"(f));
    const uint32_t u = __float_as_uint(f), m = (u >> 13) & 0x3ffu;
    const uint32_t nan = ((u >> 16) & 0x8000u) | 0x7e00u | (m == 0u ? 1u : m);
    const uint32_t h = __builtin_bit_cast(uint16_t, (_Float16)f);
    return (u & 0x7fffffffu) > 0x7f800000u ? nan : h;
}

// Lane i receives lane i + K of its 16-lane row (a DPP row shift; lanes
// whose source lies past the row receive 0, and are not used below).
template <int K>
__device__ inline float from_lane_up(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x100 + K, 0xf, 0xf, true));
}

__device__ inline float max_sel(float a, float b) { return b > a ? b : a; }

// Reductions over a wave without LDS round trips: DPP within the 16-lane
// rows, then the gfx950 row and half swaps (each returns both lanes' values).
__device__ inline uint2 swap16(uint32_t x) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return make_uint2(r[0], r[1]);
}
__device__ inline uint2 swap32(uint32_t x) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return make_uint2(r[0], r[1]);
}

__device__ inline float wave_max(float x) {
    const int ctrls[4] = {kDppXor1, kDppXor2, kDppHalfMirror, kDppMirror};
#pragma unroll
    for (int i = 0; i < 4; i++) x = max_sel(x, __uint_as_float(dpp_u32(__float_as_uint(x), ctrls[i])));
    uint2 t = swap16(__float_as_uint(x));
    x = max_sel(__uint_as_float(t.x), __uint_as_float(t.y));
    t = swap32(__float_as_uint(x));
    return max_sel(__uint_as_float(t.x), __uint_as_float(t.y));
}

__device__ inline double wave_sum(double x) {
    const int ctrls[4] = {kDppXor1, kDppXor2, kDppHalfMirror, kDppMirror};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint64_t u = __builtin_bit_cast(uint64_t, x);
        const uint64_t o = (uint64_t)dpp_u32((uint32_t)u, ctrls[i]) |
                           ((uint64_t)dpp_u32((uint32_t)(u >> 32), ctrls[i]) << 32);
        x += __builtin_bit_cast(double, o);
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint64_t u = __builtin_bit_cast(uint64_t, x);
        const uint2 lo = i ? swap32((uint32_t)u) : swap16((uint32_t)u);
        const uint2 hi = i ? swap32((uint32_t)(u >> 32)) : swap16((uint32_t)(u >> 32));
        x = __builtin_bit_cast(double, (uint64_t)lo.x | ((uint64_t)hi.x << 32)) +
            __builtin_bit_cast(double, (uint64_t)lo.y | ((uint64_t)hi.y << 32));
    }
    return x;
}

// exp of the softmax groups: the polynomial the reference uses there (its
// constants and branch structure kept, since the result is compared bit
// for bit): x = n ln2 + b with n from the 1.5 * 2^23 rounding shift and ln2
// in two parts, a polynomial in b, and 2^n built in the exponent field;
// |n| > 126 scales by two factors, |n| > 192 saturates.
__device__ inline float expf_poly(float x) {
    const float shift = 0x1.8p23f;
    const float z = __builtin_fmaf(x, 0x1.715476p+0f, shift);
    const float n = z - shift;
    const float b = __builtin_fmaf(-n, 0x1.7f7d1cp-20f, __builtin_fmaf(-n, 0x1.62e4p-1f, x));
    const uint32_t e = __float_as_uint(z) << 23;
    const float k = __uint_as_float(e + 0x3f800000u);
    const float u = b * b;
    const float p = __builtin_fmaf(
        __builtin_fmaf(__builtin_fmaf(0x1.0e4020p-7f, b, 0x1.573e2ep-5f), u,
                       __builtin_fmaf(0x1.555e66p-3f, b, 0x1.fffdb6p-2f)),
        u, 0x1.ffffecp-1f * b);
    if (!(__builtin_fabsf(n) > 126.0f)) return __builtin_fmaf(p, k, k);
    const uint32_t g = n <= 0.0f ? 0x82000000u : 0u;
    const float s1 = __uint_as_float(g + 0x7f000000u);
    if (__builtin_fabsf(n) > 192.0f) return s1 * s1;
    const float s2 = __uint_as_float(e - g);
    return __builtin_fmaf(s2, p, s2) * s1;
}

// exp of a tail position's shifted score (positions past the last whole
// 8-group): exp in double, rounded.
__device__ inline float tail_exp(float x) { return (float)exp((double)x); }

// A workgroup's query head and 1D block index: consecutive workgroups take
// different KV heads, so that where their number is a multiple of 8 the
// launches of a KV head run on one XCD and find its rows and scores in that
// XCD's L2.
struct AttnWg {
    int hk, h, blk;
};
__device__ inline AttnWg attn_wg(const AttnArgs &A, int n_kv, int id) {
    const int rest = id / n_kv;
    AttnWg w;
    w.hk = id % n_kv;
    w.h = w.hk * A.gqa + rest % A.gqa;
    w.blk = rest / A.gqa;
    return w;
}

// ---- scores ---------------------------------------------------------------------
//
// Four lanes score one position: lane L of the quad holds accumulators
// 8 L .. 8 L + 7, so a 32-element step of the key row is one 16-byte load per
// lane and a wave's 16 rows are one contiguous span of the cache. T: 32-steps
// kept in registers (hd / 32 <= T); W: elements per load, 8 (hd % 8 == 0, keys
// 16-byte aligned), 4 (hd % 4 == 0, 8-byte aligned) or 1.
// (lane L < hd % 32 / 8 also holds elements 8 L .. + 7 past the last whole
// step in tail, zeros past hd.)
template <int T>
struct KeyRow {
    uint4 w[T];
    uint4 tail;
};

// Elements p[0 .. cnt) of eight, zeros behind (cnt > 0; with W = 8 all of
// them, with W = 4 the first four or all).
template <int W>
__device__ inline uint4 load_key8(const uint16_t *p, int cnt) {
    if constexpr (W == 8) {
        return *reinterpret_cast<const uint4 *>(p);
    } else if constexpr (W == 4) {
        const uint2 a = *reinterpret_cast<const uint2 *>(p);
        const uint2 b = cnt > 4 ? *reinterpret_cast<const uint2 *>(p + 4) : make_uint2(0, 0);
        return make_uint4(a.x, a.y, b.x, b.y);
    } else {
        uint32_t e[8];
#pragma unroll
        for (int i = 0; i < 8; i++) e[i] = i < cnt ? p[i] : 0u;
        return make_uint4(e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16));
    }
}

template <int T, int W>
__device__ inline void load_key(const uint16_t *row, int hd, int L, KeyRow<T> &k) {
    const int steps = hd >> 5;
#pragma unroll
    for (int t = 0; t < T; t++)
        if (t < steps) k.w[t] = load_key8<W>(row + 32 * t + 8 * L, 8);
    if (hd & 31)
        k.tail = 8 * L < (hd & 31) ? load_key8<W>(row + 32 * steps + 8 * L, (hd & 31) - 8 * L) : make_uint4(0, 0, 0, 0);
}

// The scaled score of the quad's row against the f16 query (q: the lane's
// elements of it, as load_key lays them out; in its tail anything past hd);
// valid in the quad's lane 0. Every lane of the wave takes part. NEXT: the row
// `next` is loaded into k, each piece as soon as it is used.
template <int T, int W, bool NEXT = false>
__device__ inline float key_score(KeyRow<T> &k, const KeyRow<T> &q, int hd, float kq_scale,
                                  const uint16_t *next = nullptr, int L = 0) {
    const int steps = hd >> 5;
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < T; t++)
        if (t < steps) {
            const h8_t kk = __builtin_bit_cast(h8_t, k.w[t]);
            const h8_t qq = __builtin_bit_cast(h8_t, q.w[t]);
#pragma unroll
            for (int e = 0; e < 8; e++) acc[e] = __builtin_fmaf((float)kk[e], (float)qq[e], acc[e]);
            if constexpr (NEXT) k.w[t] = load_key8<W>(next + 32 * t + 8 * L, 8);
        }
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] = acc[e] + from_lane_up<2>(acc[e]);  // r0 + r2, r1 + r3
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] = acc[e] + from_lane_up<1>(acc[e]);  // their sum
    float t4[4];
#pragma unroll
    for (int e = 0; e < 4; e++) t4[e] = acc[e] + acc[e + 4];
    const float res = (t4[0] + t4[1]) + (t4[2] + t4[3]);
    double total = 0.0;
    total += (double)res;
    if (hd & 31) {
        // each lane's products, added in element order (8 per lane)
        const h8_t kk = __builtin_bit_cast(h8_t, k.tail), qq = __builtin_bit_cast(h8_t, q.tail);
        float pr[8];
#pragma unroll
        for (int e = 0; e < 8; e++) pr[e] = (float)kk[e] * (float)qq[e];
        if constexpr (NEXT)
            if (8 * L < (hd & 31)) k.tail = load_key8<W>(next + 32 * steps + 8 * L, (hd & 31) - 8 * L);
        auto add = [&](auto from, int cnt) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (e % W == 0 && e >= cnt) break;
                total += (double)quad_bcast<decltype(from)::value>(pr[e]);
            }
        };
        const int cnt = hd & 31;
        add(std::integral_constant<int, 0>(), cnt);
        if (cnt > 8) add(std::integral_constant<int, 1>(), cnt - 8);
        if (cnt > 16) add(std::integral_constant<int, 2>(), cnt - 16);
        if (W < 8 && cnt > 24) add(std::integral_constant<int, 3>(), cnt - 24);
    }
    return (float)total * kq_scale;
}

// Grid ceil(n / 64) x ceil(gqa / 4) x n_kv, in one dimension (KV head
// fastest): a workgroup scores 64 positions against up to 4 query heads of
// one KV head, each key row kept in registers across the heads, and writes
// the block's maximum per head. Bound: HBM (the key rows are read once);
// all workgroups of 16k positions are resident together, so the whole read
// is in flight at once.
constexpr int kAttnScoreBlock = 64;

template <int T, int W>
__global__ __launch_bounds__(256) void attn_scores_kernel(AttnArgs A) {
    __shared__ __attribute__((aligned(16))) uint16_t q16[kAttnHeads][kAttnMaxHd];
    __shared__ float red[kAttnHeads][4];
    const int chunks = (A.gqa + kAttnHeads - 1) / kAttnHeads;
    const int id = attn_block(A), hk = id % A.n_kv, rest = id / A.n_kv;
    // (a spare block scores row n - 1 and stores nothing: to return here would
    // put a second round trip for arguments before the key loads, 0.2 us)
    const int hc = rest % chunks * kAttnHeads, blk = rest / chunks;
    const int h0 = hk * A.gqa + hc, nh = min(kAttnHeads, A.gqa - hc);
    const int hd = A.hd;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, L = lane & 3;
    const int j = blk * kAttnScoreBlock + (int)(threadIdx.x >> 2);
    // rows past n score row n - 1, unstored
    const uint16_t *row = A.k + ((int64_t)hk * A.n_ctx + (j < A.n ? j : A.n - 1)) * hd;
    KeyRow<T> kr;
    load_key<T, W>(row, hd, L, kr);
    // the query heads in f16, staged while the key loads are in flight
    for (int hh = 0; hh < nh; hh++)
        for (int i = threadIdx.x; i < hd; i += 256)
            q16[hh][i] = (uint16_t)f32_to_f16_hw(A.q[(int64_t)(h0 + hh) * hd + i]);
    __syncthreads();
    for (int hh = 0; hh < nh; hh++) {
        KeyRow<T> qr;
        load_key<T, 8>(q16[hh], hd, L, qr);
        const float v = key_score<T, W>(kr, qr, hd, A.kq_scale);
        const bool real = L == 0 && j < A.n;
        if (real) {
            A.sw[(int64_t)(h0 + hh) * A.lw + j] = v;
            if (A.sc) A.sc[(int64_t)(h0 + hh) * A.ld + j] = v;
        }
        const float mx = wave_max(real ? max_sel(-__builtin_inff(), v) : -__builtin_inff());
        if (lane == 0) red[hh][wave] = mx;
    }
    __syncthreads();
    if ((int)threadIdx.x < nh && blk < A.nbs) {
        const float *r = red[threadIdx.x];
        A.pm[(int64_t)(h0 + threadIdx.x) * A.nbs + blk] =
            max_sel(max_sel(r[0], r[1]), max_sel(r[2], r[3]));
    }
}

// ---- softmax pieces ---------------------------------------------------------------
//
// Four consecutive positions j .. j + 3 (j a multiple of 4) of a head per
// thread, neighbours (lane ^ 1) sharing an 8-group. x: their scores, on
// return their exponentials. Returns the thread's share of the total: the
// 8-group's float sum in the reference's lane order from its even thread,
// nothing from the tail [gend, n). Every lane of the wave takes part.
//
// The tail, at most seven positions, is left to as many lanes of one wave
// (tail_exp is a double exp: evaluated four times in turn by the thread that
// holds the positions it cost 2 us of a launch).
__device__ inline double exp4(float (&x)[4], int j, int gend, float mx) {
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = expf_poly(x[e] - mx);
    float a[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float o = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x[e]), kDppXor1, 0xf, 0xf, false));
        a[e] = x[e] + o;
    }
    return j < gend && !(j & 4) ? (double)((a[0] + a[2]) + (a[1] + a[3])) : 0.0;
}

// Grid ceil(n / 1024) x n_head in one dimension (attn_wg): the exponentials
// of a block of 1024 positions of a head, in place of its scores, and their
// total. The whole softmax in one workgroup per head took 14 us at n = 7000
// (three passes over the row by 32 workgroups); spread over the positions it
// takes 2-4.5 us, a launch's latency.
constexpr int kAttnExpBlock = 1024;

__global__ __launch_bounds__(256) void attn_exp_kernel(AttnArgs A) {
    __shared__ float redf[4];
    __shared__ double redd[4];
    // one round trip for the arguments, not another behind the branch
    int n_kv = A.n_kv;
    asm volatile("" : "+s"(n_kv) : "s"(A.gx), "s"(A.n), "s"(A.sw), "s"(A.lw), "s"(A.pm));
    const AttnWg W = attn_wg(A, n_kv, attn_block(A));
    if (W.blk >= A.nbe) return;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int j = W.blk * kAttnExpBlock + 4 * (int)threadIdx.x;
    float4 *const p = reinterpret_cast<float4 *>(A.sw + (int64_t)W.h * A.lw + j);
    const float4 f = *p;  // lw is a multiple of the block
    // tail position gend + tid, where it lies in this block
    const int gend = A.n & ~7, jt = gend + (int)threadIdx.x;
    const bool tail = jt < A.n && gend / kAttnExpBlock == W.blk;
    float *const pt = A.sw + (int64_t)W.h * A.lw + jt;
    float xt = 0.0f;
    if (tail) xt = *pt;
    float mx = -__builtin_inff();
    for (int i = threadIdx.x; i < A.nbs; i += 256) mx = max_sel(mx, A.pm[(int64_t)W.h * A.nbs + i]);
    mx = wave_max(mx);
    if (lane == 0) redf[wave] = mx;
    __syncthreads();
    mx = max_sel(max_sel(redf[0], redf[1]), max_sel(redf[2], redf[3]));
    float x[4] = {f.x, f.y, f.z, f.w};
    double part = exp4(x, j, gend, mx);
    if (tail) {
        xt = tail_exp(xt - mx);
        part += (double)xt;
        *pt = xt;
    }
    part = wave_sum(part);
    if (j < gend) *p = make_float4(x[0], x[1], x[2], x[3]);
    if (lane == 0) redd[wave] = part;
    __syncthreads();
    if (threadIdx.x == 0)
        A.ps[(int64_t)W.h * A.nbe + W.blk] = (redd[0] + redd[1]) + (redd[2] + redd[3]);
}

// ---- values -----------------------------------------------------------------------
//
// Grid ceil(hd / 16) x n_head in one dimension (attn_wg): a workgroup owns 16
// value rows of one query head; lane (row r, L < 16) runs accumulators 2 L
// and 2 L + 1 of row r. The value rows and the head's exponentials stream
// into LDS by DMA in chunks of 512 positions, three chunks ahead of the
// chains, so the loads are bound by the memory and not by a round trip per
// chunk (staged through registers 2048 positions at a time, one chunk's
// loads after the other's chains, 13.6 us at n = 7000), and each chunk's
// probabilities are made while the chunk before runs, so that a chunk costs
// one barrier. Row slots are padded by 64 bytes so that the four rows of a
// wave read distinct LDS banks.
constexpr int kAttnPvRows = 16;
constexpr int kAttnChunk = 512;
constexpr int kAttnRing = 4;
constexpr int kAttnRowSlot = kAttnChunk * 2 + 64;
constexpr int kAttnSlot = kAttnPvRows * kAttnRowSlot;

typedef int attn_rsrc_t __attribute__((ext_vector_type(4)));

// Copies of 1 KiB (16 bytes per lane) from a buffer straight into LDS, at
// buffer offset voff (range-checked: zeros past the buffer's end), LDS byte
// offset lds (wave-uniform). They are in flight until the wave's vmcnt covers
// them; the compiler does not count them, so every use is behind an explicit
// wait. The compiler's own m0 is put back.
__device__ inline void attn_dma(attn_rsrc_t rsrc, uint32_t voff, uint32_t lds) {
    uint32_t m0;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %2, %3, 0 offen lds\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(m0)
        : "s"(lds), "v"(voff), "s"(rsrc)
        : "memory");
}
// Four of them at voff[i] + add, the LDS offset advancing by kAttnRowSlot.
__device__ inline void attn_dma_rows(attn_rsrc_t rsrc, const uint32_t (&voff)[4], uint32_t add,
                                     uint32_t lds) {
    uint32_t m0;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %2, %6, 0 offen lds\n\t"
        "s_add_u32 m0, m0, %7\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %3, %6, 0 offen lds\n\t"
        "s_add_u32 m0, m0, %7\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %4, %6, 0 offen lds\n\t"
        "s_add_u32 m0, m0, %7\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %5, %6, 0 offen lds\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(m0)
        : "s"(lds), "v"(voff[0] + add), "v"(voff[1] + add), "v"(voff[2] + add), "v"(voff[3] + add),
          "s"(rsrc), "n"(kAttnRowSlot)
        : "memory", "scc");
}

__device__ inline attn_rsrc_t attn_rsrc(const void *p, uint32_t bytes) {
    const uint64_t a = (uint64_t)(uintptr_t)p;
    return (attn_rsrc_t){__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                         __builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32) & 0xffff),
                         __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000};
}

// The tree over the 32 accumulators of one row, 32 / NL per lane in lanes
// L = 0 .. NL - 1 of the row (acc[e] = accumulator 32 / NL * L + e); valid in
// L == 0. Every lane of the wave takes part.
__device__ inline float row_tree2(float a0, float a1) {  // 16 lanes, 2 each
    a0 += from_lane_up<8>(a0), a1 += from_lane_up<8>(a1);  // r0 + r2, r1 + r3
    a0 += from_lane_up<4>(a0), a1 += from_lane_up<4>(a1);  // their sum
    a0 += from_lane_up<2>(a0), a1 += from_lane_up<2>(a1);  // l and l + 4
    const float b = a0 + a1;
    return b + from_lane_up<1>(b);
}
__device__ inline float row_tree1(float a) {  // 32 lanes, 1 each
    a += __shfl_down(a, 16);
    a += from_lane_up<8>(a);
    a += from_lane_up<4>(a);
    a += from_lane_up<1>(a);
    return a + from_lane_up<2>(a);
}

// res plus the tail [body, n) of a dot, added in order in double; v and p:
// f16 rows of the 32-element block at body (LDS, 16-byte aligned, v with
// ALIGNED).
template <bool ALIGNED>
__device__ inline float add_tail(float res, const uint16_t *v, const uint16_t *p, int cnt) {
    double total = 0.0;
    total += (double)res;
    if (cnt > 0) {
        h8_t vv[4], pp[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if constexpr (ALIGNED) {
                vv[i] = reinterpret_cast<const h8_t *>(v)[i];
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) vv[i][e] = reinterpret_cast<const _Float16 *>(v)[8 * i + e];
            }
            pp[i] = reinterpret_cast<const h8_t *>(p)[i];
        }
#pragma unroll
        for (int i = 0; i < 31; i++)
            if (i < cnt) total += (double)((float)vv[i >> 3][i & 7] * (float)pp[i >> 3][i & 7]);
    }
    return (float)total;
}

// VEC: n_ctx % 8 == 0, v 16-byte aligned and the workgroup's rows within a
// buffer's 4 GiB. Else the rows start anywhere in a 16-byte granule of memory:
// a row's 16 lanes, which alone read it, load the whole granules that hold
// its chunk (65 of them; a granule with an element of the row lies in the
// row's pages, and what else it holds is not used) a chunk ahead into registers
// and put them into its LDS slot, and the chains read at the row's shift. (By single elements, a
// chunk at a time: 8B shape at n = 4000, n_ctx 4001, 59.5 us per layer; so 14.9.)
template <bool VEC>
__global__ __launch_bounds__(256) void attn_pv_kernel(AttnArgs A) {
    constexpr int kR = VEC ? kAttnRing : 1;
    __shared__ __attribute__((aligned(16))) uint8_t ring[kR * kAttnSlot];
    __shared__ __attribute__((aligned(16))) float se[kR][kAttnChunk];
    __shared__ __attribute__((aligned(16))) uint16_t sp[2][kAttnChunk];
    const AttnWg W = attn_wg(A, A.n_kv, (int)blockIdx.x);
    const int tid = (int)threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = tid >> 4, L = tid & 15;
    const int rows = min(kAttnPvRows, A.hd - W.blk * kAttnPvRows);
    const int n = A.n, body = n & ~31;
    const uint16_t *const vb = A.v + ((int64_t)W.hk * A.hd + W.blk * kAttnPvRows) * A.n_ctx;
    const float *const eb = A.sw + (int64_t)W.h * A.lw;
    const int nchunk = (n + kAttnChunk - 1) / kAttnChunk;
    const uint32_t lds_v = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)ring;
    const uint32_t lds_e = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float *)&se[0][0];
    attn_rsrc_t vr, er;
    if constexpr (VEC) {
        vr = attn_rsrc(vb, (uint32_t)(rows * A.n_ctx * 2));
        er = attn_rsrc(eb, (uint32_t)(A.lw * 4));
    }
    // this wave's KiB of chunk ch's exponentials (waves 2 and 3 copy what 0
    // and 1 copy, the same bytes, so that every wave issues the same number)
    uint32_t voff[4];
#pragma unroll
    for (int i = 0; i < 4; i++) voff[i] = (uint32_t)(4 * wave + i) * (uint32_t)(A.n_ctx * 2) + lane * 16;
    const uint32_t voff_e = (uint32_t)(wave & 1) * 1024 + lane * 16;
    auto uni = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
    auto dma_e = [&](int ch) {
        const uint32_t cc = (uint32_t)min(ch, nchunk - 1);
        attn_dma(er, voff_e + cc * (kAttnChunk * 4),
                 uni(lds_e + (uint32_t)(ch % kR) * (kAttnChunk * 4) + (wave & 1) * 1024));
    };
    // value rows 4 wave .. + 3 of chunk ch (rows past hd read zeros), then
    // the exponentials of chunk ch + 1; chunks past the end copy the last one
    // again
    auto dma = [&](int ch) {
        const uint32_t cc = (uint32_t)min(ch, nchunk - 1);
        attn_dma_rows(vr, voff, cc * (kAttnChunk * 2),
                      uni(lds_v + (uint32_t)(ch % kR) * kAttnSlot + 4 * wave * kAttnRowSlot));
        dma_e(ch + 1);
    };
    // 1 / total, the block totals added in a fixed order
    double part = 0.0;
    for (int i = lane; i < A.nbe; i += 64) part += A.ps[(int64_t)W.h * A.nbe + i];
    if constexpr (VEC) {
        dma_e(0);
#pragma unroll
        for (int i = 0; i + 1 < kR; i++) dma(i);
    }
    const float scale = (float)(1.0 / wave_sum(part));
    // without VEC: the granules of this lane's row, 64 a chunk and one more
    const uint16_t *const vrow = vb + (int64_t)min(r, rows - 1) * A.n_ctx;
    const int shift = VEC ? 0 : (int)((uintptr_t)vrow & 15) / 2, last = (shift + n - 1) >> 3;
    const uint4 *const gran = reinterpret_cast<const uint4 *>(vrow - shift);
    struct Staged {
        uint4 v0, v1, v2, v3, v4;
        float2 e;
    };
    auto load_v = [&](int ch) {
        const int g = ch * (kAttnChunk / 8) + L;
        return Staged{gran[min(g, last)], gran[min(g + 16, last)], gran[min(g + 32, last)], gran[min(g + 48, last)],
                      L == 0 ? gran[min(g + 64, last)] : make_uint4(0, 0, 0, 0),
                      reinterpret_cast<const float2 *>(eb + (int64_t)ch * kAttnChunk)[tid]};
    };
    Staged st{};
    if constexpr (!VEC) st = load_v(0);
    // the probabilities of chunk ch from its exponentials e
    auto put_p = [&](int ch, float2 e) {
        const uint32_t p0 = f32_to_f16_hw(e.x * scale), p1 = f32_to_f16_hw(e.y * scale);
        reinterpret_cast<uint32_t *>(sp[ch & 1])[tid] = p0 | (p1 << 16);
        if (A.p16 && W.blk == 0) {
            const int64_t j = (int64_t)ch * kAttnChunk + 2 * tid;
            if (j < n) A.p16[(int64_t)W.h * A.ld + j] = (uint16_t)p0;
            if (j + 1 < n) A.p16[(int64_t)W.h * A.ld + j + 1] = (uint16_t)p1;
        }
    };
    if constexpr (VEC) {
        // the first exponentials: 15 younger copies
        static_assert(kAttnRing == 4, "wait counts");
        asm volatile("s_waitcnt vmcnt(15)" ::: "memory");
        __syncthreads();
        put_p(0, reinterpret_cast<const float2 *>(se[0])[tid]);
    }
    float a0 = 0.0f, a1 = 0.0f;
    const uint8_t *slot = ring;
    for (int ch = 0; ch < nchunk; ch++) {
        const int s0 = ch * kAttnChunk;
        if constexpr (VEC) {
            slot = ring + ch % kR * kAttnSlot;
            // chunk ch and the next exponentials have arrived (two younger
            // chunks of five copies in flight), this chunk's probabilities
            // are written, and every wave is done with chunk ch - 1
            asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
            __syncthreads();
            dma(ch + kR - 1);
        } else {
            uint4 *const dst = reinterpret_cast<uint4 *>(ring + r * kAttnRowSlot) + L;
            dst[0] = st.v0, dst[16] = st.v1, dst[32] = st.v2, dst[48] = st.v3;
            if (L == 0) dst[64] = st.v4;
            put_p(ch, st.e);
            st = load_v(min(ch + 1, nchunk - 1));
            __syncthreads();
        }
        const uint32_t *const vs = reinterpret_cast<const uint32_t *>(slot + r * kAttnRowSlot) + (shift >> 1) + L;
        const uint32_t *const ps = reinterpret_cast<const uint32_t *>(sp[ch & 1]) + L;
        // elements 2 L and 2 L + 1 of step t (across two words where the row's
        // shift is odd: an unaligned LDS read of a word took 4 times as long)
        auto pair = [&](int t) -> uint32_t {
            if constexpr (VEC) return vs[16 * t];
            else return __builtin_amdgcn_alignbit(vs[16 * t + 1], vs[16 * t], (uint32_t)(shift & 1) * 16);
        };
        auto chain = [&](uint32_t vw, uint32_t pw) {
            a0 = __builtin_fmaf(f16_bits_to_f32(vw & 0xffffu), f16_bits_to_f32(pw & 0xffffu), a0);
            a1 = __builtin_fmaf(f16_bits_to_f32(vw >> 16), f16_bits_to_f32(pw >> 16), a1);
        };
        const int steps = min(body - s0, kAttnChunk) >> 5;
        if (steps == kAttnChunk / 32) {
            // a whole chunk: all its reads go out first
            uint32_t vw[kAttnChunk / 32], pw[kAttnChunk / 32];
            float2 e;
            if constexpr (VEC) e = reinterpret_cast<const float2 *>(se[(ch + 1) % kR])[tid];
#pragma unroll
            for (int t = 0; t < kAttnChunk / 32; t++) vw[t] = pair(t), pw[t] = ps[16 * t];
            if constexpr (VEC) put_p(ch + 1, e);
#pragma unroll
            for (int t = 0; t < kAttnChunk / 32; t++) chain(vw[t], pw[t]);
        } else {
            if (VEC && ch + 1 < nchunk) put_p(ch + 1, reinterpret_cast<const float2 *>(se[(ch + 1) % kR])[tid]);
#pragma unroll 4
            for (int t = 0; t < steps; t++) chain(pair(t), ps[16 * t]);
        }
    }
    const float res = row_tree2(a0, a1);
    // the tail lies in the last chunk, still in LDS
    if (L == 0 && r < rows) {
        const int b0 = body % kAttnChunk;
        A.out[(int64_t)W.h * A.hd + W.blk * kAttnPvRows + r] =
            add_tail<VEC>(res, reinterpret_cast<const uint16_t *>(slot + r * kAttnRowSlot) + shift + b0,
                          sp[(nchunk - 1) & 1] + b0, n - body);
    }
    // no copy may land in the LDS of a workgroup that has ended
    if constexpr (VEC) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// ---- one launch -------------------------------------------------------------------
//
// Grid ceil(row blocks / rb) x n_head in one dimension (attn_wg), 8 waves: a
// workgroup scores all n positions of its query head (16 rows per wave and
// pass, the next pass's key rows in flight), runs the softmax in LDS and the
// chains of its rb blocks of 16 value rows, one block after another, one
// accumulator per thread. Every workgroup of a head repeats the scores (n * hd *
// 2 bytes from the L2 each), which costs less than the launches and round trips
// through memory that it saves until the rows grow long (8B shape, per layer:
// n = 600 15.5 -> 8.5 us against a scores launch and a value launch with the
// softmax in it) or the workgroups many: the host chooses rb for one workgroup
// per CU. What bounds it: 6 us at n = 16, the chain of one launch's start, the
// key and query loads, three barriers and the store; about 1.5 us for each
// further block, a round trip for its value rows.
// LDS (dynamic, attn_fused_lds): scores, probabilities, value rows, query.
constexpr int kAttnFusedThreads = 512;
constexpr int kAttnFuseCap = 1536;  // the largest the kernel takes (64 KiB of LDS)

__host__ __device__ inline int attn_fused_np(int n) { return (n + 31) / 32 * 32; }
__host__ __device__ inline int attn_fused_lds(int n) {
    const int np = attn_fused_np(n);
    return np * 4 + np * 2 + kAttnPvRows * (np * 2 + 64) + kAttnMaxHd * 2;
}

// VEC: value rows by 16-byte loads (n_ctx % 8 == 0, v 16-byte aligned). ONE: rb is
// 1, a kernel of its own (32 heads of 128 at n = 600 9.0 us per layer against 9.2
// with the loop over blocks).
template <int T, int KW, bool VEC, bool ONE>
__device__ inline void attn_fused_body(const AttnArgs &A) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    __shared__ float redf[8];
    __shared__ double redd[8];
    // one round trip for the arguments, not another for rb before the value loads
    // (0.25 us of a launch)
    int n_kv = A.n_kv;
    asm volatile("" : "+s"(n_kv) : "s"(A.n_ctx), "s"(A.k), "s"(A.rb));
    const int rb = ONE ? 1 : A.rb;
    const AttnWg W = attn_wg(A, n_kv, (int)blockIdx.x);
    const int n = A.n, np = attn_fused_np(n), hd = A.hd;
    uint16_t *const sq = reinterpret_cast<uint16_t *>(smem);
    float *const ss = reinterpret_cast<float *>(smem + kAttnMaxHd * 2);
    uint16_t *const sp = reinterpret_cast<uint16_t *>(ss + np);
    uint8_t *const sv = reinterpret_cast<uint8_t *>(sp + np);
    const int vslot = np * 2 + 64;
    const int tid = (int)threadIdx.x, wave = tid >> 6, lane = tid & 63;
    // scores: 128 positions per pass, four lanes each
    const int L4 = lane & 3, jr = tid >> 2;
    const uint16_t *const kb = A.k + (int64_t)W.hk * A.n_ctx * hd;
    auto key_row = [&](int pass) {
        const int j = 128 * pass + jr;
        return kb + (int64_t)(j < n ? j : n - 1) * hd;
    };
    const int passes = (n + 127) / 128;
    // passes of key rows held; with one, a pass's row is replaced piece by
    // piece (8 heads of 512 at n = 800: 14.3 us against 15.9 loaded after it)
    constexpr int kD = T <= 8 ? 2 : 1;
    KeyRow<T> kr[kD];
    load_key<T, KW>(key_row(0), hd, L4, kr[0]);
    float qv = 0.0f;
    if (tid < hd) qv = A.q[(int64_t)W.h * hd + tid];
#pragma unroll
    for (int i = 1; i < kD; i++)
        if (i < passes) load_key<T, KW>(key_row(i), hd, L4, kr[i]);
    // value rows, a block of 16 after another: 32 lanes per row; rows past hd
    // repeat the last, positions past n are not used
    const int r = tid >> 5, a = tid & 31;
    const int b1 = min((W.blk + 1) * rb, (hd + kAttnPvRows - 1) / kAttnPvRows);
    constexpr int kVP = kAttnFuseCap / 256;
    const int per8 = (n + 7) / 8;
    uint4 vq[kVP];
    uint8_t *const svr = sv + r * vslot;
    auto value_row = [&](int b) {
        return A.v + ((int64_t)W.hk * hd + min(b * kAttnPvRows + r, hd - 1)) * A.n_ctx;
    };
    auto load_v = [&](int b) {
        if constexpr (VEC) {
            const uint4 *const p = reinterpret_cast<const uint4 *>(value_row(b));
#pragma unroll
            for (int i = 0; i < kVP; i++) vq[i] = 32 * i < per8 ? p[min(32 * i + a, per8 - 1)] : make_uint4(0, 0, 0, 0);
        }
    };
    // block b (VEC: loaded before) to LDS: its row's lanes alone read it
    auto put_v = [&](int b) {
        if constexpr (VEC) {
#pragma unroll
            for (int i = 0; i < kVP; i++)
                if (32 * i + a < per8) *reinterpret_cast<uint4 *>(svr + (32 * i + a) * 16) = vq[i];
        } else {
            const uint16_t *const p = value_row(b);
            for (int i = a; i < n; i += 32) reinterpret_cast<uint16_t *>(svr)[i] = p[i];
        }
    };
    int b = W.blk * rb;
    load_v(b);
    if (tid < hd) sq[tid] = (uint16_t)f32_to_f16_hw(qv);
    __syncthreads();
    KeyRow<T> qr;
    load_key<T, 8>(sq, hd, L4, qr);
    float mx = -__builtin_inff();
    for (int p0 = 0; p0 < passes; p0 += kD) {
#pragma unroll
        for (int u = 0; u < kD; u++) {
            const int pass = p0 + u;
            if (pass < passes) {
                float v;
                if constexpr (kD == 1) {
                    v = key_score<T, KW, true>(kr[u], qr, hd, A.kq_scale, key_row(min(pass + 1, passes - 1)), L4);
                } else {
                    v = key_score<T, KW>(kr[u], qr, hd, A.kq_scale);
                    if (pass + kD < passes) load_key<T, KW>(key_row(pass + kD), hd, L4, kr[u]);
                }
                const int j = 128 * pass + jr;
                if (L4 == 0 && j < n) {
                    ss[j] = v;
                    mx = max_sel(mx, v);
                    if (A.sc && W.blk == 0) A.sc[(int64_t)W.h * A.ld + j] = v;
                }
            }
        }
    }
    put_v(b);
    if (!ONE && b + 1 < b1) load_v(b + 1);
    mx = wave_max(mx);
    if (lane == 0) redf[wave] = mx;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; i++) mx = max_sel(mx, redf[i]);
    const int j = 4 * tid;
    float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (j < np) {
        const float4 f = *reinterpret_cast<const float4 *>(ss + j);
        x[0] = f.x, x[1] = f.y, x[2] = f.z, x[3] = f.w;
    }
    // tail position gend + tid
    const int gend = n & ~7, jt = gend + tid;
    double part = exp4(x, j, gend, mx);
    float xt = 0.0f;
    if (jt < n) {
        xt = tail_exp(ss[jt] - mx);
        part += (double)xt;
    }
    part = wave_sum(part);
    if (lane == 0) redd[wave] = part;
    __syncthreads();
    part = ((redd[0] + redd[1]) + (redd[2] + redd[3])) + ((redd[4] + redd[5]) + (redd[6] + redd[7]));
    const float scale = (float)(1.0 / part);
    auto out_p = [&](int jj, uint32_t p) {
        if (A.p16 && W.blk == 0) A.p16[(int64_t)W.h * A.ld + jj] = (uint16_t)p;
    };
    if (j < gend) {
        uint32_t p[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            p[e] = f32_to_f16_hw(x[e] * scale);
            out_p(j + e, p[e]);
        }
        *reinterpret_cast<uint2 *>(sp + j) = make_uint2(p[0] | (p[1] << 16), p[2] | (p[3] << 16));
    }
    if (jt < n) {
        const uint32_t p = f32_to_f16_hw(xt * scale);
        sp[jt] = (uint16_t)p;
        out_p(jt, p);
    }
    __syncthreads();
    const uint16_t *const vs = reinterpret_cast<const uint16_t *>(svr);
    const int body = n & ~31;
    for (;;) {
        float acc = 0.0f;
#pragma unroll 8
        for (int i = a; i < body; i += 32)
            acc = __builtin_fmaf(f16_bits_to_f32(vs[i]), f16_bits_to_f32(sp[i]), acc);
        const float res = row_tree1(acc);
        const int c = b * kAttnPvRows + r;
        // (opaque, or the tail's 31 conditions are kept across the blocks in
        // scalar registers that spill)
        int cnt = n - body;
        if constexpr (!ONE) asm volatile("" : "+s"(cnt));
        if (a == 0 && c < hd) A.out[(int64_t)W.h * hd + c] = add_tail<true>(res, vs + body, sp + body, cnt);
        if (ONE || ++b >= b1) break;
        put_v(b);
        if (b + 1 < b1) load_v(b + 1);
    }
}

template <int T, int KW, bool VEC>
__global__ __launch_bounds__(kAttnFusedThreads)
__attribute__((amdgpu_waves_per_eu(T <= 4 ? 4 : 2))) void attn_fused_kernel(AttnArgs A) {
    attn_fused_body<T, KW, VEC, true>(A);
}
template <int T, int KW, bool VEC>
__global__ __launch_bounds__(kAttnFusedThreads)
__attribute__((amdgpu_waves_per_eu(T <= 4 ? 4 : 2))) void attn_fused_blocks_kernel(AttnArgs A) {
    attn_fused_body<T, KW, VEC, false>(A);
}

}  // namespace sihip
