// GEMM for short prompts of K-quant weights (Q2_K .. Q6_K) on
// v_mfma_i32_16x16x64_i8 (gfx950): Y_i[M x n_out_i] = X[M x n_in] * W_i^T for
// a group of matrices that share X, with X quantized per row to Q8_K by the
// bit-exact quantizer (reference kernels.c:561-595), each output within the
// tolerance of the reference dot (reference kernels.c:249-523).
//
// At 17 to about 100 activation rows a call is one pass over the weights
// with little matrix work per byte, so it is bound by how well the weights
// stream. A workgroup owns 16 NT weight rows of one matrix and a block of
// 16 MT activation rows, and its KW waves split the super-blocks among
// themselves (wave w takes c = w, w + KW, ...): the whole chip's waves
// stream separate runs of the weights, no wave waits for another until the
// tile's partial sums meet once in LDS, and no partial sums go through
// memory. Each super-block is decoded once, for the MT m tiles of the wave.
// The weights are the near-GGUF-size copy of gemmks.h, the activations 16-row
// records in MFMA operand order (gemm2_quantize_x<16>), read straight from
// the L2; both are loaded a whole super-block ahead of their use.
//
// Arithmetic per super-block, weight row n, activation row m:
//   S[m,n] = sum over the 16- or 32-element groups of scale * sum q x,
//   T[m,n] = sum_g min_g * bsum_g   (both exact),
//   y += dx * (d * S - dmin * T).
// The scaled quants are one or two int8 operands, made when a super-block
// is decoded, so the MFMAs accumulate S over the super-block themselves:
//   Q2_K: s q <= 45, one operand.
//   Q3_K: (4 - q) s in -128..124 (s = scale - 32), one operand; d negated.
//   Q4_K: s = 8 sh + sl: sh q and sl q (<= 105); S = 8 H + L.
//   Q5_K: the same, sh q and sl q <= 217 held as P - 128;
//         S = 8 H + L + 1152 sum x, the last term the MFMA's C input.
//   Q6_K: 2 (q - 32) s = 256 hi + lo, hi in -32..32, lo in -128..126 (even);
//         2 S = 256 H + L.
// The mins run on one v_mfma_f32_16x16x32_f16 against the group sums.
#pragma once

#include "agent.h"
#include "gemmks.h"

namespace sihip {

constexpr int kSKMaxSegs = 4;

struct GSKSeg {
    const uint8_t *w;   // gemmks.h chunks [nblk][nb]
    float *y;           // Y[m * ldy + n]
    int64_t ldy, n_out;
    uint32_t type;
    int nblk;           // blocks of 16 NT rows
    int wg0;            // first workgroup of the segment (a multiple of 8)
};

struct GSKArgs {
    const uint8_t *x;   // activation records [16-row block][nb] (g2_rec_bytes(16))
    int64_t M;
    int nb;             // super-blocks per row (n_in / 256)
    int MB;             // m blocks of 16 MT rows
    int nseg;
    GSKSeg seg[kSKMaxSegs];
};

// A lane's weights of one super-block, as stored: NT 16-row n tiles of a
// 32-row block (NT = 1: tile `half` of it).
template <uint32_t FMT, int NT>
struct SKRaw {
    uint2 qn[KS<FMT>::nib ? 4 : 1][NT];         // nibble formats: K-step, n tile
    uint32_t q2[KS<FMT>::nib ? 1 : 4][NT];      // 2-bit formats: the same
    uint32_t hb[KS<FMT>::QB > 0 ? 4 : 1][NT];   // Q6_K: the high fields; Q5_K, Q3_K: the extra bits, tile's at bit 0 ..
    uint4 sc[NT];    // the row's 16 scale bytes (Q3_K, Q6_K: word x, of lane group g)
    uint32_t sw[FMT == T_Q2_K ? NT : 1];  // Q2_K: the scale word of lane group g
    uint32_t d[NT];  // f16 d and dmin (Q3_K, Q6_K: the word holding d)
};

// Default cache policy: with the nontemporal hint of the M <= 8 kernels the
// same loads took 16-25% longer here (8B layer, 17 matrices' worth of calls:
// M = 37 94.5 against 79.2 us, M = 130 155 against 140): the m blocks and the
// two halves of a 32-row block read the lines again.
template <uint32_t FMT, int NT>
__device__ inline void sk_load_w(__amdgpu_buffer_rsrc_t wr, int c, int half, int lane, SKRaw<FMT, NT> &s) {
    using F = KS<FMT>;
    const int g = lane >> 4, r16 = lane & 15;
    auto ld4 = [&](int voff, int s_off) {
        return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wr, voff, s_off, 0));
    };
    const int so = __builtin_amdgcn_readfirstlane(c) * F::chunk;
    // words [K-step][n tile], 16 bytes per K-step pair
    auto pairs = [&](int off, uint32_t (*dst)[NT]) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint4 v = ld4(off + lane * 32 + j * 16, so);
            if constexpr (NT == 2) {
                dst[2 * j][0] = v.x, dst[2 * j][1] = v.y;
                dst[2 * j + 1][0] = v.z, dst[2 * j + 1][1] = v.w;
            } else {
                dst[2 * j][0] = half ? v.y : v.x;
                dst[2 * j + 1][0] = half ? v.w : v.z;
            }
        }
    };
    if constexpr (F::nib) {
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            if constexpr (NT == 2) {
                const uint4 v = ld4(ks * 1024 + lane * 16, so);
                s.qn[ks][0] = make_uint2(v.x, v.y);
                s.qn[ks][1] = make_uint2(v.z, v.w);
            } else {
                s.qn[ks][0] = __builtin_bit_cast(
                    uint2, __builtin_amdgcn_raw_buffer_load_b64(wr, ks * 1024 + lane * 16 + 8 * half, so, 0));
            }
        }
    } else {
        pairs(0, s.q2);
    }
    if constexpr (FMT == T_Q6_K) {
        pairs(F::QA, s.hb);
    } else if constexpr (F::QB > 0) {
        const uint4 v = ld4(F::QA + lane * 16, so);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) s.hb[ks][nt] = w[ks];
    }
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int row = 16 * (NT == 2 ? nt : half) + r16;
        if constexpr (F::mins) {
            s.sc[nt] = ld4(F::SC + row * 16, so);
            s.d[nt] = __builtin_amdgcn_raw_buffer_load_b32(wr, F::D + row * 4, so, 0);
            if constexpr (FMT == T_Q2_K)
                s.sw[nt] = __builtin_amdgcn_raw_buffer_load_b32(wr, F::SC + row * 16 + 4 * g, so, 0);
        } else {
            s.sc[nt].x = __builtin_amdgcn_raw_buffer_load_b32(wr, F::SC + row * 16 + 4 * g, so, 0);
            s.d[nt] = __builtin_amdgcn_raw_buffer_load_b32(wr, F::D + (row >> 1) * 4, so, 0);
        }
    }
}

// The loads sk_load_w issues for two n tiles.
template <uint32_t FMT>
__host__ __device__ constexpr int sk_loads() {
    return (KS<FMT>::nib ? 4 : 2) + (FMT == T_Q6_K ? 2 : KS<FMT>::QB > 0 ? 1 : 0) + (FMT == T_Q2_K ? 6 : 4);
}

// Wait until at most N of the wave's memory operations are in flight.
template <int N>
__device__ inline void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt field");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// The same, and until its LDS reads have returned: what a wave has to wait for
// before a bare s_barrier after which others overwrite what it has read.
template <int N>
__device__ inline void wait_vm_lds() {
    static_assert(N >= 0 && N < 64, "vmcnt field");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// The stored quants of K-step ks, n tile nt (16 slots, byte b of word i = slot
// 4 i + b).
template <uint32_t FMT, int NT>
__device__ inline void sk_quants(const SKRaw<FMT, NT> &s, int ks, int nt, int half, uint32_t (&q)[4]) {
    const uint32_t m4 = 0x0F0F0F0Fu, m2 = 0x03030303u, m1 = 0x01010101u;
    if constexpr (KS<FMT>::nib) {
        const uint2 w = s.qn[ks][nt];
        q[0] = w.x & m4;
        q[1] = w.y & m4;
        q[2] = (w.x >> 4) & m4;
        q[3] = (w.y >> 4) & m4;
    } else {
#pragma unroll
        for (int t = 0; t < 4; t++) q[t] = (s.q2[ks][nt] >> (2 * t)) & m2;
    }
    if constexpr (FMT == T_Q6_K) {
        const uint32_t H = s.hb[ks][nt];
        q[0] |= (H << 4) & 0x30303030u;
        q[1] |= (H << 2) & 0x30303030u;
        q[2] |= H & 0x30303030u;
        q[3] |= (H >> 2) & 0x30303030u;
    }
    if constexpr (FMT == T_Q5_K || FMT == T_Q3_K) {
        // slot word t's bits at bit t + 4 (n tile) of each byte
        const uint32_t Fw = NT == 2 ? s.hb[ks][nt] : s.hb[ks][nt] >> (4 * half);
        constexpr int pos = FMT == T_Q5_K ? 4 : 2;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int sh = t + (NT == 2 ? 4 * nt : 0) - pos;
            q[t] |= (sh >= 0 ? Fw >> sh : Fw << -sh) & (m1 << pos);
        }
    }
}

__device__ inline uint32_t sk_mul16(uint32_t a, uint32_t b) {  // two 16-bit products
    return __builtin_bit_cast(uint32_t, (u16x2b_t)(__builtin_bit_cast(u16x2b_t, a) * __builtin_bit_cast(u16x2b_t, b)));
}
__device__ inline uint32_t sk_mad16(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, (u16x2b_t)(__builtin_bit_cast(u16x2b_t, a) * __builtin_bit_cast(u16x2b_t, b) +
                                                   __builtin_bit_cast(u16x2b_t, c)));
}

template <uint32_t FMT>
constexpr bool sk_two() {  // two operands per K-step
    return FMT == T_Q4_K || FMT == T_Q5_K || FMT == T_Q6_K;
}

// The decoded operands of a super-block.
template <uint32_t FMT, int NT>
struct SKOps {
    v4i2_t lo[4][NT], hi[sk_two<FMT>() ? 4 : 1][NT];
    v8h2_t mn[NT];  // min operand (f16, groups 8 g .. + 7 in lane groups 0 and 1, zeros in 2 and 3)
    float d[NT], dm[NT];
};

template <uint32_t FMT, int NT>
__device__ inline void sk_decode(const SKRaw<FMT, NT> &s, int half, int lane, SKOps<FMT, NT> &o) {
    const int g = lane >> 4, r16 = lane & 15;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        if constexpr (FMT == T_Q4_K || FMT == T_Q5_K) {
            // this lane's units 2 ks + g / 2: scale bytes ks of word x or z
            const uint32_t sw = g & 2 ? s.sc[nt].z : s.sc[nt].x;
            const uint32_t shw = (sw >> 3) & 0x07070707u, slw = sw & 0x07070707u;
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                uint32_t q[4];
                sk_quants<FMT, NT>(s, ks, nt, half, q);
                const uint32_t sel = 0x0c000c00u | ks | (ks << 16);
                const uint32_t sh = __builtin_amdgcn_perm(0, shw, sel), sl = __builtin_amdgcn_perm(0, slw, sel);
                constexpr uint32_t flip = FMT == T_Q5_K ? 0x80808080u : 0u;
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    o.hi[ks][nt][t] = (int)(sk_mul16(q[t], sh) ^ flip);
                    o.lo[ks][nt][t] = (int)(sk_mul16(q[t], sl) ^ flip);
                }
            }
            // mins of units 4 (g % 2) .. + 3 as f16, each twice (two groups
            // per unit): units 0 2 4 6 are bytes 0..3 of word y, 1 3 5 7 of w
            const uint32_t sel0 = g & 1 ? 2 : 0;
            uint32_t p[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t w = u & 1 ? s.sc[nt].w : s.sc[nt].y;
                const uint32_t byte = sel0 + (u >> 1);
                const uint32_t m = __builtin_amdgcn_perm(0, w, 0x0c000c00u | byte | (byte << 16));
                const _Float16 one = (_Float16)(float)(m & 0xffu);
                const uint32_t h = __builtin_bit_cast(uint16_t, one);
                p[u] = g < 2 ? h | (h << 16) : 0u;
            }
            o.mn[nt] = __builtin_bit_cast(v8h2_t, make_uint4(p[0], p[1], p[2], p[3]));
        } else if constexpr (FMT == T_Q2_K) {
            // group 4 ks + g at byte ks of word g: scale low, min high nibble
            const uint32_t sl4 = s.sw[nt] & 0x0F0F0F0Fu;
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                uint32_t q[4];
                sk_quants<FMT, NT>(s, ks, nt, half, q);
                const uint32_t sl = __builtin_amdgcn_perm(0, sl4, 0x0c000c00u | ks | (ks << 16));
#pragma unroll
                for (int t = 0; t < 4; t++) o.lo[ks][nt][t] = (int)sk_mul16(q[t], sl);
            }
            // mins of groups 8 g + e = 4 (2 g + e / 4) + e % 4: byte 2 g + e / 4 of word e % 4
            uint32_t p[4];
#pragma unroll
            for (int e2 = 0; e2 < 4; e2++) {
                const uint32_t w0 = e2 & 1 ? s.sc[nt].z : s.sc[nt].x, w1 = e2 & 1 ? s.sc[nt].w : s.sc[nt].y;
                const uint32_t byte = 2 * (g & 1) + (e2 >> 1);
                const _Float16 h0 = (_Float16)(float)((w0 >> (8 * byte + 4)) & 15u);
                const _Float16 h1 = (_Float16)(float)((w1 >> (8 * byte + 4)) & 15u);
                p[e2] = g < 2 ? (uint32_t)__builtin_bit_cast(uint16_t, h0) |
                                    ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16)
                              : 0u;
            }
            o.mn[nt] = __builtin_bit_cast(v8h2_t, make_uint4(p[0], p[1], p[2], p[3]));
        } else {
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                uint32_t q[4];
                sk_quants<FMT, NT>(s, ks, nt, half, q);
                const uint32_t sv = (uint32_t)sbfe8(s.sc[nt].x, 8u * (uint32_t)ks) & 0xffffu;
                const uint32_t s2 = sv | (sv << 16);  // the scale in both halves
                uint32_t f, a;
                if constexpr (FMT == T_Q6_K) {  // 2 s q + 128 - 64 s
                    f = sk_mul16(s2, 0x00020002u);
                    a = sk_mad16(s2, 0xffc0ffc0u, 0x00800080u);
                } else {  // 4 s - s q
                    f = sk_mul16(s2, 0xffffffffu);
                    a = sk_mul16(s2, 0x00040004u);
                }
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const uint32_t e = q[t] & 0x00ff00ffu, od = (q[t] >> 8) & 0x00ff00ffu;
                    const uint32_t ve = sk_mad16(e, f, a), vo = sk_mad16(od, f, a);
                    // bytes of slots 4 t .. + 3: low bytes of ve, vo interleaved
                    const uint32_t lo = __builtin_amdgcn_perm(vo, ve, 0x06020400u);
                    if constexpr (FMT == T_Q6_K) {
                        o.lo[ks][nt][t] = (int)(lo ^ 0x80808080u);
                        o.hi[ks][nt][t] = (int)__builtin_amdgcn_perm(vo, ve, 0x07030501u);
                    } else {
                        o.lo[ks][nt][t] = (int)lo;
                    }
                }
            }
        }
        if constexpr (KS<FMT>::mins) {
            o.d[nt] = half_to_float(s.d[nt] & 0xffffu);
            o.dm[nt] = -half_to_float(s.d[nt] >> 16);
        } else {
            const float d = half_to_float((s.d[nt] >> (16 * (r16 & 1))) & 0xffffu);
            o.d[nt] = FMT == T_Q6_K ? 0.5f * d : -d;
        }
    }
}

// An m tile's activations of one super-block.
struct SKAct {
    v4i2_t a[4];
    v8h2_t bs;   // group sums 8 (g % 2) .. + 7 of row l % 16
    float4 dx;   // block scales of rows 4 g .. + 3
    v4i2_t sx;   // 1152 times their quant sums (Q5_K)
};

template <uint32_t FMT>
__device__ inline void sk_load_x(__amdgpu_buffer_rsrc_t xr, int rec, int lane, SKAct &s) {
    const int g = lane >> 4, r16 = lane & 15;
    const int so = __builtin_amdgcn_readfirstlane(rec) * g2_rec_bytes(16);
#pragma unroll
    for (int ks = 0; ks < 4; ks++) s.a[ks] = __builtin_bit_cast(v4i2_t, ks_ld4(xr, lane * 16, so + ks * 1024));
    if constexpr (KS<FMT>::mins)
        s.bs = __builtin_bit_cast(v8h2_t, ks_ld4(xr, g2_rec_bsum(16) + r16 * 32 + (g & 1) * 16, so));
    s.dx = __builtin_bit_cast(float4, ks_ld4(xr, g2_rec_dx(16) + g * 16, so));
    if constexpr (FMT == T_Q5_K) s.sx = __builtin_bit_cast(v4i2_t, ks_ld4(xr, g2_rec_sx(16) + g * 16, so));
}

template <uint32_t FMT, int NT>
__device__ inline void sk_compute(const SKOps<FMT, NT> &o, const SKAct &s, v4f2_t (&y)[NT]) {
    const v4i2_t zi = {0, 0, 0, 0};
    const v4f2_t zf = {0.0f, 0.0f, 0.0f, 0.0f};
    v4f2_t t[NT];
    if constexpr (KS<FMT>::mins) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++) t[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.bs, o.mn[nt], zf, 0, 0, 0);
    }
    v4i2_t h[NT], l[NT];
#pragma unroll
    for (int ks = 0; ks < 4; ks++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            l[nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(s.a[ks], o.lo[ks][nt], ks ? l[nt] : FMT == T_Q5_K ? s.sx : zi, 0, 0, 0);
            if constexpr (sk_two<FMT>())
                h[nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(s.a[ks], o.hi[ks][nt], ks ? h[nt] : zi, 0, 0, 0);
        }
    const float dxv[4] = {s.dx.x, s.dx.y, s.dx.z, s.dx.w};
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            int S = l[nt][i];
            if constexpr (FMT == T_Q6_K) S += 256 * h[nt][i];
            else if constexpr (sk_two<FMT>()) S += 8 * h[nt][i];
            float u;
            if constexpr (KS<FMT>::mins)
                u = fma_f32(o.d[nt], (float)S, o.dm[nt] * t[nt][i]);
            else
                u = o.d[nt] * (float)S;
            y[nt][i] = fma_f32(dxv[i], u, y[nt][i]);
        }
}

// LDS of a launch: the waves' partial tiles.
__host__ __device__ constexpr int sk_lds_bytes(int MT, int NT, int KW) { return KW * MT * NT * 1024; }

template <uint32_t FMT, int MT, int NT, int KW>
__device__ inline void sk_body(const GSKArgs &A, const GSKSeg &sg, int t, float *lds) {
    // XCD-aware order: workgroups go round-robin over the 8 XCDs, so the m
    // blocks of one n block, which read the same weights, are consecutive
    // workgroups of one XCD
    const int q = t >> 3, mblk = q % A.MB, nblk = q / A.MB * 8 + (t & 7);
    if (nblk >= sg.nblk) return;
    const int half = NT == 2 ? 0 : nblk & 1;  // n tile of the 32-row block
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(sg.w + (int64_t)(NT == 2 ? nblk : nblk >> 1) * A.nb * KS<FMT>::chunk), (short)0, A.nb * KS<FMT>::chunk, 0x00020000);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(A.x + (int64_t)mblk * MT * A.nb * g2_rec_bytes(16)), (short)0,
        MT * A.nb * g2_rec_bytes(16), 0x00020000);
    v4f2_t y[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) y[mt][nt] = (v4f2_t){0.0f, 0.0f, 0.0f, 0.0f};
    if (wave < A.nb) {
        // the next super-block's weights and activations are loaded into the
        // same registers as soon as these are used; loads past the wave's
        // last super-block read it again (nothing computes them), so every
        // load is unconditional
        SKRaw<FMT, NT> raw;
        SKAct act[MT];
        // keep the order of issue: loads retire in it, and the first decode
        // waits for its weights alone
        auto fence = [] {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
        sk_load_w<FMT, NT>(wr, wave, half, lane, raw);
        fence();
#pragma unroll
        for (int mt = 0; mt < MT; mt++) sk_load_x<FMT>(xr, mt * A.nb + wave, lane, act[mt]);
        fence();
        for (int c = wave; c < A.nb; c += KW) {
            const int cn = c + KW < A.nb ? c + KW : c;
            SKOps<FMT, NT> o;
            sk_decode<FMT, NT>(raw, half, lane, o);
            sk_load_w<FMT, NT>(wr, cn, half, lane, raw);
            fence();
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                sk_compute<FMT, NT>(o, act[mt], y[mt]);
                sk_load_x<FMT>(xr, mt * A.nb + cn, lane, act[mt]);
                fence();
            }
        }
    }
    // the waves' partial tiles in register order: float (NT mt + nt) 256 +
    // 64 i + l of wave w's 256 NT MT floats
    float *const pw = lds + wave * (MT * NT * 256) + lane;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int i = 0; i < 4; i++) pw[((NT * mt + nt) * 4 + i) * 64] = y[mt][nt][i];
    __syncthreads();
    // four consecutive floats of the tile per thread, added in wave order:
    // one row, four columns
    for (int k = (int)threadIdx.x * 4; k < MT * NT * 256; k += KW * 256) {
        float4 v = *reinterpret_cast<const float4 *>(lds + k);
#pragma unroll
        for (int w = 1; w < KW; w++) {
            const float4 p = *reinterpret_cast<const float4 *>(lds + w * (MT * NT * 256) + k);
            v.x += p.x, v.y += p.y, v.z += p.z, v.w += p.w;
        }
        const int l = k & 63, i = (k >> 6) & 3, tile = k >> 8;
        const int64_t m = (int64_t)(mblk * MT + tile / NT) * 16 + 4 * (l >> 4) + i;
        const int64_t n = (int64_t)nblk * (16 * NT) + 16 * (tile % NT) + (l & 15);
        if (m >= A.M) continue;
        float *const dst = sg.y + m * sg.ldy + n;
        if (n + 3 < sg.n_out && ((uintptr_t)dst & 15) == 0) {
            *reinterpret_cast<float4 *>(dst) = v;
        } else {
            const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (n + j < sg.n_out) dst[j] = e[j];
        }
    }
}

// Grid: per segment ceil(nblk / 8) * 8 * MB workgroups of KW waves; dynamic
// LDS sk_lds_bytes(MT, NT, KW).
template <uint32_t F0, uint32_t F1, int MT, int NT, int KW>
__global__ __launch_bounds__(64 * KW)
__attribute__((amdgpu_waves_per_eu(2))) void gemmsk_kernel(GSKArgs A) {
    extern __shared__ __attribute__((aligned(16))) float sk_lds[];
    const int b = (int)blockIdx.x;
    GSKSeg sg = A.seg[0];
#pragma unroll
    for (int k = 1; k < kSKMaxSegs; k++)
        if (k < A.nseg && b >= A.seg[k].wg0) sg = A.seg[k];
    if constexpr (F0 == F1) {
        sk_body<F0, MT, NT, KW>(A, sg, b - sg.wg0, sk_lds);
    } else {
        if (sg.type == F0)
            sk_body<F0, MT, NT, KW>(A, sg, b - sg.wg0, sk_lds);
        else
            sk_body<F1, MT, NT, KW>(A, sg, b - sg.wg0, sk_lds);
    }
}

}  // namespace sihip
