// GEMM for prompts of F16 weights and of the formats that pair with Q8_0
// activations (Q4_0, Q5_0, Q8_0), for a group of matrices of one format that
// share X: Y_i[M x n_out_i] = X[M x n_in] * W_i^T, each output within the
// tolerance of the reference dot (reference kernels.c:189-247). The weight
// copies, the activation records and the arithmetic of a block are those of
// gemmh.h and gemmq.h.
//
// Tiles as in gemmx.h: a workgroup of 4 waves computes BM = 16 MT activation
// rows against 128 weight rows, wave w rows 32 w .. 32 w + 31; the matrices of
// the group are segments of one grid, and K slices split a tile's steps over
// several workgroups where the tiles alone leave CUs idle.
//
// What bounds it: at few rows the memory round trips, as a step is 16 to 48
// MFMAs per wave, a fraction of a microsecond, and one step of loads ahead does
// not cover one; at more rows the LDS reads of the activations (F16, 0.12 us
// per m tile and step) or the epilogue's 12 VALU instructions per MFMA (Q8_0
// pairs, 0.26 us). Layer of 7 matrices, four groups called one after another, us on
// the kernels of gemmh.h and gemmq.h -> here: 1.1B F16 M = 40 61 -> 42, M = 200
// 120 -> 68, M = 500 202 -> 98; Q8_0 M = 200 148 -> 91, 0.5B M = 300 98 -> 72;
// Q5_0 M = 64 82 -> 61. The records of the next gd_ring(MT) - 1 steps are copied
// to LDS by DMA and the weights of the next gd_wdepth(MT) are loaded into
// registers; each
// step waits for its own record by count and meets the other waves at a bare
// s_barrier. The ring is at least as deep as the weights run ahead: loads
// retire in order, and a record must not wait for weights of later steps.
#pragma once

#include "gemmh.h"
#include "gemmq.h"
#include "gemmx.h"

namespace sihip {

struct GDSeg {
    const uint8_t *w;     // weight chunks of whole 128-row blocks
    float *y;             // Y[m * ldy + n]
    int64_t ldy, n_out;
    int nb0;              // the segment's first n block (128 rows) in the grid
};

struct GDArgs {
    const uint8_t *x;     // activation records [MB][nk]
    int64_t M;
    int nk, MB, NB;       // steps; m blocks of BM rows; n blocks of 128 rows (all segments)
    int S, SBK;           // K slices, steps per slice
    float *part;
    uint32_t *cnt;
    int nseg;
    GDSeg seg[kG2MaxSegs];
};

template <uint32_t FMT>
__host__ __device__ constexpr int gd_rec_bytes(int BM) {
    return FMT == T_F16 ? gh_rec_bytes(BM) : gq_rec_bytes(BM);
}

// Two workgroups per CU share 160 KiB of LDS and leave 256 VGPRs per wave. Weights
// run three steps ahead, or two: with four m tiles of the Q8_0 pairs three unroll a
// round of 12 steps (Q8_0 63 KB of code, with two 25 KB) and take 184 VGPRs (146,
// which leave three waves per SIMD). Gate + up in Q8_0, 9344 rows of 2816 at M =
// 1234 242 -> 208 us, 16000 of 3712 at M = 510 217 -> 193; Q4_0 and Q5_0 1%.
template <uint32_t FMT>
__host__ __device__ constexpr int gd_ring(int MT) {
    return FMT == T_F16 && MT > 4 ? 3 : 4;
}
template <uint32_t FMT>
__host__ __device__ constexpr int gd_wdepth(int MT) {
    return MT <= (FMT == T_F16 ? 4 : 3) ? 3 : 2;
}

// A lane's weights of one step: two 16-row n tiles.
template <uint32_t FMT>
struct GDRaw {
    v8hh_t h[FMT == T_F16 ? 4 : 1][2];   // F16: [K-step][nt]
    uint2 q8[FMT == T_Q8_0 ? 4 : 1][2];  // Q8_0: [block][nt]
    uint4 nib[2];                        // Q4_0/Q5_0: [nt], word per block
    uint32_t hb[2];                      // Q5_0: [nt], the fifth bits of the 4 blocks
    float4 d[2];                         // [nt], d of the lane's row for the 4 blocks
};

template <uint32_t FMT>
__host__ __device__ constexpr int gd_loads() {
    return FMT == T_F16 ? 8 : FMT == T_Q8_0 ? 10 : FMT == T_Q5_0 ? 6 : 4;
}

template <uint32_t FMT>
__device__ inline void gd_load_w(__amdgpu_buffer_rsrc_t wr, int so, int lane, GDRaw<FMT> &o) {
    if constexpr (FMT == T_F16) {
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
#pragma unroll
            for (int nt = 0; nt < 2; nt++)
                o.h[ks][nt] = __builtin_bit_cast(
                    v8hh_t, __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16, so + (2 * ks + nt) * 1024, 0));
        return;
    }
    if constexpr (FMT == T_Q8_0) {
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int nt = 0; nt < 2; nt++)
                o.q8[j][nt] = __builtin_bit_cast(
                    uint2, __builtin_amdgcn_raw_buffer_load_b64(wr, lane * 8, so + (2 * j + nt) * 512, 0));
    } else {
#pragma unroll
        for (int nt = 0; nt < 2; nt++)
            o.nib[nt] = __builtin_bit_cast(
                uint4, __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16, so + nt * 1024, 0));
        if constexpr (FMT == T_Q5_0) {
#pragma unroll
            for (int nt = 0; nt < 2; nt++)
                o.hb[nt] = __builtin_amdgcn_raw_buffer_load_b32(wr, lane * 4, so + kGQHigh + nt * 256, 0);
        }
    }
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
        o.d[nt] = __builtin_bit_cast(
            float4, __builtin_amdgcn_raw_buffer_load_b128(wr, (lane & 15) * 16, so + gq_d_off<FMT>() + nt * 256, 0));
}

// The MFMA operand (8 quants) of block j, n tile nt.
template <uint32_t FMT>
__device__ inline long gd_operand(const GDRaw<FMT> &o, int j, int nt) {
    if constexpr (FMT == T_Q8_0) {
        return __builtin_bit_cast(long, o.q8[j][nt]);
    } else {
        const uint32_t w = j == 0 ? o.nib[nt].x : j == 1 ? o.nib[nt].y : j == 2 ? o.nib[nt].z : o.nib[nt].w;
        uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
        if constexpr (FMT == T_Q5_0) {
            lo |= (o.hb[nt] >> j) & 0x10101010u;
            hi |= (o.hb[nt] << (4 - j)) & 0x10101010u;
        }
        return __builtin_bit_cast(long, make_uint2(lo, hi));
    }
}

// Sums per output, added at the end. Unsliced rows are long chains of f32
// additions, so F16 sums a step by itself before it joins, and the Q8_0 pairs
// keep the two halves of a step apart (error against 64-bit sums, F16 M = 200
// of the 1.1B shapes: 3.4e-7 in one chain, 1.2e-7 so; 0.5B Q8_0 M = 300: 1.2e-7
// and 8.9e-8).
template <uint32_t FMT>
__host__ __device__ constexpr int gd_sums() { return FMT == T_F16 ? 1 : 2; }

// One step against the record X of the m block.
template <uint32_t FMT, int MT>
__device__ inline void gd_compute(const GDRaw<FMT> &o, const uint8_t *X, int lane, v4f2_t (&y)[gd_sums<FMT>()][MT][2]) {
    constexpr int BM = 16 * MT;
    const int g = lane >> 4;
    if constexpr (FMT == T_F16) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            v4f2_t t[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const v8hh_t a = *reinterpret_cast<const v8hh_t *>(X + (4 * mt + ks) * 1024 + lane * 16);
#pragma unroll
                for (int nt = 0; nt < 2; nt++)
                    t[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, o.h[ks][nt], t[nt], 0, 0, 0);
            }
            y[0][mt][0] += t[0];
            y[0][mt][1] += t[1];
        }
    } else {
        constexpr int bias = FMT == T_Q4_0 ? 8 : FMT == T_Q5_0 ? 16 : 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const long b0 = gd_operand<FMT>(o, j, 0), b1 = gd_operand<FMT>(o, j, 1);
            const float dw0 = j == 0 ? o.d[0].x : j == 1 ? o.d[0].y : j == 2 ? o.d[0].z : o.d[0].w;
            const float dw1 = j == 0 ? o.d[1].x : j == 1 ? o.d[1].y : j == 2 ? o.d[1].z : o.d[1].w;
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const long a = *reinterpret_cast<const long *>(X + (4 * mt + j) * 512 + lane * 8);
                const int off = (j * BM + 16 * mt + 4 * g) * 4;
                v4iq_t cb = {0, 0, 0, 0};
                if constexpr (bias != 0) cb = *reinterpret_cast<const v4iq_t *>(X + gq_rec_bs(BM) + off);
                const v4iq_t s0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b0, cb, 0, 0, 0);
                const v4iq_t s1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b1, cb, 0, 0, 0);
                const float4 dx = *reinterpret_cast<const float4 *>(X + gq_rec_dx(BM) + off);
                const float dxv[4] = {dx.x, dx.y, dx.z, dx.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    y[j >> 1][mt][0][i] = fma_f32((float)s0[i], dw0 * dxv[i], y[j >> 1][mt][0][i]);
                    y[j >> 1][mt][1][i] = fma_f32((float)s1[i], dw1 * dxv[i], y[j >> 1][mt][1][i]);
                }
            }
        }
    }
}

template <uint32_t FMT, int MT>
__global__ __launch_bounds__(kG2Threads)
__attribute__((amdgpu_waves_per_eu(2))) void gemmd_kernel(GDArgs A) {
    constexpr int R = gd_ring<FMT>(MT), DW = gd_wdepth<FMT>(MT);
    constexpr int BM = 16 * MT, kRec = gd_rec_bytes<FMT>(BM);
    // whole KiBs, one wave instruction each, the same number per wave; the
    // last may read into the next record (zero past the buffer), into LDS
    // that no step reads
    constexpr int kPieces = (kRec + 1023) / 1024, kD = (kPieces + 3) / 4;
    constexpr int kSlot = kPieces * 1024;
    // distinct LDS objects, as in gemmx.h
    __shared__ __attribute__((aligned(16))) uint8_t s0[kSlot];
    __shared__ __attribute__((aligned(16))) uint8_t s1[kSlot];
    __shared__ __attribute__((aligned(16))) uint8_t s2[kSlot];
    __shared__ __attribute__((aligned(16))) uint8_t s3[R > 3 ? kSlot : 16];
    const int b = blockIdx.x;
    const int xcd = b & 7, t = b >> 3;
    const int per = A.MB * A.S;
    const int nblk = (t / per) * 8 + xcd, rest = t % per;
    const int slice = rest / A.MB, mblk = rest % A.MB;
    if (nblk >= A.NB) return;
    GDSeg sg = A.seg[0];
#pragma unroll
    for (int k = 1; k < kG2MaxSegs; k++)
        if (k < A.nseg && nblk >= A.seg[k].nb0) sg = A.seg[k];
    auto slot = [&](auto u) -> uint8_t * {
        constexpr int k = decltype(u)::value % R;
        return k == 0 ? s0 : k == 1 ? s1 : k == 2 ? s2 : s3;
    };
    const int lblk = nblk - sg.nb0;
    const int c0 = slice * A.SBK;
    const int c1 = c0 + A.SBK < A.nk ? c0 + A.SBK : A.nk;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
    // F16: the chunks of a 32-row block one after another; the others: those of
    // the four 32-row blocks side by side
    constexpr int kChunk = FMT == T_F16 ? kGHChunk : gq_chunk<FMT == T_F16 ? T_Q8_0 : FMT>();
    constexpr int kStep = FMT == T_F16 ? kChunk : 4 * kChunk;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(sg.w + (FMT == T_F16 ? (int64_t)(lblk * 4 + wave) * A.nk * kChunk
                                      : (int64_t)lblk * A.nk * 4 * kChunk + wave * kChunk)),
        (short)0, FMT == T_F16 ? A.nk * kChunk : A.nk * 4 * kChunk - wave * kChunk, 0x00020000);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(A.x + (int64_t)mblk * A.nk * kRec), (short)0, A.nk * kRec, 0x00020000);
    auto dma = [&](int c, uint8_t *dst) {
#pragma unroll
        for (int k = 0; k < kD; k++) {
            const int i = wave + 4 * k < kPieces ? wave + 4 * k : kPieces - 1;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                xr, (__attribute__((address_space(3))) void *)(dst + i * 1024), 16, lane * 16,
                c * kRec + i * 1024, 0, 0);
        }
    };
    auto fence = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto clamp = [&](int c) { return c < c1 ? c : c1 - 1; };
    v4f2_t ys[gd_sums<FMT>()][MT][2];
#pragma unroll
    for (int k = 0; k < gd_sums<FMT>(); k++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int nt = 0; nt < 2; nt++) ys[k][mt][nt] = (v4f2_t){0.0f, 0.0f, 0.0f, 0.0f};
    GDRaw<FMT> raw[DW];
    gx_unroll<(R - 1 > DW ? R - 1 : DW)>([&](auto i) {
        if constexpr (i < R - 1) dma(clamp(c0 + i), slot(i));
        fence();
        if constexpr (i < DW) gd_load_w<FMT>(wr, clamp(c0 + i) * kStep, lane, raw[i]);
        fence();
    });
    constexpr int kW = gd_loads<FMT>();
    auto step = [&](int c, auto younger, const uint8_t *X, uint8_t *Xn, GDRaw<FMT> &rw) {
        // the record has arrived, and this wave's reads of the slot before have
        // returned, which the copy below overwrites
        wait_vm_lds<decltype(younger)::value>();
        __builtin_amdgcn_s_barrier();
        fence();
        dma(clamp(c + R - 1), Xn);
        fence();
        gd_compute<FMT, MT>(rw, X, lane, ys);
        gd_load_w<FMT>(wr, clamp(c + DW) * kStep, lane, rw);
        fence();
    };
    // ring slot and weight set static: whole rounds without conditions, then
    // the last partial round
    constexpr int U = R % DW == 0 ? R : R * DW;
    int c = c0;
    auto run = [&](auto u, auto last) {
        constexpr int v = decltype(u)::value, kY = gx_younger(R, DW, kD, kW, U, decltype(last)::value ? v : -1);
        step(c + v, std::integral_constant<int, kY>(), slot(u), slot(std::integral_constant<int, (v + R - 1) % R>()),
             raw[v % DW]);
    };
    for (; c + U <= c1; c += U) gx_unroll<U>([&](auto u) { run(u, std::false_type()); });
    gx_unroll<U - 1>([&](auto u) {
        if (c + u < c1) run(u, std::true_type());
    });
    v4f2_t(&y)[MT][2] = ys[0];
    if constexpr (gd_sums<FMT>() == 2) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int nt = 0; nt < 2; nt++) y[mt][nt] += ys[1][mt][nt];
    }
    wait_vm<0>();  // no copy may land in the LDS of a workgroup that has ended
    const int64_t n0 = (int64_t)lblk * kG2BN + 32 * wave;
    const int64_t m0 = (int64_t)mblk * BM;
    if (A.S == 1) {
        const bool full = n0 + 32 <= sg.n_out && m0 + BM <= A.M;
#pragma unroll
        for (int nt = 0; nt < 2; nt++) {
            const int64_t n = n0 + 16 * nt + r16;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int64_t m = m0 + 16 * mt + 4 * g + i;
                    if (full || (m < A.M && n < sg.n_out)) sg.y[m * sg.ldy + n] = y[mt][nt][i];
                }
        }
        return;
    }
    const int64_t per_slice = (int64_t)A.MB * A.NB * (BM * kG2BN);
    float *const pt = A.part + ((int64_t)mblk * A.NB + nblk) * (BM * kG2BN);
    g2_store_partial<MT>(pt + slice * per_slice, wave, lane, y, 1.0f, A.M - m0);
    g2_slices_finish<MT>(pt, per_slice, A.cnt + (int64_t)mblk * A.NB + nblk, A.S, m0, A.M,
                         (int64_t)lblk * kG2BN, sg.n_out, sg.y, sg.ldy);
}

// ---- small products ------------------------------------------------------------
//
// Where the 128-row tiles are too few for the CUs, the work of a workgroup is
// cut as in gemmsk.h: 32 weight rows and 16 MT activation rows, whose steps
// the four waves split among themselves (wave w takes c = w, w + 4, ...), each
// reading both operands straight into registers, gds_depth steps ahead; the
// waves' partial tiles meet once in LDS.
constexpr int kGDSWaves = 4;

struct GDSSeg {
    const uint8_t *w;
    float *y;
    int64_t ldy, n_out;
    int nblk;             // blocks of 32 rows
    int wg0;              // first workgroup of the segment (a multiple of 8)
};

struct GDSArgs {
    const uint8_t *x;     // activation records [16-row block][nk]
    int64_t M;
    int nk, MB;           // steps; m blocks of 16 MT rows
    int nseg;
    GDSSeg seg[kG2MaxSegs];
};

// A lane's operands of one step of a 16-row m tile.
template <uint32_t FMT>
struct GDSAct {
    v8hh_t a[FMT == T_F16 ? 4 : 1];                       // F16: [K-step]
    long q[FMT == T_F16 ? 1 : 4];                         // [block]
    float4 dx[FMT == T_F16 ? 1 : 4];                      // [block], rows 4 g .. 4 g + 3
    v4iq_t bs[FMT == T_Q4_0 || FMT == T_Q5_0 ? 4 : 1];    // the MFMA's C input
};

// rec: the record's offset in bytes.
template <uint32_t FMT>
__device__ inline void gds_load_x(__amdgpu_buffer_rsrc_t xr, int rec, int lane, GDSAct<FMT> &s) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if constexpr (FMT == T_F16) {
            s.a[j] = __builtin_bit_cast(
                v8hh_t, __builtin_amdgcn_raw_buffer_load_b128(xr, lane * 16, rec + j * 1024, 0));
        } else {
            s.q[j] = __builtin_bit_cast(
                long, __builtin_amdgcn_raw_buffer_load_b64(xr, lane * 8, rec + j * 512, 0));
            s.dx[j] = __builtin_bit_cast(
                float4, __builtin_amdgcn_raw_buffer_load_b128(xr, (lane >> 4) * 16, rec + gq_rec_dx(16) + j * 64, 0));
            if constexpr (FMT != T_Q8_0)
                s.bs[j] = __builtin_bit_cast(
                    v4iq_t, __builtin_amdgcn_raw_buffer_load_b128(xr, (lane >> 4) * 16, rec + gq_rec_bs(16) + j * 64, 0));
        }
    }
}

template <uint32_t FMT>
__device__ inline void gds_compute(const GDRaw<FMT> &o, const GDSAct<FMT> &s, v4f2_t (&y)[2]) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
#pragma unroll
        for (int nt = 0; nt < 2; nt++) {
            if constexpr (FMT == T_F16) {
                y[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.a[j], o.h[j][nt], y[nt], 0, 0, 0);
            } else {
                const float4 d = o.d[nt];
                const float dw = j == 0 ? d.x : j == 1 ? d.y : j == 2 ? d.z : d.w;
                v4iq_t cb = {0, 0, 0, 0};
                if constexpr (FMT != T_Q8_0) cb = s.bs[j];
                const v4iq_t r = __builtin_amdgcn_mfma_i32_16x16x32_i8(s.q[j], gd_operand<FMT>(o, j, nt), cb, 0, 0, 0);
                const float dxv[4] = {s.dx[j].x, s.dx[j].y, s.dx[j].z, s.dx[j].w};
#pragma unroll
                for (int i = 0; i < 4; i++) y[nt][i] = fma_f32((float)r[i], dw * dxv[i], y[nt][i]);
            }
        }
    }
}

// Steps of both operands in registers, as many as leave two waves per SIMD.
template <uint32_t FMT>
__host__ __device__ constexpr int gds_depth(int MT) {
    const int w = FMT == T_F16 ? 32 : FMT == T_Q8_0 ? 24 : 18;
    const int x = FMT == T_F16 ? 16 : FMT == T_Q8_0 ? 24 : 40;
    return w + MT * x <= 48 ? 3 : w + MT * x <= 96 ? 2 : 1;
}

template <uint32_t FMT, int MT>
__global__ __launch_bounds__(64 * kGDSWaves)
__attribute__((amdgpu_waves_per_eu(2))) void gemmds_kernel(GDSArgs A) {
    constexpr int KW = kGDSWaves, kTile = 512 * MT;  // floats of the output tile
    __shared__ __attribute__((aligned(16))) float sk_lds[KW * kTile];
    constexpr int D = gds_depth<FMT>(MT);
    const int b = (int)blockIdx.x;
    GDSSeg sg = A.seg[0];
#pragma unroll
    for (int k = 1; k < kG2MaxSegs; k++)
        if (k < A.nseg && b >= A.seg[k].wg0) sg = A.seg[k];
    // XCD-aware order, as in gemmsk.h
    const int t = b - sg.wg0, q = t >> 3, mblk = q % A.MB, nblk = q / A.MB * 8 + (t & 7);
    if (nblk >= sg.nblk) return;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    constexpr int kChunk = FMT == T_F16 ? kGHChunk : gq_chunk<FMT == T_F16 ? T_Q8_0 : FMT>();
    constexpr int kStep = FMT == T_F16 ? kChunk : 4 * kChunk;
    constexpr int kRec = gd_rec_bytes<FMT>(16);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(sg.w + (FMT == T_F16 ? (int64_t)nblk * A.nk * kChunk
                                      : (int64_t)(nblk >> 2) * A.nk * 4 * kChunk + (nblk & 3) * kChunk)),
        (short)0, FMT == T_F16 ? A.nk * kChunk : A.nk * 4 * kChunk - (nblk & 3) * kChunk, 0x00020000);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(A.x + (int64_t)mblk * MT * A.nk * kRec), (short)0, MT * A.nk * kRec, 0x00020000);
    auto fence = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    v4f2_t y[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < 2; nt++) y[mt][nt] = (v4f2_t){0.0f, 0.0f, 0.0f, 0.0f};
    if (wave < A.nk) {
        GDRaw<FMT> raw[D];
        GDSAct<FMT> act[D][MT];
        // steps past the wave's last read that one again (nothing computes
        // them), so every load is unconditional
        const int last = wave + (A.nk - 1 - wave) / KW * KW;
        auto load = [&](int c, GDRaw<FMT> &rw, GDSAct<FMT> (&ac)[MT]) {
            const int cc = c < last ? c : last;
            gd_load_w<FMT>(wr, cc * kStep, lane, rw);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) gds_load_x<FMT>(xr, (mt * A.nk + cc) * kRec, lane, ac[mt]);
            fence();
        };
        auto step = [&](int c, GDRaw<FMT> &rw, GDSAct<FMT> (&ac)[MT]) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) gds_compute<FMT>(rw, ac[mt], y[mt]);
            fence();
            load(c + D * KW, rw, ac);
        };
#pragma unroll
        for (int u = 0; u < D; u++) load(wave + u * KW, raw[u], act[u]);
        int c = wave;
        for (; c + (D - 1) * KW < A.nk; c += D * KW) {
#pragma unroll
            for (int u = 0; u < D; u++) step(c + u * KW, raw[u], act[u]);
        }
#pragma unroll
        for (int u = 0; u + 1 < D; u++)
            if (c + u * KW < A.nk) step(c + u * KW, raw[u], act[u]);
    }
    // the waves' partial tiles in register order, then four consecutive floats
    // (one row, four columns) per thread, added in wave order, as in gemmsk.h
    float *const pw = sk_lds + wave * kTile + lane;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < 2; nt++)
#pragma unroll
            for (int i = 0; i < 4; i++) pw[((2 * mt + nt) * 4 + i) * 64] = y[mt][nt][i];
    __syncthreads();
    for (int k = (int)threadIdx.x * 4; k < kTile; k += KW * 256) {
        float4 v = *reinterpret_cast<const float4 *>(sk_lds + k);
#pragma unroll
        for (int w = 1; w < KW; w++) {
            const float4 p = *reinterpret_cast<const float4 *>(sk_lds + w * kTile + k);
            v.x += p.x, v.y += p.y, v.z += p.z, v.w += p.w;
        }
        const int l = k & 63, i = (k >> 6) & 3, tile = k >> 8;
        const int64_t m = (int64_t)(mblk * MT + tile / 2) * 16 + 4 * (l >> 4) + i;
        const int64_t n = (int64_t)nblk * 32 + 16 * (tile % 2) + (l & 15);
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

}  // namespace sihip
