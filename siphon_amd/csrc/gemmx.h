// GEMM for longer prompts of K-quant weights (Q2_K .. Q6_K) on
// v_mfma_i32_16x16x64_i8 (gfx950): Y_i[M x n_out_i] = X[M x n_in] * W_i^T for
// a group of matrices that share X, each output within the tolerance of the
// reference dot (reference kernels.c:249-523). The arithmetic, the weight copy
// and a super-block's decode are gemmsk.h's.
//
// Tiles. A workgroup of 4 waves computes BM = 16 MT activation rows against
// 128 weight rows, wave w rows 32 w .. 32 w + 31 (two 16-column n tiles). Per
// super-block a wave decodes its weights once and applies them to the MT m
// tiles in turn, whose activation fragments all four waves read from LDS. The
// matrices of a group are segments of one grid, and K slices split a tile's
// super-blocks over several workgroups where the tiles alone leave CUs idle
// (the host's plan weighs both).
//
// Pipeline. The activation records of the next one or two super-blocks are
// copied to LDS by DMA (a ring of gx_ring(MT) slots), the weights of the next
// one or two are loaded into registers (gx_wdepth(MT)). Each step waits for
// its own record by count, younger copies and loads staying in flight, and
// meets the other waves at a bare s_barrier: __syncthreads would wait for every
// copy in flight.
//
// What bounds it: issue. A SIMD hides about two VALU instructions behind one
// MFMA; at MT = 8 Q4_K has 72 MFMAs and 245 VALU instructions per 16 weight
// rows and super-block (85 to decode, 20 per m tile in the epilogue).
#pragma once

#include <type_traits>

#include "agent.h"
#include "gemmsk.h"

namespace sihip {

struct GXSeg {
    const uint8_t *w;     // gemmks.h chunks [nblk32][nb]
    float *y;             // Y[m * ldy + n]
    int64_t ldy, n_out;
    uint32_t type;
    int nblk32;           // 32-row blocks that exist
    int nb0;              // the segment's first n block (128 rows) in the grid
};

struct GXArgs {
    const uint8_t *x;     // activation records [MB][nb]
    int64_t M;
    int nb, MB, NB;       // super-blocks; m blocks of BM rows; n blocks of 128 rows (all segments)
    int S, SBK;           // K slices, super-blocks per slice
    float *part;
    uint32_t *cnt;
    int nseg;
    GXSeg seg[kG2MaxSegs];
};

// LDS slots of activation records (two workgroups per CU share 160 KiB), and
// super-blocks of weights in registers (what 256 VGPRs leave room for).
__host__ __device__ constexpr int gx_ring(int MT) { return MT <= 5 ? 3 : 2; }
__host__ __device__ constexpr int gx_wdepth(int MT) { return MT <= 3 ? 2 : 1; }

// f(0), f(1), .. f(N - 1) with constant arguments.
template <int N, int I = 0, class F>
__device__ inline void gx_unroll(F f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        gx_unroll<N, I + 1>(f);
    }
}

// The wave's operations younger than a step's record when the step waits for
// it, at least: the records of the R - 2 later steps (kD copies each) and the
// weights (kW loads a step) issued since, which are min(R - 1, DW) steps' worth
// from the prologue on. Step u of the last partial round of U (u < 0: any step
// of a whole one) counts only weights that a later step uses: the compiler may
// drop the loads issued for steps U - 1 and beyond, one step's worth for each
// step from U - 1 - DW on.
__host__ __device__ constexpr int gx_younger(int R, int DW, int kD, int kW, int U, int u) {
    const int kept = R - 1 < DW ? R - 1 : DW, dropped = u > U - 1 - DW ? u - (U - 1 - DW) : 0;
    return (R - 2) * kD + (kept > dropped ? kept - dropped : 0) * kW;
}

template <uint32_t FMT, int MT>
__device__ inline void gx_body(const GXArgs &A, const GXSeg &sg, int nblk, int mblk, int slice,
                               uint8_t *s0, uint8_t *s1, uint8_t *s2) {
    constexpr int R = gx_ring(MT), DW = gx_wdepth(MT);
    auto slot = [&](auto u) -> uint8_t * {
        constexpr int k = decltype(u)::value % R;
        return k == 0 ? s0 : k == 1 ? s1 : s2;
    };
    constexpr int BM = 16 * MT;
    constexpr int kRec = g2_rec_bytes(BM);
    constexpr int kPieces = kRec / 1024, kD = (kPieces + 3) / 4;
    const int lblk = nblk - sg.nb0;
    const int c0 = slice * A.SBK;
    const int c1 = c0 + A.SBK < A.nb ? c0 + A.SBK : A.nb;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, r16 = lane & 15;
    // a wave past the last row block computes it again (nothing stores it)
    const int blk = lblk * 4 + wave < sg.nblk32 ? lblk * 4 + wave : sg.nblk32 - 1;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(sg.w + (int64_t)blk * A.nb * KS<FMT>::chunk), (short)0, A.nb * KS<FMT>::chunk, 0x00020000);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(A.x + (int64_t)mblk * A.nb * kRec), (short)0, A.nb * kRec, 0x00020000);
    auto dma = [&](int c, uint8_t *dst) {
#pragma unroll
        for (int k = 0; k < kD; k++) {
            const int i = wave + 4 * k < kPieces ? wave + 4 * k : kPieces - 1;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                xr, (__attribute__((address_space(3))) void *)(dst + i * 1024), 16, lane * 16,
                c * kRec + i * 1024, 0, 0);
        }
    };
    // keep the order of issue: the counted waits rest on a record's copies coming
    // before the weights of its step
    auto fence = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto clamp = [&](int c) { return c < c1 ? c : c1 - 1; };
    v4f2_t y[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < 2; nt++) y[mt][nt] = (v4f2_t){0.0f, 0.0f, 0.0f, 0.0f};
    SKRaw<FMT, 2> raw[DW];
    gx_unroll<(R - 1 > DW ? R - 1 : DW)>([&](auto i) {
        if constexpr (i < R - 1) dma(clamp(c0 + i), slot(i));
        fence();
        if constexpr (i < DW) sk_load_w<FMT, 2>(wr, clamp(c0 + i), 0, lane, raw[i]);
        fence();
    });
    constexpr int kW = sk_loads<FMT>();  // weight loads of a super-block
    auto step = [&](int c, auto younger, const uint8_t *X, uint8_t *Xn, SKRaw<FMT, 2> &rw) {
        // the record has arrived, and this wave's reads of the slot before have
        // returned, which the copy below overwrites
        wait_vm_lds<decltype(younger)::value>();
        __builtin_amdgcn_s_barrier();
        fence();
        SKOps<FMT, 2> o;
        sk_decode<FMT, 2>(rw, 0, lane, o);
        dma(clamp(c + R - 1), Xn);
        fence();
        sk_load_w<FMT, 2>(wr, clamp(c + DW), 0, lane, rw);
        fence();
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            SKAct s;
#pragma unroll
            for (int ks = 0; ks < 4; ks++)
                s.a[ks] = *reinterpret_cast<const v4i2_t *>(X + (4 * mt + ks) * 1024 + lane * 16);
            if constexpr (KS<FMT>::mins)
                s.bs = *reinterpret_cast<const v8h2_t *>(X + g2_rec_bsum(BM) + (16 * mt + r16) * 32 + (g & 1) * 16);
            s.dx = *reinterpret_cast<const float4 *>(X + g2_rec_dx(BM) + (16 * mt + 4 * g) * 4);
            if constexpr (FMT == T_Q5_K)
                s.sx = *reinterpret_cast<const v4i2_t *>(X + g2_rec_sx(BM) + (16 * mt + 4 * g) * 4);
            sk_compute<FMT, 2>(o, s, y[mt]);
        }
    };
    constexpr int U = R * DW;  // steps per round: ring slot and weight set static
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

template <uint32_t F0, uint32_t F1, int MT>
__global__ __launch_bounds__(kG2Threads)
__attribute__((amdgpu_waves_per_eu(2))) void gemmx_kernel(GXArgs A) {
    constexpr int R = gx_ring(MT), kRec = g2_rec_bytes(16 * MT);
    // distinct LDS objects: a step reads one while copies into the others are
    // in flight, and only distinct objects let the compiler see that
    __shared__ __attribute__((aligned(16))) uint8_t s0[kRec];
    __shared__ __attribute__((aligned(16))) uint8_t s1[kRec];
    __shared__ __attribute__((aligned(16))) uint8_t s2[R > 2 ? kRec : 16];
    const int b = blockIdx.x;
    const int xcd = b & 7, t = b >> 3;
    const int per = A.MB * A.S;
    const int nblk = (t / per) * 8 + xcd, rest = t % per;
    const int slice = rest / A.MB, mblk = rest % A.MB;
    if (nblk >= A.NB) return;
    GXSeg sg = A.seg[0];
#pragma unroll
    for (int k = 1; k < kG2MaxSegs; k++)
        if (k < A.nseg && nblk >= A.seg[k].nb0) sg = A.seg[k];
    if (F0 == F1 || sg.type == F0) gx_body<F0, MT>(A, sg, nblk, mblk, slice, s0, s1, s2);
    else gx_body<F1, MT>(A, sg, nblk, mblk, slice, s0, s1, s2);
}

}  // namespace sihip
