// gemm_small.hip — bf16/fp16 GEMM for small and medium shapes on gfx950, and
// the implicit-GEMM convolution of the shapes the persistent kernel does not take.
//
// C[M,N] = epi(alpha * A[M,K] * op(B) + beta * C), fp32 accumulation, B stored
// [N,K] ("nt") or [K,N] ("nn", the layout of the reference's default bf16
// symbol cutlass_gemm_tensorcore_bf16, reference
// src/compiler/cutlass_kernels/gemm/kernel.cu:71-84), for the shapes below the
// persistent 256 x 256 kernel's range. A register-staged kernel that prefetches
// one k-step pays a global round trip per step: 17 us for a 512^3 bf16 GEMM on
// 16 workgroups. Here the tile's operands move global -> LDS by LDS-DMA
// through a ring of up to 160 KB of LDS.
//
// 8 waves, two per SIMD: two groups of four, each group 2 x 2 over the tile
// ((BM/2) x (BN/2) per wave, 16 x 16 fragments of v_mfma_f32_16x16x32_{bf16,f16})
// and each on half the k of every ring slot, so that one group's MFMAs run
// while the other waits at the barrier, on its LDS reads or on its DMA issue;
// the two sums are added through LDS at the end in a fixed order. A slot is one
// 64-k stage of a 128-wide tile (each group takes 32 of its k) or 2 or 4 stages
// of the smaller ones (each group takes half the stages).
// The B fragment is the first operand of the MFMA, so each lane ends with four
// adjacent columns of C.
// A and [N,K] B stage rows are 128 bytes (64 k), 16-byte chunk c of row r at
// c ^ (r & 7). [K,N] B stages are 64 k-rows of BN columns, 32-byte segment s
// (16 columns) of k-row k at s ^ f(k): a transpose read (ds_read_b64_tr_b16)
// by 32 lanes touches 32 bytes of k-rows k0..k0+3 and k0+8..k0+11, which f
// spreads over the eight 32-byte slots of a 256-byte bank window.
//
// Code that runs once per tile is kept short (rolled prologue, results through
// LDS into a rolled store loop): a launch starts with a cold instruction cache,
// and straight-line code cost about 0.35 us per KiB of it (a 128 x 128 tile with
// an unrolled epilogue, 13 KiB: 7.1 us for K = 128, where a 3 KiB kernel took 3.1).
//
// SRC: where a stage's operands come from.
//  kDense  K a multiple of 64: a load's offset is the lane's row offset plus a
//          scalar advance per stage.
//  kTail   K a multiple of 8: chunks past K (and [K,N] k-rows past K) get an
//          offset past the buffer's end, which the descriptor reads as zeros
//          (both operands: a neighbouring row may hold an infinity).
//  kConv   NHWC convolution, A row = output pixel, k = (r, s, c), B = the KRSC
//          filter [K_out, R*S*C], C % 8 == 0: a lane's 16-byte chunk is 8
//          channels of one tap. It is the same k for every row the lane loads,
//          so a stage's tap is found once per lane (two multiplications by
//          rounded-up reciprocals); taps in the padding, pixels past the last
//          and k past R*S*C get the past-the-end offset.
//  kAny    any K, N, alignment and size: rows that are no whole 16-byte chunks
//          on 16-byte boundaries cannot go by LDS-DMA, so a wave loads its
//          chunks into registers (unaligned 16-byte loads, those that would
//          cross the end of their row moved back to end there and shifted), two
//          slots ahead, and writes them to one of two LDS slots. Rows of at
//          least 8 elements. f16 [3218,7424] x [7424,922]:
//          470 us on register-staged tiles that loaded such rows by elements.
#include <stdint.h>

#include "common.hpp"
#include "lds_dma.hpp"

namespace pyc {

constexpr int kSmBK = 64;
enum { kDense = 0, kTail = 1, kConv = 2, kAny = 3 };
constexpr uint32_t kSmPastEnd = 0xFFFFFFF0u;  // not below any descriptor's byte count

struct SmConv {
    int H, W, C, S, P, Q, ph, pw, sh, sw;
    uint32_t rc, rs;    // ceil(2^32 / C), ceil(2^32 / S) (0 for S == 1)
    uint32_t x_bytes;
};

// Ring slots of a BM x BN tile (KS stages of 64 k per slot): as many as fit, or
// the two that register staging alternates between.
constexpr int sm_slots(int bm, int bn, int ks, int src) {
    return src == kAny ? 2 : 160 * 1024 / (ks * (bm + bn) * 128);
}
constexpr size_t sm_lds_bytes(int bm, int bn, int ks, int src) {
    return (size_t)sm_slots(bm, bn, ks, src) * ks * (bm + bn) * 128;
}

// segment swizzle f of a [K,N] k-row: (k * BN / 16 + (s ^ f(k))) % 8 differs
// over k0..k0+3 and k0+8..k0+11
template <int BN> __device__ inline int sm_kswz(int k) {
    if constexpr (BN == 32) return (k >> 3) & 1;
    else if constexpr (BN == 64) return ((k >> 1) & 1) | (((k >> 3) & 1) << 1);
    else return (k & 3) | (((k >> 3) & 1) << 2);
}

template <typename T, bool BT, int BM, int BN, int KS, int SRC>
__global__ void __launch_bounds__(512, SRC == kAny && BM < 128 ? 4 : 2)
gemm_small_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, uint16_t* __restrict__ C,
                  int M, int N, int K, float alpha, float beta, const float* __restrict__ bias, int epi,
                  int tiles_m, int tiles_n, int m_base, int n_base, int vec_c, SmConv cg) {
    constexpr uint32_t A_BYTES = BM * 128, B_BYTES = BN * 128;  // one stage: 64 k of BM and of BN rows
    constexpr uint32_t STAGE_BYTES = A_BYTES + B_BYTES;
    constexpr uint32_t SLOT_BYTES = KS * STAGE_BYTES;
    constexpr int SLOTS = sm_slots(BM, BN, KS, SRC);
    constexpr bool HALF = KS == 1;                           // a group takes 32 k of each stage, else KS/2 stages
    constexpr int NST = HALF ? 1 : KS / 2;                   // stages a wave loads and multiplies per slot
    constexpr int NLW = HALF ? 8 : 4;                        // waves that load a stage
    constexpr int NQA = BM / 8 / NLW, NQB = BN / 8 / NLW;    // DMA instructions per wave, operand and stage
    constexpr int LOADS = NQA + NQB;
    constexpr int FM = BM / 32, FN = BN / 32;                // fragments per wave
    constexpr int SEGS = BN / 16;                            // 32-byte segments per [K,N] k-row
    constexpr int CH = BN / 8;                               // 16-byte chunks of a wave's row of fp32 results
    static_assert(SRC == kAny || SLOTS >= 3 && (SLOTS - 2) * NST * LOADS <= 60, "ring");
    static_assert(SRC != kConv || BT, "the filter is the [N,K] operand");
    static_assert(BM * BN * 4 <= SLOTS * SLOT_BYTES, "results through the ring's LDS");
    __shared__ __attribute__((aligned(1024))) uint16_t smem[SLOTS * SLOT_BYTES / 2];
    static_assert(sizeof(smem) == sm_lds_bytes(BM, BN, KS, SRC), "registered LDS figure");

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kh = wave >> 2, quad = wave & 3;               // group (k half), place in the tile
    const int lw = HALF ? wave : quad;
    const int wm = quad >> 1, wn = quad & 1;
    const int lrow = lane & 15, lgrp = lane >> 4;
    // tiles in groups of 4 tile rows, column by column (neighbouring workgroups share B columns)
    const int gm = tiles_m < 4 ? tiles_m : 4;
    const int span = gm * tiles_n;
    const int grp = blockIdx.x / span;
    const int first_m = grp * gm;
    const int gsz = min(tiles_m - first_m, gm);
    const int in = blockIdx.x - grp * span;
    const int m0 = m_base + (first_m + in % gsz) * BM;
    const int n0 = n_base + (in / gsz) * BN;
    const int KT = (K + kSmBK - 1) / kSmBK;

    const i32x4 ra = make_buf_rsrc(A, SRC == kConv ? cg.x_bytes : (uint32_t)((size_t)M * K * 2));
    const i32x4 rb = make_buf_rsrc(B, (uint32_t)((size_t)N * K * 2));
    // DMA instruction q = NQ lw + h of an operand fills LDS bytes
    // 1024 q .. +1023 of its stage: 8 rows of 128 bytes (A, [N,K] B; lane i at
    // 16-byte position i % 8 of row i / 8) or 1024 / (2 BN) k-rows of [K,N] B
    const int lch = (lane & 7) ^ (lane >> 3);  // logical chunk of this lane, the same in every row it loads
    uint32_t va[NQA], vb[NQB];
    int ih0[SRC == kConv ? NQA : 1], iw0[SRC == kConv ? NQA : 1];
#pragma unroll
    for (int h = 0; h < NQA; ++h) {
        const int m = m0 + 8 * (NQA * lw + h) + lane / 8;
        if constexpr (SRC == kConv) {
            const int pq = cg.P * cg.Q;
            const int n = m / pq, r = m - n * pq;
            const int p = r / cg.Q, q = r - p * cg.Q;
            ih0[h] = m < M ? p * cg.sh - cg.ph : -(1 << 30);  // no tap of a pixel past the last is inside
            iw0[h] = q * cg.sw - cg.pw;
            va[h] = ((uint32_t)(n * cg.H + p * cg.sh - cg.ph) * (uint32_t)cg.W + (uint32_t)iw0[h]) * (uint32_t)cg.C;
            asm volatile("" : "+v"(ih0[h]), "+v"(iw0[h]));
        } else {
            va[h] = (uint32_t)(((size_t)m * K + 8 * lch) * 2);
        }
        asm volatile("" : "+v"(va[h]));
    }
#pragma unroll
    for (int h = 0; h < NQB; ++h) {
        const int q = NQB * lw + h;
        if constexpr (BT) {
            vb[h] = (uint32_t)(((size_t)(n0 + 8 * q + lane / 8) * K + 8 * lch) * 2);
        } else {
            // k-row kr, 16-byte position pp: chunk pair (segment) pp / 2 holds segment (pp / 2) ^ f(kr)
            constexpr int CPR = BN / 8;  // 16-byte chunks per k-row
            const int kr = (1024 * q + 16 * lane) / (2 * BN), pp = lane % CPR;
            const int c = ((((pp >> 1) ^ sm_kswz<BN>(kr)) << 1) | (pp & 1));
            vb[h] = (uint32_t)(((size_t)kr * N + n0 + 8 * c) * 2);
        }
        asm volatile("" : "+v"(vb[h]));
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

    // What one stage's loads share: scalar advances (kDense), or whether the
    // lane's chunk is inside K and (kConv) the tap it belongs to. Stages past
    // the last are issued too, so that the count of outstanding loads is the
    // same every step; they read past the buffer's end and cost no traffic.
    struct Src {
        uint32_t sa, sb;
        bool in;
        int r, s;
        uint32_t tap;
    };
    auto src_of = [&](int kt) {
        Src x{};
        x.sa = (uint32_t)kt * (kSmBK * 2);
        x.sb = BT ? x.sa : (uint32_t)kt * kSmBK * (uint32_t)N * 2;
        if constexpr (SRC == kDense) {
            x.in = kt < KT;
        } else {
            const uint32_t k = (uint32_t)(kt * kSmBK + 8 * lch);
            x.in = k < (uint32_t)K;
            if constexpr (SRC == kConv) {
                const uint32_t t = __umulhi(k, cg.rc);
                const uint32_t c = k - t * (uint32_t)cg.C;
                x.r = cg.rs ? (int)__umulhi(t, cg.rs) : (int)t;
                x.s = (int)t - x.r * cg.S;
                x.tap = (uint32_t)(x.r * cg.W + x.s) * (uint32_t)cg.C + c;
            }
        }
        return x;
    };
    // load d (< NQA: A, else B) of a stage whose slot part starts at LDS byte `base`
    auto dma = [&](int d, const Src& x, uint32_t base) {
        i32x4 r = d < NQA ? ra : rb;
        if constexpr (SRC == kDense) r.z = x.in ? r.z : 0;  // a stage past the last: an empty buffer
        if (d < NQA) {
            const int h = d;
            const uint32_t lds = base + (uint32_t)(NQA * lw + h) * 1024;
            if constexpr (SRC == kDense) {
                lds_dma_buf_b128_u(r, va[h], x.sa, lds);
            } else if constexpr (SRC == kTail) {
                lds_dma_buf_b128_u(r, x.in ? va[h] + x.sa : kSmPastEnd, 0u, lds);
            } else {
                const bool ok = x.in & ((unsigned)(ih0[h] + x.r) < (unsigned)cg.H) &
                                ((unsigned)(iw0[h] + x.s) < (unsigned)cg.W);
                lds_dma_buf_b128_u(r, ok ? (va[h] + x.tap) * 2u : kSmPastEnd, 0u, lds);
            }
        } else {
            const int h = d - NQA;
            const uint32_t lds = base + A_BYTES + (uint32_t)(NQB * lw + h) * 1024;
            // [K,N]: the whole offset goes through the range check (a scalar
            // offset would not), which columns past N of the last k-row and
            // k-rows past K need
            if constexpr (!BT) lds_dma_buf_b128_u(r, vb[h] + x.sb, 0u, lds);
            else if constexpr (SRC == kDense) lds_dma_buf_b128_u(r, vb[h], x.sb, lds);
            else lds_dma_buf_b128_u(r, x.in ? vb[h] + x.sb : kSmPastEnd, 0u, lds);
        }
    };

    // kAny: chunk d of stage kt, as dma() would move it. Rows past the end are
    // read from the last valid row (never stored), columns and k past it are
    // 0. `edge` (uniform): some chunk of the stage reaches past its row.
    auto load_any = [&](int d, int kt, bool edge) {
        const uint16_t* row;
        int c, end;  // first element of the chunk in its row, elements in the row
        bool in = true;
        if (d < NQA || BT) {
            const bool a = d < NQA;
            const int r = a ? m0 + 8 * (NQA * lw + d) + lane / 8 : n0 + 8 * (NQB * lw + d - NQA) + lane / 8;
            row = a ? A + (size_t)min(r, M - 1) * K : B + (size_t)min(r, N - 1) * K;
            c = kt * kSmBK + 8 * lch;
            end = K;
        } else {
            constexpr int CPR = BN / 8;
            const int kr = (1024 * (NQB * lw + d - NQA) + 16 * lane) / (2 * BN), pp = lane % CPR;
            in = kt * kSmBK + kr < K;
            row = B + (size_t)min(kt * kSmBK + kr, K - 1) * N;
            c = n0 + 8 * ((((pp >> 1) ^ sm_kswz<BN>(kr)) << 1) | (pp & 1));
            end = N;
        }
        u32x4 v;
        __builtin_memcpy(&v, row + (edge ? min(c, end - 8) : c), 16);  // the device runs with unaligned access on
        if (edge) {
            const int sh = in ? c + 8 - min(c + 8, end) : 8;  // elements past the end
            uint64_t lo = (uint64_t)v[0] | ((uint64_t)v[1] << 32), hi = (uint64_t)v[2] | ((uint64_t)v[3] << 32);
            lo = sh >= 4 ? hi : lo;
            hi = sh >= 4 ? 0 : hi;
            const int b = 16 * (sh & 3);
            lo = (lo >> b) | ((hi << 1) << (63 - b));
            hi >>= b;
            if (sh >= 8) lo = hi = 0;
            v = u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
        }
        return v;
    };

    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // [K,N] transpose reads: lane L of 16-lane group g addresses k-row
    // 8 g + L / 4 (+ 4 for the second read) of a k-step, columns
    // 4 (L % 4) .. +3 of fragment j's 16 columns
    const int tr_k = 8 * lgrp + (lrow >> 2);
    const int tr_c = 4 * (lrow & 3);

    // stage t (< NST) of this wave's share of a slot, and its first k stage
    auto own = [&](int t) { return HALF ? 0 : kh * NST + t; };
    const int steps = (KT + KS - 1) / KS;
    constexpr int KSTEPS = HALF ? 1 : 2;               // 32-k steps a wave multiplies per stage
    constexpr int NM = FM * FN * KSTEPS;               // MFMAs per stage and wave
    constexpr int GAP = NM / LOADS > 0 ? NM / LOADS : 1;  // MFMAs between two DMAs
    // this wave's MFMAs on stage t of its share of slot `cur`; each(d) is called
    // for d < LOADS with MFMAs in between
    auto multiply = [&](int cur, int t, auto&& each) {
        const uint16_t* As = smem + (uint32_t)cur * (SLOT_BYTES / 2) + (uint32_t)own(t) * (STAGE_BYTES / 2);
        const uint16_t* Bs = As + A_BYTES / 2;
        u32x4 fa[KSTEPS][FM], fb[KSTEPS][FN];
#pragma unroll
        for (int u = 0; u < KSTEPS; ++u) {
            const int ks = HALF ? kh : u;  // which 32 k of the stage
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                const int r = wm * (BM / 2) + 16 * i + lrow;
                fa[u][i] = *reinterpret_cast<const u32x4*>(As + r * 64 + 8 * ((4 * ks + lgrp) ^ (r & 7)));
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                if constexpr (BT) {
                    const int r = wn * (BN / 2) + 16 * j + lrow;
                    fb[u][j] = *reinterpret_cast<const u32x4*>(Bs + r * 64 + 8 * ((4 * ks + lgrp) ^ (r & 7)));
                } else {
                    const int seg = wn * (SEGS / 2) + j;  // the fragment's 16 columns
                    const int k0 = 32 * ks + tr_k, k1 = k0 + 4;
                    const u32x2 lo = lds_read_tr16(Bs + k0 * BN + 16 * (seg ^ sm_kswz<BN>(k0)) + tr_c);
                    const u32x2 hi = lds_read_tr16(Bs + k1 * BN + 16 * (seg ^ sm_kswz<BN>(k1)) + tr_c);
                    fb[u][j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
                }
            }
        }
        int d = 0;
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int u = m / (FM * FN), q = m % (FM * FN);
            acc[q / FN][q % FN] = mfma16x16x32(fb[u][q % FN], fa[u][q / FN], acc[q / FN][q % FN], T{});
            if (m % GAP == GAP - 1 && d < LOADS) each(d++);
            if (GAP > 1 && SRC != kAny) __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (; d < LOADS; ++d) each(d);
    };
    if constexpr (SRC == kAny) {
        // rg[s & 1] is slot s in registers; slot s + 1 goes to LDS and slot
        // s + 3 starts loading while slot s is multiplied
        u32x4 rg[2][NST * LOADS];
        const bool edge_n = !BT && n0 + BN > N;
        auto fetch = [&](int st, u32x4 (&r)[NST * LOADS]) {
            if (edge_n || (st + 1) * KS * kSmBK > K) {
#pragma unroll
                for (int t = 0; t < NST; ++t)
#pragma unroll
                    for (int d = 0; d < LOADS; ++d) r[t * LOADS + d] = load_any(d, st * KS + own(t), true);
            } else {
#pragma unroll
                for (int t = 0; t < NST; ++t)
#pragma unroll
                    for (int d = 0; d < LOADS; ++d) r[t * LOADS + d] = load_any(d, st * KS + own(t), false);
            }
        };
        auto put = [&](int st, const u32x4 (&r)[NST * LOADS]) {
#pragma unroll
            for (int t = 0; t < NST; ++t)
#pragma unroll
                for (int d = 0; d < LOADS; ++d) {
                    const uint32_t off = d < NQA ? (uint32_t)(NQA * lw + d) * 1024
                                                 : A_BYTES + (uint32_t)(NQB * lw + d - NQA) * 1024;
                    *reinterpret_cast<u32x4*>(smem + (((st & 1) * SLOT_BYTES + own(t) * STAGE_BYTES + off) / 2 +
                                                      lane * 8)) = r[t * LOADS + d];
                }
        };
        fetch(0, rg[0]);
        fetch(1, rg[1]);
        put(0, rg[0]);
        fetch(2, rg[0]);
        __syncthreads();
        for (int st = 0; st < steps; st += 2) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {  // slots past the last are zeros
                put(st + u + 1, rg[(u + 1) & 1]);
                fetch(st + u + 3, rg[(u + 1) & 1]);
#pragma unroll
                for (int t = 0; t < NST; ++t) multiply(u, t, [](int) {});
                __syncthreads();
            }
        }
    } else {
        // The prologue fills all slots but one; then every step issues one slot
        // into the place the previous step freed, so each wave has SLOTS - 2
        // slots of its loads outstanding at the top of every step.
#pragma unroll 1
        for (int p = 0; p < SLOTS - 1; ++p)
#pragma unroll
            for (int t = 0; t < NST; ++t) {
                const Src x = src_of(p * KS + own(t));
#pragma unroll
                for (int d = 0; d < LOADS; ++d)
                    dma(d, x, lds0 + (uint32_t)p * SLOT_BYTES + (uint32_t)own(t) * STAGE_BYTES);
            }
        int cur = 0, nxt = SLOTS - 1;  // slot of this step, slot that is issued now
        for (int st = 0; st < steps; ++st) {
            wait_vmem_le<(SLOTS >= 2 ? SLOTS - 2 : 0) * NST * LOADS>();  // own loads of this step's slot landed
            __syncthreads();  // every wave's part of it is in LDS; the previous step's slot is consumed
#pragma unroll
            for (int t = 0; t < NST; ++t) {
                const Src x = src_of((st + SLOTS - 1) * KS + own(t));
                const uint32_t base = lds0 + (uint32_t)nxt * SLOT_BYTES + (uint32_t)own(t) * STAGE_BYTES;
                multiply(cur, t, [&](int d) { dma(d, x, base); });
            }
            nxt = cur;
            cur = cur + 1 == SLOTS ? 0 : cur + 1;
        }
    }
    if constexpr (SRC != kAny) wait_vmem_le<0>();  // the loads past the last stage have landed too
    __syncthreads();    // every wave is done with the ring; it takes the results

    // Results as fp32 in LDS, BM/2 x BN/2 per quadrant, 16-byte chunk c of row
    // r at c ^ (r % CH): acc[i][j] is row 16 i + lrow, columns 16 j + 4 lgrp .. +3.
    // Group 1 hands over its sums, group 0 adds them to its own, and all eight
    // waves write C, half a quadrant's rows each, CH lanes to a row segment.
    f32x4* const res = reinterpret_cast<f32x4*>(smem) + quad * (BM / 2) * CH;
    auto at = [&](int r, int c) { return r * CH + (c ^ (r & (CH - 1))); };
    if (kh) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) res[at(16 * i + lrow, 4 * j + lgrp)] = acc[i][j];
    }
    __syncthreads();
    if (!kh) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                f32x4* p = &res[at(16 * i + lrow, 4 * j + lgrp)];
                *p = acc[i][j] + *p;
            }
    }
    __syncthreads();
    constexpr int RPI = kWave / CH;  // rows per pass of a wave
    static_assert(BM / 4 % RPI == 0 || BM / 4 < RPI, "row passes");
    const bool relu = (epi & 2) != 0;
    const int c = lane % CH;
    const int gn = n0 + wn * (BN / 2) + 4 * c;
    f32x4 bv = f32x4{0.f, 0.f, 0.f, 0.f};
    if ((epi & 1) && bias != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (gn + e < N) bv[e] = bias[gn + e];
    }
#pragma unroll 1
    for (int r = kh * (BM / 4) + lane / CH; r < (kh + 1) * (BM / 4); r += RPI) {
        const int gm = m0 + wm * (BM / 2) + r;
        if (gm >= M || gn >= N) break;
        f32x4 v = res[at(r, c)];
        uint16_t* cp = C + (size_t)gm * N + gn;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = alpha * v[e];
        if (beta != 0.f) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (gn + e < N) v[e] += beta * elem<T>::to_f32(cp[e]);
        }
        uint16_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float x = v[e] + bv[e];
            if (relu) x = x > 0.f ? x : 0.f;
            o[e] = elem<T>::from_f32(x);
        }
        if (vec_c) {  // N % 4 == 0: a lane's 4 columns are all in or all out
            *reinterpret_cast<u32x2*>(cp) =
                u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (gn + e < N) cp[e] = o[e];
        }
    }
}

// The part of C a launch computes: rows m0 .. m1 - 1, columns n0 .. n1 - 1 (both
// ends whole tiles from the start, or the end of C).
struct SmPart {
    int m0, m1, n0, n1;
};

template <typename T, bool BT, int SRC>
static int launch_small(int bm, int bn, int M, int N, int K, const void* A, const void* B, void* C, float alpha,
                        float beta, const float* bias, int epi, const SmPart& pt, hipStream_t s, const SmConv& cg) {
    if (pt.m0 < 0 || pt.m0 >= pt.m1 || pt.m1 > M || pt.n0 < 0 || pt.n0 >= pt.n1 || pt.n1 > N) return 1;
    const int tiles_m = (pt.m1 - pt.m0 + bm - 1) / bm, tiles_n = (pt.n1 - pt.n0 + bn - 1) / bn;
    const long tiles = (long)tiles_m * tiles_n;
    if (tiles > 0x7FFFFFFFL) return 1;
    const dim3 grid((unsigned)tiles), block(8 * kWave);
    const uint16_t* a = (const uint16_t*)A;
    const uint16_t* b = (const uint16_t*)B;
    uint16_t* c = (uint16_t*)C;
    const int vec_c = N % 4 == 0 && ((uintptr_t)C & 7) == 0;
#define PYC_SMALL(BM, BN, KS)                                                                                  \
    hipLaunchKernelGGL((gemm_small_kernel<T, BT, BM, BN, KS, SRC>), grid, block, 0, s, a, b, c, M, N, K, alpha, \
                       beta, bias, epi, tiles_m, tiles_n, pt.m0, pt.n0, vec_c, cg)
    if (bm == 32 && bn == 32) PYC_SMALL(32, 32, 4);
    else if (bm == 64 && bn == 64) PYC_SMALL(64, 64, 2);
    else if (bm == 128 && bn == 64) PYC_SMALL(128, 64, 1);
    else if (bm == 128 && bn == 128) PYC_SMALL(128, 128, 1);
    else if constexpr (SRC != kAny) {
        if (bm == 128 && bn == 256) PYC_SMALL(128, 256, 1);
        else return 1;
    } else return 1;
#undef PYC_SMALL
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace pyc

// Which of these tiles run a product (host only, no launch): 2 = all of them, by
// LDS-DMA (K a multiple of 8 and, for [K,N] B, N of 4, with A and B 16-byte
// aligned and below 4 GiB), 1 = those up to 128 x 128, staged through registers
// (rows of at least 8 elements), 0 = none.
extern "C" int pyc_hip_gemm_small_takes(int b_trans, int M, int N, int K, const void* A, const void* B) {
    using namespace pyc;
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    // [K,N] k-rows past K that are multiplied (against zeros of A) must read zeros and
    // not wrap round to the first ones: they end with a slot's last stage, less than
    // 5 stages past K. Later stages are issued too and may wrap, but nothing reads them.
    const size_t kpad = (size_t)K + 16 * kSmBK;
    if (K % 8 || (!b_trans && N % 4) || (((uintptr_t)A | (uintptr_t)B) & 15) || (size_t)M * K * 2 > kSmPastEnd ||
        (size_t)N * K * 2 > kSmPastEnd || ((K % kSmBK || !b_trans) && (size_t)N * kpad * 2 > kSmPastEnd))
        return K < 8 || (!b_trans && N < 8) ? 0 : 1;
    return 2;
}

// bm x bn: one of the tiles above; m0 .. n1: the part of C (SmPart). Rows of A (and of [N,K] B) past the end are
// read as zeros through the buffer descriptors, [K,N] B columns past N read
// neighbouring data, and only the rows and columns of C inside M x N are
// written. Returns 1 for an unknown tile and for one that does not take the
// product (pyc_hip_gemm_small_takes), 0 on launch, -2 on a launch error.
extern "C" int pyc_hip_gemm_small_launch(int is_bf16, int b_trans, int bm, int bn, int M, int N, int K, const void* A,
                                         const void* B, void* C, float alpha, float beta, const float* bias,
                                         int epi, int m0, int m1, int n0, int n1, void* stream) {
    using namespace pyc;
    const int takes = pyc_hip_gemm_small_takes(b_trans, M, N, K, A, B);
    if (takes == 0) return 1;
    const SmPart pt{m0, m1, n0, n1};
    const bool any = takes == 1, tail = K % kSmBK != 0;
    hipStream_t s = (hipStream_t)stream;
    const SmConv cg{};
#define PYC_GO(TY, BT)                                                                                              \
    (any    ? launch_small<TY, BT, kAny>(bm, bn, M, N, K, A, B, C, alpha, beta, bias, epi, pt, s, cg)                   \
     : tail ? launch_small<TY, BT, kTail>(bm, bn, M, N, K, A, B, C, alpha, beta, bias, epi, pt, s, cg)                  \
            : launch_small<TY, BT, kDense>(bm, bn, M, N, K, A, B, C, alpha, beta, bias, epi, pt, s, cg))
    if (is_bf16) return b_trans ? PYC_GO(bf16_t, true) : PYC_GO(bf16_t, false);
    return b_trans ? PYC_GO(f16_t, true) : PYC_GO(f16_t, false);
#undef PYC_GO
}

// Reciprocals of a filter's tap split: k / C and t / S by a multiplication with the
// rounded-up rc = ceil(2^32 / C) and rs = ceil(2^32 / S) (*rs 0 for S == 1: no
// division). x * ceil(2^32 / d) is x * e / 2^32 above x / d * 2^32, with e =
// d * ceil(2^32 / d) - 2^32, so floor is exact while x * e < 2^32. Returns 1 where
// that holds for every k < R*S*C and every tap t < R*S, else 0. Host only.
extern "C" int pyc_hip_conv2d_tap_split(int R, int S, int C, uint32_t* rc, uint32_t* rs) {
    const uint64_t two32 = 1ull << 32;
    if (R <= 0 || S <= 0 || C <= 1 || (uint64_t)R * S > 0x7FFFFFFFull / C) return 0;
    const uint64_t taps = (uint64_t)R * S, c = (uint64_t)C, s = (uint64_t)S;
    const uint64_t qc = (two32 + c - 1) / c, qs = (two32 + s - 1) / s;
    *rc = (uint32_t)qc;
    *rs = S == 1 ? 0u : (uint32_t)qs;
    return taps * c * c < two32 && (taps - 1) * (qs * s - two32) < two32;  // (e < C)
}

// NHWC convolution on the same tiles (bm output pixels x bn output channels),
// output pixels m0 .. m1 - 1.
// Returns 1 outside its preconditions (C % 8 == 0, x and w 16-byte aligned and
// below 4 GiB, exact reciprocals: pyc_hip_conv2d_tap_split), 0 on launch, -2 on a
// launch error.
extern "C" int pyc_hip_conv2d_small_launch(int is_bf16, int bm, int bn, int Nimg, int H, int W, int C, int Kout,
                                           int R, int S, int ph, int pw, int sh, int sw, const void* x,
                                           const void* w, const float* bias, int relu, void* y, int m0, int m1,
                                           void* stream) {
    using namespace pyc;
    const long long P = (H + 2LL * ph - R) / sh + 1, Q = (W + 2LL * pw - S) / sw + 1;
    const long long M = (long long)Nimg * P * Q, Kg = (long long)R * S * C;
    const unsigned long long lim = kSmPastEnd;
    if (C % 8 || P <= 0 || Q <= 0 || M > 0x7FFFFF00LL || Kg > 0x7FFFFF00LL) return 1;
    uint32_t rc = 0, rs = 0;
    if (!pyc_hip_conv2d_tap_split(R, S, C, &rc, &rs)) return 1;
    if ((unsigned long long)Nimg * H * W * C * 2 > lim || (unsigned long long)Kout * Kg * 2 > lim) return 1;
    if (H >= (1 << 28) || W >= (1 << 28) || ph >= (1 << 28) || pw >= (1 << 28)) return 1;
    if (((uintptr_t)x | (uintptr_t)w) & 15) return 1;
    const SmConv cg{H, W, C, S, (int)P, (int)Q, ph, pw, sh, sw, rc, rs, (uint32_t)((size_t)Nimg * H * W * C * 2)};
    const SmPart pt{m0, m1 > 0 ? m1 : (int)M, 0, Kout};  // m1 <= 0: to the last pixel
    const int epi = (bias ? 1 : 0) | (relu ? 2 : 0);
    hipStream_t st = (hipStream_t)stream;
    if (is_bf16)
        return launch_small<bf16_t, true, kConv>(bm, bn, (int)M, Kout, (int)Kg, x, w, y, 1.0f, 0.0f, bias, epi, pt, st,
                                                 cg);
    return launch_small<f16_t, true, kConv>(bm, bn, (int)M, Kout, (int)Kg, x, w, y, 1.0f, 0.0f, bias, epi, pt, st,
                                                 cg);
}

// Registry figures: the ring allows one 8-wave workgroup per CU.
extern "C" int pyc_hip_kinfo_small(int tile, int b_trans, int is_bf16, pyc_hip_kinfo* out) {
    using namespace pyc;
    if (!out || (tile != 64 && tile != 128)) return -1;
    out->threads = 512;
    out->waves_per_simd = 2;
    out->lds_bytes = sm_lds_bytes(tile, tile, tile == 64 ? 2 : 1, kDense);
    out->name = tile == 64 ? "gemm_small_kernel<64>" : "gemm_small_kernel<128>";
#define PYC_KI(TY, BT) \
    out->fn = tile == 64 ? reinterpret_cast<const void*>(&gemm_small_kernel<TY, BT, 64, 64, 2, kDense>) \
                         : reinterpret_cast<const void*>(&gemm_small_kernel<TY, BT, 128, 128, 1, kDense>)
    if (is_bf16) {
        if (b_trans) PYC_KI(bf16_t, true); else PYC_KI(bf16_t, false);
    } else {
        if (b_trans) PYC_KI(f16_t, true); else PYC_KI(f16_t, false);
    }
#undef PYC_KI
    return 0;
}
