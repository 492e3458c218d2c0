// gemm_f32.hip — true-fp32 GEMM on gfx950 MFMA (v_mfma_f32_16x16x4_f32).
//
// The fp32 lane of the run path: C[M,N] = epi(alpha*A[M,K]*op(B) + beta*C) with
// fp32 inputs, fp32 products and fp32 accumulation (no TF32 / xf32 rounding of
// the inputs; the reference's cuBLAS lane defaulted to TF32,
// reference src/compiler/runtime/cuda_backend.c:728-738). Replaces
// cutlass_gemm_simt_f32 and ada_gemm_k64_warp32_async_f32
// (reference gemm/kernel.cu:89-99, gemm/ada_async_kernel.cu:150-320), and fuses
// the row-bias + ReLU epilogue the reference ran on the host after the copy
// back (reference cuda_backend.c:1697-1742).
//
// Tile 64x64x64, 8 waves: waves 0-3 and 4-7 each cover the tile as 2x2 of
// 32x32, the first four on k 0-31 and the second four on k 32-63 of every
// k-tile; the two halves are added through LDS at the end (fixed order). Two
// waves per SIMD let one wave's MFMAs run while the other waits at the
// barrier or on LDS, which one wave per SIMD (one 64x64 tile per CU at
// 1024^3) could not hide. Each lane reads 4 consecutive k of its row as one
// 16-byte LDS load and issues 4 MFMAs, one per element, so A and B use the
// same k permutation {4*(lane/16)+e}. B is staged in LDS as [n][k] for both
// layouts ([K,N] tiles are transposed on the LDS store). Waves 0-3 stage B,
// waves 4-7 stage A.
//
// gemm_f32_dma_kernel takes nearly all shapes (whole tiles, and ragged ones on
// 64x64 or 32x32 tiles) with both operands moved to LDS by LDS-DMA; the
// register-staged gemm_f32_kernel takes operands past 32-bit offsets and
// many ragged tiles of a short k (see pyc_hip_gemm_f32_launch).
#include "common.hpp"
#include "lds_dma.hpp"

namespace pyc {

constexpr int kF32BM = 64;
constexpr int kF32BN = 64;
// K depth 64: one tile's MFMAs cover the global loads of the next tile,
// which depth 32 did not
constexpr int kF32BK = 64;
constexpr int kF32Ch = kF32BK / 4;  // 16-byte chunks per LDS row (16)
constexpr int kF32Ld = kF32BM * kF32Ch / 256;  // 16-byte loads per staging thread (4)

__device__ inline int swz8(int row, int chunk) { return chunk ^ (row & 7); }

template <bool BT, bool GUARD>
__global__ void __launch_bounds__(512, 2)
gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
                int M, int N, int K, float alpha, float beta, const float* __restrict__ bias,
                int epi) {
    __shared__ __attribute__((aligned(16))) float As[2][kF32BM * kF32BK];
    __shared__ __attribute__((aligned(16))) float Bs[2][kF32BN * kF32BK];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int quad = wave & 3;
    const int kh = wave >> 2;      // k half of every k-tile this wave multiplies
    const int wm = quad >> 1;
    const int wn = quad & 1;
    const bool stage_a = kh != 0;  // waves 4-7 stage A, waves 0-3 stage B
    const int t = tid & 255;
    const int m0 = blockIdx.y * kF32BM;
    const int n0 = blockIdx.x * kF32BN;
    const bool vec_k = (K & 3) == 0;
    const bool vec_n = (N & 3) == 0;

    // 64 rows x 16 chunks = 1024 chunks per operand tile -> 4 per staging thread.
    f32x4 rg[kF32Ld];

    auto ld4 = [&](const float* base, int r, int rmax, int c, int cmax, bool vec, size_t ld) -> f32x4 {
        if (!GUARD) return *reinterpret_cast<const f32x4*>(base + (size_t)r * ld + c);
        if (r < rmax && vec && c + 4 <= cmax) return *reinterpret_cast<const f32x4*>(base + (size_t)r * ld + c);
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (r < rmax && c + j < cmax) ? base[(size_t)r * ld + c + j] : 0.f;
        return v;
    };
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < kF32Ld; ++i) {
            const int q = t + i * 256;
            const int row = q / kF32Ch, ch = q % kF32Ch;
            if (stage_a) {
                rg[i] = ld4(A, m0 + row, M, k0 + ch * 4, K, vec_k, (size_t)K);
            } else if (BT) {
                rg[i] = ld4(B, n0 + row, N, k0 + ch * 4, K, vec_k, (size_t)K);
            } else {
                // [K,N] tile: thread t holds the 4 x 4 block of k rows
                // 4*(t/16) + i and columns 4*(t%16) .. +3 (16 threads read
                // one whole 256-byte row segment)
                rg[i] = ld4(B, k0 + 4 * (t >> 4) + i, K, n0 + 4 * (t & 15), N, vec_n, (size_t)N);
            }
        }
    };
    auto store = [&](int buf) {
        if (stage_a || BT) {
            float* dst = stage_a ? As[buf] : Bs[buf];
#pragma unroll
            for (int i = 0; i < kF32Ld; ++i) {
                const int q = t + i * 256;
                const int row = q / kF32Ch, ch = q % kF32Ch;
                *reinterpret_cast<f32x4*>(&dst[row * kF32BK + swz8(row, ch) * 4]) = rg[i];
            }
        } else {
            // the 4 x 4 block transposed in registers: column j of it is the
            // 16-byte chunk t/16 (k = 4*(t/16) .. +3) of LDS row n
            const int kc = t >> 4;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int n = 4 * (t & 15) + j;
                *reinterpret_cast<f32x4*>(&Bs[buf][n * kF32BK + swz8(n, kc) * 4]) =
                    f32x4{rg[0][j], rg[1][j], rg[2][j], rg[3][j]};
            }
        }
    };

    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int ktiles = (K + kF32BK - 1) / kF32BK;
    load(0);
    store(0);
    __syncthreads();
    const int lrow = lane & 15, lgrp = lane >> 4;
    for (int kt = 0; kt < ktiles; ++kt) {
        const int buf = kt & 1;
        const bool more = kt + 1 < ktiles;
        if (more) load((kt + 1) * kF32BK);
#pragma unroll
        for (int kk = 0; kk < kF32BK / 32; ++kk) {
            const int ch = (kh * 2 + kk) * 4 + lgrp;
            f32x4 af[2], bfr[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int r = wm * 32 + i * 16 + lrow;
                af[i] = *reinterpret_cast<const f32x4*>(&As[buf][r * kF32BK + swz8(r, ch) * 4]);
                const int n = wn * 32 + i * 16 + lrow;
                bfr[i] = *reinterpret_cast<const f32x4*>(&Bs[buf][n * kF32BK + swz8(n, ch) * 4]);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[i][e], bfr[j][e], acc[i][j], 0, 0, 0);
        }
        if (more) store(buf ^ 1);
        __syncthreads();
    }

    // k halves: waves 4-7 hand their sums to waves 0-3 through As[0] (free
    // after the loop's last barrier); [quad][element][lane] keeps each store
    // and load one contiguous 256-byte row per wave
    float* red = As[0];
    if (kh) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) red[(quad * 16 + (i * 2 + j) * 4 + r) * 64 + lane] = acc[i][j][r];
    }
    __syncthreads();
    if (kh) return;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] += red[(quad * 16 + (i * 2 + j) * 4 + r) * 64 + lane];

    const bool has_bias = (epi & 1) && bias != nullptr;
    const bool relu = (epi & 2) != 0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int gn = n0 + wn * 32 + j * 16 + lrow;
        if (GUARD && gn >= N) continue;
        const float bv = has_bias ? bias[gn] : 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gm = m0 + wm * 32 + i * 16 + lgrp * 4 + r;
                if (GUARD && gm >= M) continue;
                float* cp = C + (size_t)gm * N + gn;
                float v = alpha * acc[i][j][r];
                if (beta != 0.f) v += beta * *cp;
                v += bv;
                if (relu) v = v > 0.f ? v : 0.f;
                *cp = v;
            }
        }
    }
}

// Whole-tile form (M, N, K multiples of 64): the same 8-wave 64x64 tile and
// k-half split, with the operands moved global->LDS by LDS-DMA through a
// 4-stage ring instead of through VGPRs. Three k-tiles are in flight while
// the fourth is multiplied, so the HBM/L2 latency (longer than one k-tile's
// MFMAs, ~2048 cycles per SIMD) is off the critical path; one barrier per
// k-tile. Each DMA instruction fills 1 KiB of LDS (lane i -> +16 i): four
// 64-float rows. A (and B as [N,K]) rows keep the k-chunk swizzle of the
// register-staged kernel (chunk c of row r at c ^ (r & 7)), applied on the
// global side. B as [K,N] is stored untransposed, [k][n], chunk c of row k at
// c ^ 4((k >> 2) & 3), and read one element per lane (ds_read_b32): the 16
// lanes of each k slot read 16 consecutive n of rows 4 apart, which the
// swizzle puts in four different 16-bank groups.
//
// RAG: any M, N, K (fp32 rows start on 4-byte boundaries, which is what a
// dword-multiple load needs; the rows of the whole-tile form are 16-byte
// aligned). Every load carries its whole offset in the vector register, so that
// the descriptor's range check, which works dword by dword, zeroes what lies
// past the operand: rows past M (or N), [K,N] k-rows past K, and the 16-byte
// chunks past K of an A or [N,K] row get an offset past its end. A chunk that
// crosses the end of its row brings the next row's first elements along: they
// are overwritten with zeros in LDS before the last k-tile is read. k-tiles past
// the last are issued too, all past the end (no traffic).
// TILE 32: the same kernel with a quarter of the tile (each wave one 16x16
// block of a k half, a ring of 8 stages), for products with few 64x64 tiles:
// a k-tile takes about 0.4 us instead of 1.0.
constexpr int kF32Stages = 4, kF32Stages32 = 8;
constexpr size_t kF32DmaLds = (size_t)kF32Stages * 2 * kF32BM * kF32BK * 4;
constexpr uint32_t kF32PastEnd = 0xFFFFFFF0u;  // not below any descriptor's byte count

// SIG: the launch ends a synchronous run, and the kernel itself tells the host
// when its results are complete (instead of a separate one-lane kernel behind
// it on the stream). C is stored with agent-scope stores, which write through
// the XCD's L2 to the coherent level; once a workgroup's stores have completed
// its thread 0 counts it in `done_count` (run_signal_arrive), and the last
// arrival re-arms the counters and stores `done_seq` into the pinned host
// word. A kernel on any stream that the host starts after seeing the word
// reads the whole of C, although the grid's last waves may still be exiting.
template <bool BT, bool SIG, int TILE, bool RAG>
__global__ void __launch_bounds__(512, 1)
gemm_f32_dma_kernel(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
                    int M, int N, int K, float alpha, float beta, const float* __restrict__ bias,
                    int epi, int group_m, uint32_t* __restrict__ done_word, uint32_t* __restrict__ done_count,
                    uint32_t done_seq) {
    constexpr int BK = kF32BK;
    constexpr int STAGES = TILE == 64 ? kF32Stages : kF32Stages32;
    constexpr int F = TILE / 32;                       // 16-wide fragments per wave and operand
    constexpr int NH = TILE / 32;                      // DMA instructions per wave and operand per k-tile
    constexpr int NDMA = 2 * NH;
    constexpr uint32_t OP_BYTES = TILE * BK * 4;       // one operand's part of a stage
    constexpr int CPR = TILE / 4;                      // 16-byte chunks per [K,N] k-row
    constexpr int NSWZ = TILE == 64 ? 3 : 1;           // k-row groups that its swizzle tells apart, minus one
    __shared__ __attribute__((aligned(1024))) float smem[STAGES * 2 * TILE * BK];
    static_assert(sizeof(smem) == kF32DmaLds, "registered LDS figure");

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int quad = wave & 3;
    const int kh = wave >> 2;
    const int wm = quad >> 1;
    const int wn = quad & 1;
    // Tile order: workgroups go to the 8 XCDs round robin, so consecutive
    // tile indices are given to one XCD; tiles are numbered in groups of
    // group_m tile rows, column by column, so the tiles an XCD holds at once
    // share a few A row panels and B column panels in its L2.
    const int tiles_n = (N + TILE - 1) / TILE, tiles_m = (M + TILE - 1) / TILE;
    int bid = blockIdx.x;
    const int nblk = gridDim.x;
    if ((nblk & 7) == 0) bid = (bid & 7) * (nblk >> 3) + (bid >> 3);
    const int span = group_m * tiles_n;
    const int grp = bid / span;
    const int first_m = grp * group_m;
    const int gsz = min(tiles_m - first_m, group_m);
    const int in = bid - grp * span;
    const int m0 = (first_m + in % gsz) * TILE;
    const int n0 = (in / gsz) * TILE;
    const int KT = (K + BK - 1) / BK;

    const i32x4 ra = make_buf_rsrc(A, (uint32_t)((size_t)M * K * 4));
    const i32x4 rb = make_buf_rsrc(B, (uint32_t)((size_t)N * K * 4));
    // wave w issues TILE / 8 rows of the A tile and of the [N,K] B tile (four
    // rows of 16 chunks per instruction; lane i writes chunk position p = i % 16
    // of row i / 16) and 8 k-rows of a [K,N] B tile
    uint32_t va[NH], vb[NH];
    int lch[NH];  // the lane's logical chunk in those rows
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        const int row = TILE / 8 * wave + 4 * h + (lane >> 4), p = lane & 15;
        lch[h] = p ^ (row & 7);
        va[h] = (uint32_t)(((size_t)(m0 + row) * K + 4 * lch[h]) * 4);
        if constexpr (BT) {
            vb[h] = (uint32_t)(((size_t)(n0 + row) * K + 4 * lch[h]) * 4);
        } else {
            const int kr = 8 * wave + h * (64 / CPR) + lane / CPR;
            vb[h] = (uint32_t)(((size_t)kr * N + n0 + 4 * ((lane % CPR) ^ (4 * ((kr >> 2) & NSWZ)))) * 4);
        }
        asm volatile("" : "+v"(va[h]), "+v"(vb[h]));
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    // DMA d (< NDMA) of k-tile kt into ring slot `slot`: d / 2 = h, A if d even
    auto issue_one = [&](int kt, int slot_i, int d) {
        const uint32_t slot = lds0 + (uint32_t)slot_i * 2 * OP_BYTES;
        const uint32_t sa = (uint32_t)kt * BK * 4;
        const uint32_t sb = BT ? sa : (uint32_t)kt * BK * (uint32_t)N * 4;
        const int h = d >> 1;
        const uint32_t off = (uint32_t)(TILE / 8 * wave + 4 * h) * BK * 4;  // = (8 wave + h 64 / CPR) TILE 4
        const bool inside = !RAG || kt * BK + 4 * lch[h] < K;
        if ((d & 1) == 0) {
            if constexpr (RAG) lds_dma_buf_b128_u(ra, inside ? va[h] + sa : kF32PastEnd, 0u, slot + off);
            else lds_dma_buf_b128_u(ra, va[h], sa, slot + off);
        } else {
            if constexpr (RAG) lds_dma_buf_b128_u(rb, !BT || inside ? vb[h] + sb : kF32PastEnd, 0u, slot + OP_BYTES + off);
            else lds_dma_buf_b128_u(rb, vb[h], sb, slot + OP_BYTES + off);
        }
    };
    static_assert(TILE / 8 * BK == 8 * TILE && 4 * BK == 64 / CPR * TILE, "one LDS offset for both B layouts");

    f32x4 acc[F][F];
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int lrow = lane & 15, lgrp = lane >> 4;
    // fragment f of half kk (16 k: 4 per k slot) of the k-tile in ring slot
    // kt % STAGES: f < F the A rows 16 f.., f >= F the B columns 16 (f - F)..
    auto rd = [&](int kt, int kk, int f, f32x4 (&af)[F], f32x4 (&bfr)[F]) {
        const float* As = smem + (kt % STAGES) * 2 * TILE * BK;
        const float* Bs = As + TILE * BK;
        const int ch = (kh * 2 + kk) * 4 + lgrp;
        const int i = f % F;
        if (f < F) {
            const int r = wm * (TILE / 2) + i * 16 + lrow;
            af[i] = *reinterpret_cast<const f32x4*>(&As[r * BK + swz8(r, ch) * 4]);
        } else {
            const int n = wn * (TILE / 2) + i * 16 + lrow;
            if constexpr (BT) {
                bfr[i] = *reinterpret_cast<const f32x4*>(&Bs[n * BK + swz8(n, ch) * 4]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int k = 4 * ch + e;  // (k >> 2) & 3 == lgrp
                    bfr[i][e] = Bs[k * TILE + (((n >> 2) ^ (4 * (lgrp & NSWZ))) << 2) + (n & 3)];
                }
            }
        }
    };
    // RAG: zeros over the elements of the last k-tile that its row-crossing
    // chunks brought from the next row (K % 4 of them are real)
    auto clear_crossing = [&]() {
        float* As = smem + ((KT - 1) % STAGES) * 2 * TILE * BK;
        const int c = (K % BK) / 4;
        if (tid < (BT ? 2 : 1) * TILE) {
            float* row = (tid < TILE ? As : As + TILE * BK) + (tid % TILE) * BK + swz8(tid % TILE, c) * 4;
            for (int e = K % 4; e < 4; ++e) row[e] = 0.f;
        }
        __syncthreads();
    };
    const bool crossing = RAG && K % 4 != 0;

    // Ring: while k-tile kt is multiplied, kt+1 has landed, the next ones are in
    // flight and kt+STAGES-1 (whole tiles: clamped to the last k-tile, a
    // duplicate into the free slot) is issued into the slot kt-1 left, so the
    // wait count is the same every step. Per step the MFMAs go out in program
    // order (sched_barrier) in groups of two: the second half's fragment reads
    // ride on the first groups, the next k-tile's first-half reads on the first
    // groups of the second half (it landed before this step's barrier), and
    // the DMAs on the last groups.
    auto stage_of = [&](int kt) { return RAG ? kt : min(kt, KT - 1); };
    constexpr int NGH = 2 * F * F;  // groups of two MFMAs per half
    constexpr int NFR = 2 * F;      // fragment reads per half
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
#pragma unroll
        for (int d = 0; d < NDMA; ++d) issue_one(stage_of(s), s, d);
    wait_vmem_le<(STAGES - 2) * NDMA>();  // this wave's loads of k-tile 0 landed
    __syncthreads();
    if (crossing && KT == 1) clear_crossing();
    f32x4 af0[F], bf0[F];
#pragma unroll
    for (int f = 0; f < NFR; ++f) rd(0, 0, f, af0, bf0);
    for (int kt = 0; kt < KT; ++kt) {
        wait_vmem_le<(STAGES - 3) * NDMA>();  // own loads of k-tile kt+1 landed (later ones may be in flight)
        // every wave's part of k-tile kt+1 is in LDS, and k-tile kt-1 (and
        // the prefetch of kt) is consumed
        __syncthreads();
        if (crossing && kt == KT - 2) clear_crossing();
        const int kn = stage_of(kt + STAGES - 1);
        f32x4 af1[F], bf1[F];
#pragma unroll
        for (int g = 0; g < 2 * NGH; ++g) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int q = (2 * g + u) % (2 * NGH);  // MFMA q of the half: element e, block (i, j)
                const int e = q / (F * F), i = q / F % F, j = q % F;
                if (g < NGH) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af0[i][e], bf0[j][e], acc[i][j], 0, 0, 0);
                else acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(af1[i][e], bf1[j][e], acc[i][j], 0, 0, 0);
            }
            if (g < NFR) rd(kt, 1, g, af1, bf1);
            if (g >= NGH && g < NGH + NFR) rd(kt + 1, 0, g - NGH, af0, bf0);  // past the last k-tile: unused
            if (g >= 2 * NGH - NDMA) issue_one(kn, (kt + STAGES - 1) % STAGES, g - (2 * NGH - NDMA));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    wait_vmem_le<0>();  // the loads past the last k-tile have landed too
    __syncthreads();  // every wave is done with the ring

    // k halves summed through LDS (waves 4-7 hand theirs to waves 0-3)
    float* red = smem;
    if (kh) {
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) red[(quad * 4 * F * F + (i * F + j) * 4 + r) * 64 + lane] = acc[i][j][r];
    }
    __syncthreads();
    if (!SIG && kh) return;
    if (!kh) {
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[i][j][r] += red[(quad * 4 * F * F + (i * F + j) * 4 + r) * 64 + lane];

        const bool has_bias = (epi & 1) && bias != nullptr;
        const bool relu = (epi & 2) != 0;
#pragma unroll
        for (int j = 0; j < F; ++j) {
            const int gn = n0 + wn * (TILE / 2) + j * 16 + lrow;
            if (RAG && gn >= N) continue;
            const float bv = has_bias ? bias[gn] : 0.f;
#pragma unroll
            for (int i = 0; i < F; ++i) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int gm = m0 + wm * (TILE / 2) + i * 16 + lgrp * 4 + r;
                    if (RAG && gm >= M) continue;
                    float* cp = C + (size_t)gm * N + gn;
                    float v = alpha * acc[i][j][r];
                    if (beta != 0.f) v += beta * *cp;
                    v += bv;
                    if (relu) v = v > 0.f ? v : 0.f;
                    if constexpr (SIG) __hip_atomic_store(cp, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    else *cp = v;
                }
            }
        }
    }
    if constexpr (SIG) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part of C reached the coherent level
        __syncthreads();
        if (tid == 0) run_signal_arrive(done_count, done_word, done_seq);
    }
}

}  // namespace pyc

// 64 or 32: the tile that takes less time, by estimated microseconds: a start
// and end per round of one tile per CU, and a time per k-tile. Measured on the
// MI355X, 64 / 32 (and the register-staged kernel that took ragged shapes), in
// us, [K,N] B: 512 x 128 x 2638 52 / 20.8 (119), 440^3 13.1 / 6.7 (20.4), 512^3
// 11.5 / 6.8, 700 x 701 x 702 18.7 / 16.5 (38), 768^3 16.4 / 23, 1000^3 24.2 / 38
// (40), 1024^3 20.5 / 37, 2624 x 256 x 280 11 / 13.8 (15.5).
static int tile_f32(long M, long N, long K, bool whole) {
    const double kt = (double)((K + 63) / 64);
    const long t64 = ((M + 63) / 64) * ((N + 63) / 64), t32 = ((M + 31) / 32) * ((N + 31) / 32);
    const double c64 = (double)((t64 + 255) / 256) * (2.5 + kt * (whole && t64 <= 256 ? 1.0 : 1.25));
    const double c32 = (double)((t32 + 255) / 256) * (2.2 + kt * 0.43);
    return c32 < c64 ? 32 : 64;
}

// What runs an fp32 product (host only, no launch): 64 or 32 = the LDS-DMA kernel
// with that tile, 0 = the register-staged kernel. The pointers are looked at for
// their alignment.
extern "C" int pyc_hip_gemm_f32_form(int b_trans, int M, int N, int K, const void* A, const void* B) {
    using namespace pyc;
    const bool even = (M % kF32BM == 0) && (N % kF32BN == 0) && (K % kF32BK == 0);
    // the LDS-DMA kernel addresses each operand through a buffer descriptor
    // (32-bit byte offsets, rows and k padded to whole tiles and ring stages)
    // and moves 16-byte chunks, of whole tiles on 16-byte boundaries
    const size_t pad = 16 * kF32BK;
    const bool whole = even && ((uintptr_t)A % 16 == 0) && ((uintptr_t)B % 16 == 0);
    const bool dma = ((uintptr_t)A % 4 == 0) && ((uintptr_t)B % 4 == 0) &&
                     (whole ? (size_t)M * K * 4 < (1ull << 32) && (size_t)N * K * 4 < (1ull << 32)
                            : ((size_t)M + pad) * ((size_t)K + pad) * 4 < kF32PastEnd &&
                                  ((size_t)N + pad) * ((size_t)K + pad) * 4 < kF32PastEnd);
    const int tile = tile_f32(M, N, K, whole);
    if (!dma || whole) return dma ? tile : 0;
    // A short k on the register-staged kernel: starts and ends count, and two of its
    // workgroups share a CU where one ring takes it. More ragged 64 x 64 tiles than CUs,
    // us, ring / register-staged, [K,N] B: 1728 x 2568 x 64 26.8 / 20.3, 1015 x 2944 x 128
    // 21.1 / 19.1, 2805 x 1600 x 140 38 / 36, 1465 x 3792 x 404 91 / 82, 2676 x 560 x 448
    // 25.7 / 27.6; odd rows 910 x 1651 x 144 23 / 20, 1472 x 1980 x 194 28.8 / 36; [N,K] B
    // 2916 x 448 x 192 16.2 / 14.2, 512 x 2440 x 512 27.3 / 26.6, 3435 x 2968 x 664 195 /
    // 173. Whole tiles whose operands start off a 16-byte boundary, which that kernel
    // takes without guards: 3520 x 7424 x 320 346 / 224, 1664 x 7936 x 576 220 / 178, 1280 x
    // 1088 x 320 20.3 / 16.8; [N,K] 8320 x 2176 x 832 363 / 300, 5504 x 2112 x 1664 432 /
    // 386, 384 x 1536 x 192 8.3 / 6.9; from k = 2000 on the ring is level or ahead.
    const long t64 = (long)((M + 63) / 64) * ((N + 63) / 64);
    int k_staged = 0;
    if (even)
        k_staged = t64 > 1024 ? 1792 : t64 > 512 ? 1280 : t64 > 256 ? 1024 : b_trans ? 448 : 320;
    else if (tile == 64 && t64 > 256) {
        const bool wide = K % 4 == 0 && (b_trans || N % 4 == 0);
        k_staged = !wide ? (b_trans ? 128 : 160) : !b_trans ? 416 : t64 > 1024 ? 768 : 512;
    }
    return K <= k_staged ? 0 : tile;
}

extern "C" int pyc_hip_gemm_f32_launch(int b_trans, int M, int N, int K, const void* A,
                                       const void* B, void* C, float alpha, float beta,
                                       const float* bias, int epi, void* stream) {
    using namespace pyc;
    dim3 grid((N + kF32BN - 1) / kF32BN, (M + kF32BM - 1) / kF32BM), block(512);
    const bool even = (M % kF32BM == 0) && (N % kF32BN == 0) && (K % kF32BK == 0);
    hipStream_t s = (hipStream_t)stream;
    const float* a = (const float*)A;
    const float* b = (const float*)B;
    float* c = (float*)C;
    const bool whole = even && ((uintptr_t)A % 16 == 0) && ((uintptr_t)B % 16 == 0);
    const int tile = pyc_hip_gemm_f32_form(b_trans, M, N, K, A, B);
    if (tile) {
        const int tiles_m = (M + tile - 1) / tile, tiles_n = (N + tile - 1) / tile;
        const dim3 tiles((unsigned)(tiles_m * tiles_n));
        const int gm = tiles_m < 4 ? tiles_m : 4;
        RunSignal sg{nullptr, nullptr, 0u};
        // when this launch ends the run, it stores the completion word itself; ragged
        // rows reach the coherent level more slowly than the run's own signal
        // takes (us, one run: 693 x 3008 x 720 74 / 67, 300 x 3008 x 72 22 / 20.6,
        // 232 x 448 x 71 17.4 / 17.2)
        const bool sig = whole && run_signal_claim(&sg);
#define PYC_F32(BT, SIG, TILE, RAG)                                                                                \
    hipLaunchKernelGGL((gemm_f32_dma_kernel<BT, SIG, TILE, RAG>), tiles, block, 0, s, a, b, c, M, N, K, alpha, beta, \
                       bias, epi, gm, sg.word, sg.count, sg.seq)
#define PYC_F32_TILE(BT, SIG)                              \
    do {                                                   \
        if (tile == 32) PYC_F32(BT, SIG, 32, true);        \
        else if (whole) PYC_F32(BT, SIG, 64, false);       \
        else PYC_F32(BT, false, 64, true);                 \
    } while (0)
        if (sig) {
            if (b_trans) PYC_F32_TILE(true, true);
            else PYC_F32_TILE(false, true);
        } else if (b_trans) {
            PYC_F32_TILE(true, false);
        } else {
            PYC_F32_TILE(false, false);
        }
#undef PYC_F32_TILE
#undef PYC_F32
        return hipGetLastError() == hipSuccess ? 0 : -2;
    }
    if (b_trans) {
        if (even) hipLaunchKernelGGL((gemm_f32_kernel<true, false>), grid, block, 0, s, a, b, c, M, N, K, alpha, beta, bias, epi);
        else hipLaunchKernelGGL((gemm_f32_kernel<true, true>), grid, block, 0, s, a, b, c, M, N, K, alpha, beta, bias, epi);
    } else {
        if (even) hipLaunchKernelGGL((gemm_f32_kernel<false, false>), grid, block, 0, s, a, b, c, M, N, K, alpha, beta, bias, epi);
        else hipLaunchKernelGGL((gemm_f32_kernel<false, true>), grid, block, 0, s, a, b, c, M, N, K, alpha, beta, bias, epi);
    }
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

// Registry figures of the LDS-DMA kernel: 128 KB of LDS, one 8-wave
// workgroup per CU (two waves per SIMD).
extern "C" int pyc_hip_kinfo_f32(int b_trans, pyc_hip_kinfo* out) {
    using namespace pyc;
    if (!out) return -1;
    out->name = "gemm_f32_dma_kernel";
    out->lds_bytes = kF32DmaLds;
    out->threads = 512;
    out->waves_per_simd = 2;
    out->fn = b_trans ? reinterpret_cast<const void*>(&gemm_f32_dma_kernel<true, false, 64, false>)
                      : reinterpret_cast<const void*>(&gemm_f32_dma_kernel<false, false, 64, false>);
    return 0;
}
