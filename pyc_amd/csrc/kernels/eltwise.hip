// eltwise.hip — GELU and LayerNorm on gfx950: the IR's PYC_IR_OP_GELU and
// PYC_IR_OP_LAYERNORM, which the reference engine reports as graph breaks and
// executes nowhere (its CPU executor rejects them, reference
// src/compiler/compiler_api.c:1877-2092; its GPU path accepts matmul chains
// only, reference src/compiler/runtime/cuda_backend.c:1201-1390; the break
// accounting is reference src/compiler/passes/pass_manager.c:313-373).
// Semantics chosen here, as PyTorch defines them:
//   GELU(x)      = 0.5 x (1 + erf(x / sqrt(2)))               (exact form,
//                  evaluated through erfc; see gelu_f)
//   LayerNorm(x) = (x - mean) / sqrt(var + eps) * gamma + beta over the last
//                  dimension, var the population variance (divide by D).
// Both are HBM-bound. Elements are fp32, bf16 or fp16; every statistic and
// every intermediate is fp32, results are rounded once (to nearest even).
#include <math.h>

#include <type_traits>

#include "common.hpp"

namespace pyc {

template <typename T> struct io;
template <> struct io<float> {
    static constexpr int kVec = 4;  // elements per 16-byte chunk
    __device__ static inline float get(const float* p, size_t i) { return p[i]; }
    __device__ static inline void put(float* p, size_t i, float v) { p[i] = v; }
    __device__ static inline void get16(const float* p, size_t i, float (&v)[4]) {
        const f32x4 c = *reinterpret_cast<const f32x4*>(p + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = c[e];
    }
    __device__ static inline void put16(float* p, size_t i, const float (&v)[4]) {
        *reinterpret_cast<f32x4*>(p + i) = f32x4{v[0], v[1], v[2], v[3]};
    }
    __device__ static inline u32x4 pack(const float (&v)[4]) {
        return u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
    }
    __device__ static inline u32x4 raw16(const float* p, size_t i) { return *reinterpret_cast<const u32x4*>(p + i); }
    __device__ static inline void unpack(const u32x4& c, float (&v)[4]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __uint_as_float(c[e]);
    }
};
template <typename H> struct io_half {
    static constexpr int kVec = 8;
    __device__ static inline float get(const uint16_t* p, size_t i) { return elem<H>::to_f32(p[i]); }
    __device__ static inline void put(uint16_t* p, size_t i, float v) { p[i] = elem<H>::from_f32(v); }
    __device__ static inline void unpack(const u32x4& c, float (&v)[8]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[2 * e] = elem<H>::to_f32((uint16_t)(c[e] & 0xFFFFu));
            v[2 * e + 1] = elem<H>::to_f32((uint16_t)(c[e] >> 16));
        }
    }
    __device__ static inline u32x4 raw16(const uint16_t* p, size_t i) { return *reinterpret_cast<const u32x4*>(p + i); }
    __device__ static inline void get16(const uint16_t* p, size_t i, float (&v)[8]) { unpack(raw16(p, i), v); }
    __device__ static inline u32x4 pack(const float (&v)[8]) {
        u32x4 c;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            c[e] = (uint32_t)elem<H>::from_f32(v[2 * e]) | ((uint32_t)elem<H>::from_f32(v[2 * e + 1]) << 16);
        return c;
    }
    __device__ static inline void put16(uint16_t* p, size_t i, const float (&v)[8]) {
        *reinterpret_cast<u32x4*>(p + i) = pack(v);
    }
};
template <> struct io<bf16_t> : io_half<bf16_t> {};
template <> struct io<f16_t> : io_half<f16_t> {};

// storage type of T in memory
template <typename T> using store_t = typename std::conditional<std::is_same<T, float>::value, float, uint16_t>::type;

// GELU through the complementary error function, branch free:
//   GELU(x) = x Phi(x),  Phi(x) = 1 - erfc(a)/2 for x >= 0 and erfc(a)/2 for
//   x < 0,  a = |x| / sqrt(2),
//   erfc(a) = exp(-a^2) t S(t),  t = 1 / (1 + p a),  S a degree-7 polynomial
// (the form of Abramowitz & Stegun 7.1.26 with more terms). p and S were
// fitted in float64 by least squares reweighted toward the minimax relative
// error of erfc(a) exp(a^2) on a in [0, 10]: relative error 9.4e-8, and
// S(1) = 1 to the fp32 rounding, so GELU(0) = 0 exactly. Evaluated in fp32 the
// result is within 8 ulp of float64 GELU for |x| < 1, 16 ulp on [-3, 3] and
// 64 ulp on [-6, 6] (the rounding of a^2 in the exponent dominates in the
// negative tail), and the negative tail keeps its relative accuracy where
// 1 + erf(x / sqrt(2)) would cancel. About 20 VALU instructions against ~38
// for the library erff's two branches, which made the bf16 kernel VALU-bound.
__device__ inline float gelu_f(float x) {
    const float a = fabsf(x) * 0.70710678118654752f;
    const float t = __builtin_amdgcn_rcpf(fmaf(0.33f, a, 1.0f));
    float s = -0.13534700870513916f;
    s = fmaf(s, t, 0.4602428376674652f);
    s = fmaf(s, t, -0.3511601984500885f);
    s = fmaf(s, t, 0.40851035714149475f);
    s = fmaf(s, t, 0.04721472039818764f);
    s = fmaf(s, t, 0.2012258619070053f);
    s = fmaf(s, t, 0.18295560777187347f);
    s = fmaf(s, t, 0.18635784089565277f);
    const float half_erfc = 0.5f * __builtin_amdgcn_exp2f(-(a * a) * 1.4426950408889634f) * t * s;
    return x * (x >= 0.0f ? 1.0f - half_erfc : half_erfc);
}

// One 16-byte chunk per thread, at any alignment (the device runs with unaligned
// access on); the n % kVec tail by elements. Bound: the copy rate. The loads in flight
// come from the wavefronts (all of a CU's slots), which start and end on their own;
// more chunks per thread start fewer of them, and a wavefront's chunks then wait for
// each other. In us, over buffers beyond the caches: one chunk / two / four / the capped
// grid of 8192 workgroups striding over up to four chunks each that this replaced, bf16:
// 4 Mi elements 5.3 / 6.0 / 6.4 / 5.8, 22.0e6 17.7 / 19.7 / 21.7 / 19.2, 64 Mi 44.8 /
// 50.4 / 49.4 / 55.8; fp32 16 Mi 23.5 / 23.5 / 24.1 / 25.8, 64 Mi 87 / 91 / 91 / 103. One
// element off the boundary, where that form went by elements, the same buffers again
// and again: bf16 22.0e6 16.5 / 23.3 (on it 15.3 / 18.0), fp32 16 Mi 20.4 / 23.1.
template <typename T>
__global__ void __launch_bounds__(256) gelu_kernel(const store_t<T>* __restrict__ x, store_t<T>* __restrict__ y,
                                                   size_t n) {
    using IO = io<T>;
    constexpr int V = IO::kVec;
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t nchunks = n / V;
    for (size_t c = tid; c < nchunks; c += stride) {
        u32x4 raw;
        __builtin_memcpy(&raw, x + c * V, 16);
        float v[V];
        IO::unpack(raw, v);
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] = gelu_f(v[e]);
        raw = IO::pack(v);
        __builtin_memcpy(y + c * V, &raw, 16);
    }
    for (size_t i = nchunks * V + tid; i < n; i += stride) IO::put(y, i, gelu_f(IO::get(x, i)));
}

__device__ inline float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// One wave per row, four rows per workgroup. Three passes over the row (sum,
// sum of squared deviations, normalize): the second and third read it from
// the caches; the two-pass variance has no cancellation for rows whose mean
// is large against their spread.
template <typename T, bool VEC>
__global__ void __launch_bounds__(256) layernorm_kernel(const store_t<T>* __restrict__ x,
                                                        const store_t<T>* __restrict__ gamma,
                                                        const store_t<T>* __restrict__ beta,
                                                        store_t<T>* __restrict__ y, int rows, int D, float eps) {
    using IO = io<T>;
    constexpr int V = VEC ? IO::kVec : 1;
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const store_t<T>* xr = x + (size_t)row * D;
    store_t<T>* yr = y + (size_t)row * D;
    const int nch = D / V;
    auto chunk = [&](const store_t<T>* p, int c, float (&v)[V]) {
        if constexpr (VEC) IO::get16(p, (size_t)c * V, v);
        else v[0] = IO::get(p, (size_t)c);
    };
    float s = 0.f;
    for (int c = lane; c < nch; c += kWave) {
        float v[V];
        chunk(xr, c, v);
#pragma unroll
        for (int e = 0; e < V; ++e) s += v[e];
    }
    const float mean = wave_sum(s) / (float)D;
    float s2 = 0.f;
    for (int c = lane; c < nch; c += kWave) {
        float v[V];
        chunk(xr, c, v);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            const float d = v[e] - mean;
            s2 += d * d;
        }
    }
    const float rstd = 1.0f / sqrtf(wave_sum(s2) / (float)D + eps);
    for (int c = lane; c < nch; c += kWave) {
        float v[V], g[V], b[V];
        chunk(xr, c, v);
        if (gamma) chunk(gamma, c, g);
        if (beta) chunk(beta, c, b);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            float o = (v[e] - mean) * rstd;
            if (gamma) o *= g[e];
            if (beta) o += b[e];
            v[e] = o;
        }
        if constexpr (VEC) IO::put16(yr, (size_t)c * V, v);
        else IO::put(yr, (size_t)c, v[0]);
    }
}

// Rows of at most CAP 16-byte chunks per lane (CAP 8: D <= 4096 bf16/fp16,
// 2048 fp32; CAP 16 for bf16 and fp32: D <= 8192 bf16, 4096 fp32) whose D is
// a multiple of 64 chunks: the row is read once into registers, both
// statistics come from the registers, and it is written once.
template <typename T, int CAP>
__global__ void __launch_bounds__(256) layernorm_reg_kernel(const store_t<T>* __restrict__ x,
                                                            const store_t<T>* __restrict__ gamma,
                                                            const store_t<T>* __restrict__ beta,
                                                            store_t<T>* __restrict__ y, int rows, int D, float eps) {
    using IO = io<T>;
    constexpr int V = IO::kVec;
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const store_t<T>* xr = x + (size_t)row * D;
    store_t<T>* yr = y + (size_t)row * D;
    const int nc = D / (V * kWave);  // chunks per lane, 1..CAP
    // bf16 rows stay in registers as raw 16-byte words, unpacked (a shift) at
    // each of their three uses, so all loads go out before the first
    // conversion and the row takes half the registers of unpacked floats; the
    // bf16 path also issues gamma's and beta's loads with the row's (reading
    // the row itself in place of an absent one, so every load is
    // unconditional), which takes their round trip off the end of the row's
    // work (at CAP 8; at CAP 16 the row alone takes 64 registers and gamma
    // and beta are read at the end). fp32 needs no unpacking, and for fp16 the
    // compiler keeps the converted floats live anyway (228 VGPRs), so both
    // keep the floats.
    constexpr bool RAW = std::is_same<T, bf16_t>::value;
    constexpr bool PF = RAW && CAP <= 8;
    u32x4 raw[RAW ? CAP : 1], graw[PF ? CAP : 1], braw[PF ? CAP : 1];
    float vf[RAW ? 1 : CAP][V];
    auto row_chunk = [&](int j, float (&v)[V]) {
        if constexpr (RAW) IO::unpack(raw[j], v);
        else
#pragma unroll
            for (int e = 0; e < V; ++e) v[e] = vf[j][e];
    };
#pragma unroll
    for (int j = 0; j < CAP; ++j)
        if (j < nc) {
            if constexpr (RAW) raw[j] = IO::raw16(xr, (size_t)(j * kWave + lane) * V);
            else IO::get16(xr, (size_t)(j * kWave + lane) * V, vf[j]);
        }
    if constexpr (PF) {
        const store_t<T>* gp = gamma ? gamma : xr;
        const store_t<T>* bp = beta ? beta : xr;
#pragma unroll
        for (int j = 0; j < CAP; ++j)
            if (j < nc) {
                graw[j] = IO::raw16(gp, (size_t)(j * kWave + lane) * V);
                braw[j] = IO::raw16(bp, (size_t)(j * kWave + lane) * V);
            }
    }
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < CAP; ++j)
        if (j < nc) {
            float v[V];
            row_chunk(j, v);
#pragma unroll
            for (int e = 0; e < V; ++e) s += v[e];
        }
    const float mean = wave_sum(s) / (float)D;
    float s2 = 0.f;
#pragma unroll
    for (int j = 0; j < CAP; ++j)
        if (j < nc) {
            float v[V];
            row_chunk(j, v);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const float d = v[e] - mean;
                s2 += d * d;
            }
        }
    const float rstd = 1.0f / sqrtf(wave_sum(s2) / (float)D + eps);
#pragma unroll
    for (int j = 0; j < CAP; ++j)
        if (j < nc) {
            const size_t off = (size_t)(j * kWave + lane) * V;
            float v[V], g[V], b[V];
            row_chunk(j, v);
            if constexpr (PF) {
                IO::unpack(graw[j], g);
                IO::unpack(braw[j], b);
            } else {
                if (gamma) IO::get16(gamma, off, g);
                if (beta) IO::get16(beta, off, b);
            }
#pragma unroll
            for (int e = 0; e < V; ++e) {
                float o = (v[e] - mean) * rstd;
                if (gamma) o *= g[e];
                if (beta) o += b[e];
                v[e] = o;
            }
            IO::put16(yr, off, v);
        }
}

// Any D from one chunk up, any alignment: W waves share a row (4 / W rows per
// workgroup), up to CAP chunks of 16 bytes per lane in registers, loaded and
// stored unaligned where rows are no whole chunks (the device runs with
// unaligned access on). A row's last chunk is moved back to end with the row:
// its first elements are then another chunk's too, so they are left out of
// the sums, and both lanes write them the same value. Every load of a row is
// complete before its first store (the sums need them all), so y may be x.
// gamma and beta are loaded with the row (the row itself in place of an
// absent one). W > 1 where one wave would need more than 8 chunks per lane,
// and for few rows, where a row's latency is what counts.
template <typename T, int CAP>
__global__ void __launch_bounds__(256) layernorm_row_kernel(const store_t<T>* __restrict__ x,
                                                            const store_t<T>* __restrict__ gamma,
                                                            const store_t<T>* __restrict__ beta,
                                                            store_t<T>* __restrict__ y, int rows, int D, int W,
                                                            float eps) {
    using IO = io<T>;
    constexpr int V = IO::kVec;
    __shared__ float part[2][4];
    const int wave = threadIdx.x >> 6;
    const int per = 4 / W, sub = wave & (W - 1);  // rows per workgroup, this wave's place in its row
    const int own = (int)blockIdx.x * per + wave / W;
    const bool live = own < rows;  // surplus waves only keep the barriers company: they read the last row, store nothing
    const int row = live ? own : rows - 1;
    const int t = sub * kWave + (threadIdx.x & 63);
    const int n = (D + V - 1) / V, skip = n * V - D;  // chunks; elements of the last one that are another's
    const store_t<T>* xr = x + (size_t)row * D;
    store_t<T>* yr = y + (size_t)row * D;
    const store_t<T>* gp = gamma ? gamma : xr;
    const store_t<T>* bp = beta ? beta : xr;
    auto at = [&](int j) { return min((t + j * W * kWave) * V, D - V); };  // first element of the lane's chunk j
    auto raw = [&](const store_t<T>* p, int i) {
        u32x4 c;
        __builtin_memcpy(&c, p + i, 16);
        return c;
    };
    u32x4 rx[CAP], rg[CAP], rb[CAP];
#pragma unroll
    for (int j = 0; j < CAP; ++j) rx[j] = raw(xr, at(j));
#pragma unroll
    for (int j = 0; j < CAP; ++j) {
        rg[j] = raw(gp, at(j));
        rb[j] = raw(bp, at(j));
    }
    // sum of f over the elements that are chunk j's own
    auto sum = [&](auto&& f) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < CAP; ++j) {
            const int c = t + j * W * kWave;
            if (c < n) {
                float v[V];
                IO::unpack(rx[j], v);
                const int from = c == n - 1 ? skip : 0;
#pragma unroll
                for (int e = 0; e < V; ++e) s += e >= from ? f(v[e]) : 0.f;
            }
        }
        return wave_sum(s);
    };
    auto row_sum = [&](float s, int k) {
        if (W == 1) return s;
        if ((threadIdx.x & 63) == 0) part[k][wave] = s;
        __syncthreads();
        float r = 0.f;
        for (int w = 0; w < W; ++w) r += part[k][(wave & ~(W - 1)) + w];
        return r;
    };
    const float mean = row_sum(sum([](float v) { return v; }), 0) / (float)D;
    const float var = row_sum(sum([&](float v) { return (v - mean) * (v - mean); }), 1) / (float)D;
    const float rstd = 1.0f / sqrtf(var + eps);
#pragma unroll
    for (int j = 0; j < CAP; ++j) {
        if (live && t + j * W * kWave < n) {
            float v[V], g[V], b[V];
            IO::unpack(rx[j], v);
            IO::unpack(rg[j], g);
            IO::unpack(rb[j], b);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                float o = (v[e] - mean) * rstd;
                if (gamma) o *= g[e];
                if (beta) o += b[e];
                v[e] = o;
            }
            const u32x4 c = IO::pack(v);
            __builtin_memcpy(yr + at(j), &c, 16);
        }
    }
}

template <typename T>
static int launch_gelu(const void* x, void* y, size_t n, hipStream_t s) {
    constexpr int V = io<T>::kVec;
    size_t blocks = ((n + V - 1) / V + 255) / 256;
    if (blocks > (1u << 23)) blocks = 1u << 23;  // a launch holds fewer than 2^32 threads; grid-stride beyond
    if (blocks == 0) blocks = 1;
    hipLaunchKernelGGL(gelu_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, s, (const store_t<T>*)x,
                       (store_t<T>*)y, n);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

constexpr int kLnFewRows = 2048;  // fewer rows than this leave SIMDs idle at one wave each

// Whether layernorm_row_kernel takes rows of D elements of 16 / V bytes; `vec`: whole
// 16-byte chunks on 16-byte boundaries, nc: chunks per lane where those are even.
// Few rows, or rows that are no whole chunks per lane. In us, one of the other kernels /
// the row kernel: 1 x 3392 bf16 6.3 / 3.5, 64 x 4096 4.9 / 3.8, 8000 x 5003 127 / 50, 6000 x
// 8190 187 / 46, 4000 x 6145 fp32 130 / 45, 5000 x 8192 fp16 59 / 39; 2000 x 4096 bf16 9.9
// / 10.0 (so whole rows of that many stay with one wave each). Not rows that
// layernorm_kernel reads with one load per lane (a chunk, or up to three elements): it
// has less to do per row there. Graph replays: fp16 14495 x 61 5.8 / 9.5, bf16 27475 x 91
// 11.0 / 14.1. The row kernel's time over the other's: by elements 1.2 to 1.8 up to D =
// 64 (fp32 1.0 to 1.2), in 16 bits with 2048 rows or more 1.1 to 1.4 up to 128 and 1.0 to
// 1.15 up to 192, below 1 past that; in chunks with 1024 rows or more 1.0 to 1.13 in 16
// bits, fp32 1.0 to 1.05 up to D = 64 and 0.8 to 1.0 past it.
static bool ln_row_form(int rows, int D, int V, bool vec, int nc, bool cap16) {
    const bool whole = (nc >= 1 && nc <= 8) || (cap16 && nc > 8 && nc <= 16);
    if (D < V || (D + V - 1) / V > 4 * kWave * 8 || (whole && rows >= kLnFewRows / 2)) return false;
    if (vec) return rows < kLnFewRows / 2 || D > (V == 8 ? kWave * V : kWave);
    return D > (V == 8 && rows >= kLnFewRows ? 3 * kWave : kWave);
}

template <typename T>
static int launch_layernorm(const void* x, const void* g, const void* b, void* y, int rows, int D, float eps,
                            hipStream_t s) {
    constexpr int V = io<T>::kVec;
    const bool vec = D % V == 0 && ((((uintptr_t)x | (uintptr_t)y | (uintptr_t)g | (uintptr_t)b) & 15) == 0);
    const dim3 grid((unsigned)((rows + 3) / 4)), block(256);
    const int nc = (vec && D % (V * kWave) == 0) ? D / (V * kWave) : 0;  // chunks per lane
    constexpr bool kCap16 = !std::is_same<T, f16_t>::value;  // fp16 rows past 8 chunks: three passes
    const int n = (D + V - 1) / V;
    if (ln_row_form(rows, D, V, vec, nc, kCap16)) {
        int W = 1;  // waves per row
        while (W < 4 && (n > W * kWave * 8 || ((long)rows * W < kLnFewRows && n > W * kWave))) W *= 2;
        const int cap = (n + W * kWave - 1) / (W * kWave);
        const dim3 g2((unsigned)(((long)rows * W + 3) / 4));
#define PYC_LN(C)                                                                                              \
    hipLaunchKernelGGL((layernorm_row_kernel<T, C>), g2, block, 0, s, (const store_t<T>*)x, (const store_t<T>*)g, \
                       (const store_t<T>*)b, (store_t<T>*)y, rows, D, W, eps)
        if (cap <= 1) PYC_LN(1);
        else if (cap <= 2) PYC_LN(2);
        else if (cap <= 4) PYC_LN(4);
        else PYC_LN(8);
#undef PYC_LN
        return hipGetLastError() == hipSuccess ? 0 : -2;
    }
    if (nc >= 1 && nc <= 8)
        hipLaunchKernelGGL((layernorm_reg_kernel<T, 8>), grid, block, 0, s, (const store_t<T>*)x,
                           (const store_t<T>*)g, (const store_t<T>*)b, (store_t<T>*)y, rows, D, eps);
    else if (kCap16 && nc > 8 && nc <= 16)
        hipLaunchKernelGGL((layernorm_reg_kernel<T, kCap16 ? 16 : 8>), grid, block, 0, s, (const store_t<T>*)x,
                           (const store_t<T>*)g, (const store_t<T>*)b, (store_t<T>*)y, rows, D, eps);
    else if (vec)
        hipLaunchKernelGGL((layernorm_kernel<T, true>), grid, block, 0, s, (const store_t<T>*)x,
                           (const store_t<T>*)g, (const store_t<T>*)b, (store_t<T>*)y, rows, D, eps);
    else
        hipLaunchKernelGGL((layernorm_kernel<T, false>), grid, block, 0, s, (const store_t<T>*)x,
                           (const store_t<T>*)g, (const store_t<T>*)b, (store_t<T>*)y, rows, D, eps);
    return hipGetLastError() == hipSuccess ? 0 : -2;
}

}  // namespace pyc

// dtype: 0 fp32, 1 bf16, 2 fp16. 0, -1 (bad arguments), -2 (HIP error).
extern "C" int pyc_hip_gelu_launch(int dtype, size_t n, const void* x, void* y, void* stream) {
    using namespace pyc;
    if (n == 0) return 0;
    if (!x || !y) return -1;
    hipStream_t s = (hipStream_t)stream;
    switch (dtype) {
        case 0: return launch_gelu<float>(x, y, n, s);
        case 1: return launch_gelu<bf16_t>(x, y, n, s);
        case 2: return launch_gelu<f16_t>(x, y, n, s);
        default: return -1;
    }
}

// 1 where layernorm_row_kernel takes the call, else 0 (host only; the pointers are
// looked at for their alignment).
extern "C" int pyc_hip_layernorm_row_form(int dtype, int rows, int D, const void* x, const void* gamma,
                                          const void* beta, const void* y) {
    using namespace pyc;
    const int V = dtype == 0 ? 4 : 8;
    const bool vec = D % V == 0 && ((((uintptr_t)x | (uintptr_t)y | (uintptr_t)gamma | (uintptr_t)beta) & 15) == 0);
    const int nc = (vec && D % (V * kWave) == 0) ? D / (V * kWave) : 0;
    return ln_row_form(rows, D, V, vec, nc, dtype != 2);
}

extern "C" int pyc_hip_layernorm_launch(int dtype, int rows, int D, float eps, const void* x, const void* gamma,
                                        const void* beta, void* y, void* stream) {
    using namespace pyc;
    if (rows == 0) return 0;
    if (rows < 0 || D <= 0 || !x || !y || !(eps >= 0.f)) return -1;
    hipStream_t s = (hipStream_t)stream;
    switch (dtype) {
        case 0: return launch_layernorm<float>(x, gamma, beta, y, rows, D, eps, s);
        case 1: return launch_layernorm<bf16_t>(x, gamma, beta, y, rows, D, eps, s);
        case 2: return launch_layernorm<f16_t>(x, gamma, beta, y, rows, D, eps, s);
        default: return -1;
    }
}

// Registry figures: GELU (kid 0) and the register-resident LayerNorm at up
// to 8 chunks per lane (kid 1), 256-thread workgroups, no LDS; dtype 0 fp32,
// 1 bf16, 2 fp16. Waves per SIMD from each instance's register count.
extern "C" int pyc_hip_kinfo_eltwise(int kid, int dtype, pyc_hip_kinfo* out) {
    using namespace pyc;
    if (!out || dtype < 0 || dtype > 2 || kid < 0 || kid > 1) return -1;
    out->threads = 256;
    out->lds_bytes = 0;
    if (kid == 0) {
        out->name = "gelu_kernel";
        out->waves_per_simd = 8;
        out->fn = dtype == 0 ? reinterpret_cast<const void*>(&gelu_kernel<float>)
                  : dtype == 1 ? reinterpret_cast<const void*>(&gelu_kernel<bf16_t>)
                               : reinterpret_cast<const void*>(&gelu_kernel<f16_t>);
    } else {
        out->name = "layernorm_reg_kernel<8>";
        out->waves_per_simd = dtype == 0 ? 7 : dtype == 1 ? 3 : 4;
        out->fn = dtype == 0 ? reinterpret_cast<const void*>(&layernorm_reg_kernel<float, 8>)
                  : dtype == 1 ? reinterpret_cast<const void*>(&layernorm_reg_kernel<bf16_t, 8>)
                               : reinterpret_cast<const void*>(&layernorm_reg_kernel<f16_t, 8>);
    }
    return 0;
}
