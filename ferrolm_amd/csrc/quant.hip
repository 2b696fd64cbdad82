// Load-time quantization on the device: QMatrix::quantize (src/quant.rs:78-143)
// and the pieces of the AWQ alpha search (src/awq.rs:152-217): the column
// scaling, the reference's matmuls in their exact accumulation order, and the
// mean squared error summed in output order.
//
// Everything here reproduces the reference's bits. The quantizer's clip search
// is per (row, group) sequential arithmetic (f32 divide and round, f64 error),
// one lane per (row, group); the matmuls are one FMA chain per output, in k
// order, as src/kernels.rs:249-289 (bf16) and src/quant.rs:285-299 (per-group
// chains, then acc = fma(group sum, scale, acc)). Contraction is off for the
// whole build, so only the explicit fmaf calls fuse.
#include "seqsum.h"

#include <algorithm>

namespace fg {

// f32::round then `as i32` (saturating, NaN to 0), then clamp(lo, hi)
__device__ __forceinline__ int clamp_code(float t, int lo, int hi) {
    if (!(t == t)) return 0;
    if (t >= (float)hi) return hi;
    if (t <= (float)lo) return lo;
    return (int)t;
}

// One wave per (32-row panel, two groups): lane l takes row 32 p + l % 32 of
// group 2 y + l / 32; the weights are multiplied by their columns' cs first
// (cs not null). Writes the reference's QMatrix layout: scales
// [panel][group][32]; codes per panel and input position, int8 one byte per
// row, int4 byte c = row c (low nibble) | row c + 16 (high nibble), each + 8;
// or (qt not null) the codes for k_mm_exact, [panel][input / 4][row][4 x int8].
// Groups whose every clip gives a non-finite error keep scale 0 and codes 0
// (the reference would keep the previous group's codes there).
//
// Bound: VALU (about 15 operations per weight and clip, three of them f64).
// The code round(v / scale), half away from zero, is that of the product with
// 1 / scale unless the product lies within NEAR of a rounding boundary (the two
// differ by under 3 * 2^-24 of the largest code that is not clamped, 2.9e-6
// and 2.5e-5): only a wave with such a lane divides. 16384 x 2048 int4 with
// importances: 821 -> 166 us.
template <bool Q8, bool IMP>
__global__ __launch_bounds__(64) void k_quantize(const float* __restrict__ w, const float* __restrict__ cs,
                                                 const float* __restrict__ imp, int cols, uint8_t* __restrict__ q,
                                                 uint32_t* __restrict__ qt, float* __restrict__ s) {
    constexpr int lo = Q8 ? -127 : -8, hi = Q8 ? 127 : 7, nclips = Q8 ? 6 : 11;
    constexpr float kNear = Q8 ? 0.4999f : 0.49999f;
    const float clips8[6] = {1.0f, 0.98f, 0.96f, 0.94f, 0.92f, 0.9f};
    const float clips4[11] = {1.0f, 0.95f, 0.9f, 0.85f, 0.8f, 0.75f, 0.7f, 0.65f, 0.6f, 0.55f, 0.5f};
    const int lane = threadIdx.x, c = lane & 31, groups = cols >> 5;
    const int p = blockIdx.x, g = blockIdx.y * 2 + (lane >> 5);
    const bool live = g < groups;
    const int gc = live ? g : groups - 1;  // lanes past the last group work on a valid copy, write nothing
    const float* src = w + ((size_t)p * 32 + c) * cols + (size_t)gc * 32;
    float v[32];
    double im[IMP ? 32 : 1];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float4 a = ((const float4*)src)[i];
        v[4 * i] = a.x;
        v[4 * i + 1] = a.y;
        v[4 * i + 2] = a.z;
        v[4 * i + 3] = a.w;
    }
    if (cs)
#pragma unroll
        for (int i = 0; i < 32; i++) v[i] = v[i] * cs[gc * 32 + i];
    if constexpr (IMP)
#pragma unroll
        for (int i = 0; i < 32; i++) im[i] = (double)imp[gc * 32 + i];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; i++) amax = fmaxf(amax, fabsf(v[i]));
    // 1 / scale where it is exact to half an ulp (a NaN, which divides, at the ends of the range)
    auto inverse = [](float scale) {
        return scale > 0x1p-100f && scale < 0x1p100f ? 1.0f / scale : scale > 0.0f ? __uint_as_float(0x7FC00000u) : 0.0f;
    };
    // the code of x at a scale, as a float
    auto code_of = [&](float x, float scale, float inv) -> float {
        const float r = x * inv, k = rintf(r);
        float t = k;
        if (__any(!(fabsf(r - k) < kNear))) {  // (a NaN is near: the division decides)
            asm volatile("");  // kept a branch: the division is rarely wanted
            t = (float)clamp_code(roundf(x / scale), lo, hi);
        }
        return fminf(fmaxf(t, (float)lo), (float)hi);
    };
    double best = INFINITY;
    float best_scale = 0.0f;
    for (int ci = 0; ci < nclips; ci++) {
        float clip = Q8 ? clips8[0] : clips4[0];
#pragma unroll
        for (int j = 1; j < nclips; j++) clip = ci == j ? (Q8 ? clips8[j] : clips4[j]) : clip;
        const float scale = clip * amax / (float)hi, inv = inverse(scale);
        double err = 0.0;
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const double d = (double)(v[i] - code_of(v[i], scale, inv) * scale);
            err = err + (IMP ? d * d * im[i] : d * d);
        }
        if (amax > 0.0f && err < best) {
            best = err;
            best_scale = scale;
        }
    }
    if (live) s[((size_t)p * groups + g) * 32 + c] = best_scale;
    // the chosen clip's codes (a function of the scale: recomputed)
    const float inv = inverse(best_scale);
    int code[32];
#pragma unroll
    for (int i = 0; i < 32; i++) {
        const float t = code_of(v[i], best_scale, inv);
        code[i] = best_scale > 0.0f ? (int)t : 0;
    }
    if (qt) {
        uint32_t* o = qt + ((size_t)p * cols + (size_t)gc * 32) * 8 + c;
        if (live)
#pragma unroll
            for (int i = 0; i < 8; i++)
                o[i * 32] = (code[4 * i] & 255) | (code[4 * i + 1] & 255) << 8 | (code[4 * i + 2] & 255) << 16 |
                            (uint32_t)(code[4 * i + 3] & 255) << 24;
        return;
    }
    uint8_t* qp = q + ((size_t)p * cols + (size_t)gc * 32) * (Q8 ? 32 : 16);
#pragma unroll
    for (int i = 0; i < 32; i++) {
        if (Q8) {
            if (live) qp[i * 32 + c] = (uint8_t)(int8_t)code[i];
        } else {
            const int up = __shfl_down(code[i], 16, 32);  // row c + 16's code
            if (live && c < 16) qp[i * 16 + c] = (uint8_t)((code[i] + 8) | ((up + 8) << 4));
        }
    }
}

// dst[r][c] = src[r][c] / s[c]
__global__ __launch_bounds__(256) void k_scale_cols(const float* __restrict__ src, int64_t n, int k,
                                                    const float* __restrict__ s, float* __restrict__ dst) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = src[i] / s[i % k];
}

// W (rows x K f32), rounded to bf16, in k_mm_exact's layout: [panel][input / 4][row][4 x bf16].
// One workgroup per (panel, 128 inputs), turned through LDS.
__global__ __launch_bounds__(256) void k_pack_bf16(const float* __restrict__ w, int K, uint2* __restrict__ o) {
    __shared__ float t[32][132];
    const int p = blockIdx.x, k0 = blockIdx.y * 128;
    for (int e = threadIdx.x; e < 32 * 128; e += 256) {
        const int r = e >> 7, k = k0 + (e & 127);
        if (k < K) t[r][e & 127] = w[((size_t)p * 32 + r) * K + k];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 32 * 32; e += 256) {
        const int r = e & 31, k4 = (e >> 5) * 4;
        if (k0 + k4 >= K) continue;
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 4; i++) h[i] = __builtin_bit_cast(uint16_t, (__bf16)t[r][k4 + i]);
        o[((size_t)p * (K >> 2) + ((k0 + k4) >> 2)) * 32 + r] = make_uint2(h[0] | h[1] << 16, h[2] | h[3] << 16);
    }
}

// y (m x rows) = x (m x K) W^T with the reference's accumulation order, one
// thread per output column j and kMmRows rows of x (blockIdx.y). wt holds W by
// panels of 32 rows, four inputs of a row together (k_pack_bf16, k_quantize's qt).
//   BF: bf16 weights; acc = fma(x_k, w_jk, acc) for k = 0, 1, ...
//   else: codes; per group g a chain gs = fma(x_k, code_jk, gs) over its 32
//       positions, then acc = fma(gs, s_jg, acc).
// Bound: the f32 FMAs (39 T/s on this card without packed ones). The rows of x
// are the same for a whole wave, so they come through scalar loads and are the
// FMA's scalar operand; a lane's weights are one 4- or 8-byte load per four
// inputs. 256 rows x 6144 x 2048: int4 codes 524 -> 177 us (one LDS
// read per FMA and a byte load per input before). The registers hold only a
// quarter of a group's rows at a time, and each part waited for the scalar
// cache to miss in turn; so a group's start touches every line of the next
// group's rows, which then miss together, once: 177 -> 152 us (64 groups of
// 288 instructions in three waves a SIMD are 92).
constexpr int kMmRows = 8;
template <bool BF>
__global__ __launch_bounds__(256) void k_mm_exact(const float* __restrict__ x, int m, int K,
                                                  const uint32_t* __restrict__ wt, const float* __restrict__ s,
                                                  int rows, float* __restrict__ y) {
    const int j = blockIdx.x * 256 + threadIdx.x, i0 = blockIdx.y * kMmRows;
    const int jc = min(j, rows - 1), p = jc >> 5, c = jc & 31, groups = K >> 5;
    const float* xr[kMmRows];  // rows past the last one re-read it
#pragma unroll
    for (int i = 0; i < kMmRows; i++) xr[i] = x + (size_t)min(i0 + i, m - 1) * K;
    float acc[kMmRows];
#pragma unroll
    for (int i = 0; i < kMmRows; i++) acc[i] = 0.0f;
    const size_t at = (size_t)p * (K >> 2) * 32 + c;
    const uint2* wb = (const uint2*)wt + at;
    const uint32_t* wq = wt + at;
    const float* sp = s + (size_t)p * groups * 32 + c;
    uint2 nb[8];
    uint32_t nq[8];
    float ns = 0.0f;
    auto fetch = [&](int g) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            if (BF)
                nb[e] = wb[((size_t)g * 8 + e) * 32];
            else
                nq[e] = wq[((size_t)g * 8 + e) * 32];
        }
        if (!BF) ns = sp[(size_t)g * 32];
    };
    // a word of each 64-byte line of group g's part of the rows
    auto warm = [&](int g) {
        const int at = min(g, groups - 1) * 32;
        float u[kMmRows], v[kMmRows];
#pragma unroll
        for (int i = 0; i < kMmRows; i++) {
            u[i] = xr[i][at];
            v[i] = xr[i][at + 16];
        }
#pragma unroll
        for (int i = 0; i < kMmRows; i++) asm volatile("" ::"s"(u[i]), "s"(v[i]));
    };
    fetch(0);
    for (int g = 0; g < groups; g++) {
        uint2 cb[8];
        uint32_t cq[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            if (BF)
                cb[e] = nb[e];
            else
                cq[e] = nq[e];
        }
        const float sc = ns;
        if (g + 1 < groups) fetch(g + 1);
        warm(g + 1);
        float gs[kMmRows];
#pragma unroll
        for (int i = 0; i < kMmRows; i++) gs[i] = BF ? acc[i] : 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float wv[4];
            if (BF) {
                wv[0] = __uint_as_float(cb[e].x << 16);
                wv[1] = __uint_as_float(cb[e].x & 0xFFFF0000u);
                wv[2] = __uint_as_float(cb[e].y << 16);
                wv[3] = __uint_as_float(cb[e].y & 0xFFFF0000u);
            } else {
#pragma unroll
                for (int b = 0; b < 4; b++) wv[b] = (float)(int8_t)(cq[e] >> (8 * b));
            }
#pragma unroll
            for (int b = 0; b < 4; b++)
#pragma unroll
                for (int i = 0; i < kMmRows; i++) gs[i] = fmaf(xr[i][g * 32 + e * 4 + b], wv[b], gs[i]);
        }
#pragma unroll
        for (int i = 0; i < kMmRows; i++) acc[i] = BF ? gs[i] : fmaf(gs[i], sc, acc[i]);
    }
    if (j < rows)
#pragma unroll
        for (int i = 0; i < kMmRows; i++)
            if (i0 + i < m) y[(size_t)(i0 + i) * rows + j] = acc[i];
}

// err[b] = sum over t of (f64)(y_b[t] - yref[t])^2 in t order from 0, divided
// by n, for the sequences y_b = y + b * ystride. The reference sums
// sequentially in f64 (each term is exact: the square of an f32 difference),
// so every rounding counts; seqsum.h turns steps into maps that compose. In
// three launches: the plain sum of each chunk of 8192 terms; each chunk's map
// for the binade that those sums predict; and one workgroup per sequence that
// applies the maps in order, and scans the chunks where the running sum is not
// in the predicted binade or leaves it (about one chunk per binade).
// 11 sequences of 1,572,864 terms: 8942 us with one lane adding (3.3 ns a
// term, the add's latency) -> 365 us (sums 20, maps 74, the walk 271).
constexpr int kErrChunk = 8192, kErrThreads = 1024, kErrPer = kErrChunk / kErrThreads;
struct ErrWork {
    double* sum;            // [sequence][chunk]
    SeqMap<double>* map;    // [sequence][chunk]
    int* e;                 // [sequence][chunk]: the map's binade
};
__host__ __device__ inline ErrWork err_work(void* p, int count, int chunks) {
    const size_t n = (size_t)count * chunks;
    return {(double*)p, (SeqMap<double>*)((char*)p + n * 8), (int*)((char*)p + n * 24)};
}
__device__ __forceinline__ double err_term(const float* y, const float* yref, int64_t i) {
    const double d = (double)(y[i] - yref[i]);
    return d * d;
}
__device__ double err_block_sum(double v, double* red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < kErrThreads / 64; w++) t += red[w];
    return t;
}

__global__ __launch_bounds__(kErrThreads) void k_err_sums(const float* __restrict__ y, int64_t ystride,
                                                          const float* __restrict__ yref, int64_t n, ErrWork w) {
    __shared__ double red[kErrThreads / 64];
    const float* yb = y + (size_t)blockIdx.y * ystride;
    const int64_t t0 = (int64_t)blockIdx.x * kErrChunk;
    double v = 0.0;
#pragma unroll
    for (int c = 0; c < kErrPer; c++) {
        const int64_t i = t0 + c * kErrThreads + threadIdx.x;
        if (i < n) v += err_term(yb, yref, i);
    }
    v = err_block_sum(v, red);
    if (threadIdx.x == 0) w.sum[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = v;
}

__global__ __launch_bounds__(kErrThreads) void k_err_maps(const float* __restrict__ y, int64_t ystride,
                                                          const float* __restrict__ yref, int64_t n, ErrWork w) {
    __shared__ double red[kErrThreads / 64];
    __shared__ SeqMap<double> tot[kErrThreads / 64];
    const float* yb = y + (size_t)blockIdx.y * ystride;
    const size_t row = (size_t)blockIdx.y * gridDim.x;
    double before = 0.0;
    for (int c = threadIdx.x; c < (int)blockIdx.x; c += kErrThreads) before += w.sum[row + c];
    before = err_block_sum(before, red);
    uint64_t mant;
    int e;
    seq_split(before, mant, e);
    const int64_t t0 = (int64_t)blockIdx.x * kErrChunk + threadIdx.x * kErrPer;
    SeqMap<double> own = {0, 0};
    bool odd = !seq_finite(before);
#pragma unroll
    for (int c = 0; c < kErrPer; c++)
        if (t0 + c < n) {
            const double x = err_term(yb, yref, t0 + c);
            odd |= !seq_finite(x);
            own = seq_then<double>(own, seq_step<double, double>(x, e));
        }
    const SeqMap<double> inc = seq_wave_scan<double>(own);
    if ((threadIdx.x & 63) == 63) tot[threadIdx.x >> 6] = inc;
    odd = __syncthreads_or(odd);
    if (threadIdx.x == 0) {
        SeqMap<double> all = tot[0];
        for (int v = 1; v < kErrThreads / 64; v++) all = seq_then<double>(all, tot[v]);
        w.map[row + blockIdx.x] = all;
        w.e[row + blockIdx.x] = odd ? -1 : e;  // -1: no map, the chunk is scanned
    }
}

__global__ __launch_bounds__(kErrThreads) void k_err_walk(const float* __restrict__ y, int64_t ystride,
                                                          const float* __restrict__ yref, int64_t n, int chunks,
                                                          ErrWork w, double* __restrict__ out) {
    __shared__ SeqShared<double> sh;
    __shared__ SeqMap<double> map[kErrThreads];
    __shared__ int es[kErrThreads];
    const float* yb = y + (size_t)blockIdx.x * ystride;
    const size_t row = (size_t)blockIdx.x * chunks;
    double S = 0.0;
    for (int c0 = 0; c0 < chunks; c0 += kErrThreads) {
        const int nc = min(kErrThreads, chunks - c0);
        __syncthreads();
        if ((int)threadIdx.x < nc) {
            map[threadIdx.x] = w.map[row + c0 + threadIdx.x];
            es[threadIdx.x] = w.e[row + c0 + threadIdx.x];
        }
        __syncthreads();
        for (int c = 0; c < nc; c++) {
            uint64_t m;
            int e;
            seq_split(S, m, e);
            const int64_t end = (int64_t)m + (int64_t)seq_move<double>(map[c], (int64_t)m);
            if (e == es[c] && end < (1ll << 53)) {
                S = seq_value(end, e);
                continue;
            }
            const int64_t t0 = (int64_t)(c0 + c) * kErrChunk;
            seq_scan<SEQ_SUM, kErrPer, double>((int)min((int64_t)kErrChunk, n - t0), S, 0.0,
                                               [&](int i) { return err_term(yb, yref, t0 + i); }, sh);
        }
    }
    if (threadIdx.x == 0) out[blockIdx.x] = S / (double)n;
}

void launch_quantize(hipStream_t st, int kind, int rows, int cols, const float* w, const float* cs, const float* imp,
                     uint8_t* q, uint32_t* qt, float* s) {
    const dim3 grid(rows / 32, (cols / 32 + 1) / 2);
    auto run = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(64), 0, st, w, cs, imp, cols, q, qt, s); };
    if (kind == INT8)
        imp ? run(k_quantize<true, true>) : run(k_quantize<true, false>);
    else
        imp ? run(k_quantize<false, true>) : run(k_quantize<false, false>);
}

void launch_scale_cols(hipStream_t st, const float* src, int64_t n, int k, const float* s, float* dst) {
    const int64_t blocks = std::min<int64_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_scale_cols, dim3((unsigned)blocks), dim3(256), 0, st, src, n, k, s, dst);
}

void launch_pack_bf16(hipStream_t st, const float* w, int rows, int K, uint32_t* wt) {
    hipLaunchKernelGGL(k_pack_bf16, dim3(rows / 32, (K + 127) / 128), dim3(256), 0, st, w, K, (uint2*)wt);
}

void launch_mm_exact(hipStream_t st, int kind, const float* x, int m, int K, const uint32_t* wt, const float* s,
                     int rows, float* y) {
    constexpr int kMost = 65535 * kMmRows;  // a grid's y is at most 65,535
    for (int i = 0; i < m; i += kMost) {
        const int mi = std::min(kMost, m - i);
        const float* xi = x + (size_t)i * K;
        float* yi = y + (size_t)i * rows;
        const dim3 grid((rows + 255) / 256, (mi + kMmRows - 1) / kMmRows);
        if (kind == BF16)
            hipLaunchKernelGGL((k_mm_exact<true>), grid, dim3(256), 0, st, xi, mi, K, wt, s, rows, yi);
        else
            hipLaunchKernelGGL((k_mm_exact<false>), grid, dim3(256), 0, st, xi, mi, K, wt, s, rows, yi);
    }
}

size_t sq_err_work(int count, int64_t n) { return (size_t)count * ((n + kErrChunk - 1) / kErrChunk) * 32; }

void launch_sq_err(hipStream_t st, const float* y, int64_t ystride, int count, const float* yref, int64_t n,
                   void* work, double* out) {
    const int chunks = (int)((n + kErrChunk - 1) / kErrChunk);
    const ErrWork w = err_work(work, count, chunks);
    hipLaunchKernelGGL(k_err_sums, dim3(chunks, count), dim3(kErrThreads), 0, st, y, ystride, yref, n, w);
    hipLaunchKernelGGL(k_err_maps, dim3(chunks, count), dim3(kErrThreads), 0, st, y, ystride, yref, n, w);
    hipLaunchKernelGGL(k_err_walk, dim3(count), dim3(kErrThreads), 0, st, y, ystride, yref, n, chunks, w, out);
}

}  // namespace fg
