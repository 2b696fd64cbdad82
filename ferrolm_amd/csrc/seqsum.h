// Sequential sums, exactly, by a whole workgroup. The reference adds (or
// subtracts) long lists of non-negative terms one after the other in f32 or
// f64, and the rounding of every step is part of its result, so the list
// cannot simply be split. But while the running sum S stays in one binade its
// ulp u is fixed and S = M u for an integer M, so adding x = (n + f) u moves M
// by n or n + 1: rounded by f, and in a tie (f = 1/2) by the parity of M + n.
// A step is thus a map on M given by two numbers, its moves for an even and
// for an odd M, and such maps compose associatively: a workgroup scans a tile
// of terms at once. The one step that leaves the binade is found from the scan
// (M is monotone), done by the floating-point unit itself, and the scan resumes
// after it in the new binade. The result has the bits of the sequential loop
// for every finite list; a list with an infinity or NaN takes that loop.
//
// What bounds it: the scan's latency (about 1 us a tile of 8192 terms) and one
// more round for each binade crossed, most of them within the first terms,
// which are therefore added directly. One lane walking the list from LDS took
// about 50 ns a term (a dependent LDS read and a branch each).
#pragma once
#include "internal.h"

namespace fg {

template <class F>
struct SeqT;
template <>
struct SeqT<float> {
    using W = uint32_t;
    using M = int32_t;
    static constexpr int kBits = 24, kBias = 150;
    static constexpr W kSat = 1u << 30;  // moves are clamped here (past any binade): sums of two still fit
};
template <>
struct SeqT<double> {
    using W = uint64_t;
    using M = int64_t;
    static constexpr int kBits = 53, kBias = 1075;
    static constexpr W kSat = 1ull << 61;
};

// x = mant * 2^(e - kBias of its type), e >= 1 (x finite, its sign ignored)
__device__ __forceinline__ void seq_split(float x, uint32_t& mant, int& e) {
    const uint32_t b = __float_as_uint(x);
    const int ex = (b >> 23) & 255;
    mant = (b & 0x7FFFFFu) | (ex ? 0x800000u : 0u);
    e = ex ? ex : 1;
}
__device__ __forceinline__ void seq_split(double x, uint64_t& mant, int& e) {
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    const int ex = (int)((b >> 52) & 2047);
    mant = (b & 0xFFFFFFFFFFFFFull) | (ex ? 1ull << 52 : 0ull);
    e = ex ? ex : 1;
}
__device__ __forceinline__ bool seq_finite(float x) { return (__float_as_uint(x) & 0x7F800000u) != 0x7F800000u; }
__device__ __forceinline__ bool seq_finite(double x) {
    return ((uint64_t)__double_as_longlong(x) & 0x7FF0000000000000ull) != 0x7FF0000000000000ull;
}
__device__ __forceinline__ float seq_value(int32_t m, int e) { return ldexpf((float)m, e - 150); }
__device__ __forceinline__ double seq_value(int64_t m, int e) { return ldexp((double)m, e - 1075); }

template <class F>
struct SeqMap {
    typename SeqT<F>::W d0, d1;  // the move of an even and of an odd M
};

// One step by x while S has ulp 2^(e - kBias). The same map serves a subtraction (M - n - f
// rounds to M - n or M - n - 1, to the even one in a tie, and n's parity is -n's).
template <class F, class V>
__device__ __forceinline__ SeqMap<F> seq_step(V x, int e) {
    using W = typename SeqT<F>::W;
    constexpr int kBitsV = SeqT<V>::kBits;
    typename SeqT<V>::W mv;
    int ex;
    seq_split(x, mv, ex);
    const W mant = mv;
    const int shift = ex - SeqT<V>::kBias - (e - SeqT<F>::kBias);
    W n, up = 0, tie = 0;
    if (shift >= 0) {
        constexpr int kMost = (sizeof(W) == 4 ? 30 : 61) - kBitsV;  // mant << kMost stays below kSat
        n = mant == 0 ? 0 : shift > kMost ? SeqT<F>::kSat : mant << shift;
    } else {
        const int r = -shift;
        if (r > kBitsV) {  // below half an ulp
            n = 0;
        } else {
            n = mant >> r;
            const W rem = mant & (((W)1 << r) - 1), half = (W)1 << (r - 1);
            up = rem > half;
            tie = rem == half;
        }
    }
    return {n + (up | (tie & n & 1)), n + (up | (tie & ((n + 1) & 1)))};
}

template <class F>
__device__ __forceinline__ SeqMap<F> seq_then(SeqMap<F> f, SeqMap<F> g) {
    using W = typename SeqT<F>::W;
    const W a = f.d0 + ((f.d0 & 1) ? g.d1 : g.d0), b = f.d1 + ((f.d1 & 1) ? g.d0 : g.d1);
    return {a < SeqT<F>::kSat ? a : SeqT<F>::kSat, b < SeqT<F>::kSat ? b : SeqT<F>::kSat};
}
template <class F>
__device__ __forceinline__ typename SeqT<F>::W seq_move(SeqMap<F> f, typename SeqT<F>::M m) {
    return (m & 1) ? f.d1 : f.d0;
}

__device__ __forceinline__ uint32_t seq_up(uint32_t v, int d) { return __shfl_up(v, d, 64); }
__device__ __forceinline__ uint64_t seq_up(uint64_t v, int d) {
    return (uint64_t)__shfl_up((unsigned long long)v, d, 64);
}
__device__ __forceinline__ float seq_lane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double seq_lane(double v, int l) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Inclusive scan of the maps over a wave, in lane order.
template <class F>
__device__ __forceinline__ SeqMap<F> seq_wave_scan(SeqMap<F> f) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const SeqMap<F> p = {seq_up(f.d0, d), seq_up(f.d1, d)};
        if (lane >= d) f = seq_then<F>(p, f);
    }
    return f;
}

template <class F>
struct SeqShared {
    SeqMap<F> tot[2][16];
    F s;
    int start, stop;
};

// Visits the terms value(0), value(1), ... value(n - 1) in order with the running sum S, as one
// thread would:
//   SEQ_SUM    S += x; never stops
//   SEQ_REACH  S += x; stops at the first S >= thr (thr > 0)
//   SEQ_WALK   stops at the first S < x, with S as it was; otherwise S -= x (S >= 0)
// Returns the index it stopped at, or n. Every thread of the workgroup (T threads, whole waves,
// at most 16) calls it with the same n and S and ends with the same result; the terms are
// non-negative. C terms per thread and tile.
enum { SEQ_SUM = 0, SEQ_REACH = 1, SEQ_WALK = 2 };
template <int MODE, int C, class F, class Value>
__device__ int seq_scan(int n, F& S, F thr, Value value, SeqShared<F>& sh) {
    using T = SeqT<F>;
    using M = typename T::M;
    using V = decltype(value(0));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
    auto visit = [&](F& s, F x) -> bool {
        if (MODE == SEQ_WALK) {
            if (s < x) return true;
            s -= x;
            return false;
        }
        s += x;
        return MODE == SEQ_REACH && s >= thr;
    };
    // the first terms one by one: most of the binades are crossed here
    const int head = min(n, 32);
    {
        const V v0 = lane < head ? value(lane) : (V)0;
        for (int j = 0; j < head; j++)
            if (visit(S, (F)seq_lane(v0, j))) return j;
    }
    int buf = 0;
    const int tile = (int)blockDim.x * C;
    for (int t0 = head; t0 < n; t0 += tile) {
        V x[C];
        bool odd = false;  // an infinity or NaN
#pragma unroll
        for (int c = 0; c < C; c++) {
            const int i = t0 + tid * C + c;
            x[c] = i < n ? value(i) : (V)0;
            odd |= !seq_finite(x[c]);
        }
        odd = __syncthreads_or(odd);
        int start = 0;
        while (start < tile) {
            if (odd || !seq_finite(S)) {
                __syncthreads();
                if (tid == 0) {
                    F s = S;
                    int at = n;
                    for (int i = t0 + start; i < n; i++)
                        if (visit(s, (F)value(i))) {
                            at = i;
                            break;
                        }
                    sh.s = s;
                    sh.stop = at;
                }
                __syncthreads();
                S = sh.s;
                const int at = sh.stop;
                __syncthreads();
                return at;
            }
            typename T::W mant;
            int e;
            seq_split(S, mant, e);
            M m = (M)mant;
            constexpr M kLow = (M)1 << (T::kBits - 1), kTop = (M)1 << T::kBits;
            M bound = kTop;
            if (MODE == SEQ_WALK) {
                if (m == kLow && e > 1) {  // a power of two: the binade below, whose ulp its successors have
                    m = kTop;
                    e--;
                }
                bound = e > 1 ? kLow : -1;
            }
            if (MODE == SEQ_REACH) {
                const double q = ceil(ldexp((double)thr, T::kBias - e));  // the first M that reaches thr
                if (q < (double)bound) bound = (M)q;
            }
            auto past = [&](M v) { return MODE == SEQ_WALK ? v <= bound : v >= bound; };
            auto moved = [&](M v, SeqMap<F> f) -> M {
                return MODE == SEQ_WALK ? v - (M)seq_move<F>(f, v) : v + (M)seq_move<F>(f, v);
            };
            SeqMap<F> own = {0, 0};
            if (tid * C + C > start)
#pragma unroll
                for (int c = 0; c < C; c++)
                    if (tid * C + c >= start) own = seq_then<F>(own, seq_step<F, V>(x[c], e));
            const SeqMap<F> inc = seq_wave_scan<F>(own);
            SeqMap<F> exc = {seq_up(inc.d0, 1), seq_up(inc.d1, 1)};
            if (lane == 0) exc = {0, 0};
            if (lane == 63) sh.tot[buf][wave] = inc;
            __syncthreads();
            M end = m, mw = m;
            for (int w = 0; w < nw; w++) {
                if (w == wave) mw = end;
                if (!past(end)) end = moved(end, sh.tot[buf][w]);
            }
            if (!past(end)) {
                S = seq_value(end, e);
                buf ^= 1;
                break;
            }
            // exactly one thread's terms hold the step that leaves the binade (or stops)
            if (!past(mw)) {
                M mt = moved(mw, exc);
                if (!past(mt) && past(moved(mt, own))) {
                    bool found = false;
#pragma unroll
                    for (int c = 0; c < C; c++)
                        if (!found && tid * C + c >= start) {
                            const M m2 = moved(mt, seq_step<F, V>(x[c], e));
                            found = past(m2);
                            if (found) {
                                F s = seq_value(mt, e);
                                const bool stop = visit(s, (F)x[c]);
                                sh.s = s;
                                sh.start = tid * C + c + 1;
                                sh.stop = stop ? t0 + tid * C + c : -1;
                            }
                            mt = m2;
                        }
                }
            }
            __syncthreads();
            S = sh.s;
            start = sh.start;
            const int at = sh.stop;
            buf ^= 1;
            if (at >= 0) {
                __syncthreads();
                return at;
            }
        }
    }
    __syncthreads();
    return n;
}

}  // namespace fg
