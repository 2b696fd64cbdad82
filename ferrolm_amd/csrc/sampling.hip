// Sampling on the device (sampler::distribution / draw, src/sampler.rs:52-103)
// and the speculative step's sampling acceptance (Engine::execute,
// src/engine.rs:575-610): min(1, p/q) acceptance, residual resampling from
// max(0, p - q), the bonus draw; each sequence draws from its own generator
// (Rng, src/rng.rs), in the reference's order.
//
// A distribution of top_k 1..kSampleCap is at most kSampleCap (token,
// probability) pairs, stored twice per row: in the reference's order (value
// descending, token ascending; draws scan this order) and in token order (for
// lookups and the residual, which the reference builds in token order). A
// wide one (top_k 0, no limit, or above kSampleCap) keeps up to the whole
// vocabulary in the reference's order plus a dense by-token copy; its kernels
// (k_wide_*, k_draw_wide, k_accept_wide) run after the small ones, each
// kind skipping the other's rows.
#include "seqsum.h"

#include <math.h>

namespace fg {

// f32::total_cmp as unsigned order
__device__ __forceinline__ uint32_t total_key(float x) {
    const uint32_t b = __float_as_uint(x);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// exp rounded to f32 from a double-precision evaluation (within a few double
// ulps): the correctly rounded expf except when exp(x) lies within about
// 1e-9 relative of a rounding boundary
__device__ __forceinline__ float expf_rounded(float x) { return (float)exp((double)x); }

// Rng (src/rng.rs:12-34): xorshift64*, uniform with 53 bits
__device__ __forceinline__ uint64_t rng_next(uint64_t& s) {
    s ^= s >> 12;
    s ^= s << 25;
    s ^= s >> 27;
    return s * 0x2545F4914F6CDD1DULL;
}
__device__ __forceinline__ double rng_uniform(uint64_t& s) {
    return (double)(rng_next(s) >> 11) / 9007199254740992.0;
}

// In-place bitonic sort of n = 1024 64-bit keys in LDS, descending; every
// thread of the 1024-thread workgroup takes part.
__device__ void bitonic_desc(uint64_t* v) {
    const int i = threadIdx.x;
    for (int size = 2; size <= kSampleCap; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            const int j = i ^ stride;
            if (j > i) {
                const bool desc = (i & size) == 0;
                const uint64_t a = v[i], b = v[j];
                if (desc ? a < b : a > b) {
                    v[i] = b;
                    v[j] = a;
                }
            }
            __syncthreads();
        }
}

// One workgroup of kSampleCap threads per logits row: the row's distribution
// (sampler::distribution). Rows of greedy sequences get n = 0.
__global__ __launch_bounds__(kSampleCap) void k_dist(const float* __restrict__ logits, int vocab, int rows_per_seq,
                                                     const SampleParams* __restrict__ prm, uint32_t* __restrict__ tok,
                                                     float* __restrict__ pr, uint32_t* __restrict__ tok_id,
                                                     float* __restrict__ pr_id, int* __restrict__ n_out, int cap) {
    __shared__ uint32_t hist[256];
    __shared__ int sel[2];
    __shared__ int scan[kSampleCap];
    __shared__ uint64_t ck[kSampleCap];
    __shared__ float ev[kSampleCap];
    __shared__ int cgt;
    __shared__ double dsum;
    __shared__ int keep_s;
    __shared__ float ssum;
    const int row = blockIdx.x, tid = threadIdx.x;
    const SampleParams p = prm[row / rows_per_seq];
    if (p.temperature <= 0.0f) {
        if (tid == 0) n_out[row] = 0;
        return;
    }
    if (sample_wide(p)) return;  // k_wide_*
    const float* lg = logits + (size_t)row * vocab;
    const float t = p.temperature > 1e-5f ? p.temperature : 1e-5f;
    const int K = min(p.top_k, vocab);
    // (1) the K-th largest key, eight bits at a time
    uint32_t prefix = 0, mask = 0;
    int need = K;
    for (int shift = 24; shift >= 0; shift -= 8) {
        if (tid < 256) hist[tid] = 0;
        __syncthreads();
        for (int i = tid; i < vocab; i += kSampleCap) {
            const uint32_t key = total_key(lg[i] / t);
            if ((key & mask) == prefix) atomicAdd(&hist[(key >> shift) & 255u], 1u);
        }
        __syncthreads();
        if (tid == 0) {
            int cum = 0, d = 255;
            for (; d > 0; d--) {
                if (cum + (int)hist[d] >= need) break;
                cum += (int)hist[d];
            }
            sel[0] = d;
            sel[1] = cum;
        }
        __syncthreads();
        need -= sel[1];
        prefix |= (uint32_t)sel[0] << shift;
        mask |= 255u << shift;
        __syncthreads();
    }
    const uint32_t kth = prefix;  // need = elements equal to kth that make the top K
    // (2) gather: keys above kth in any order, then the first `need` equal
    // keys by token index (each thread scans a contiguous range; a block scan
    // ranks the ties)
    const int per = (vocab + kSampleCap - 1) / kSampleCap, i0 = tid * per, i1 = min(vocab, i0 + per);
    int ties = 0;
    for (int i = i0; i < i1; i++) ties += total_key(lg[i] / t) == kth;
    scan[tid] = ties;
    if (tid == 0) cgt = 0;
    ck[tid] = 0;
    __syncthreads();
    for (int off = 1; off < kSampleCap; off <<= 1) {
        const int v = tid >= off ? scan[tid - off] : 0;
        __syncthreads();
        scan[tid] += v;
        __syncthreads();
    }
    int rank = scan[tid] - ties;
    for (int i = i0; i < i1; i++) {
        const uint32_t key = total_key(lg[i] / t);
        // composite: value descending, then token ascending
        const uint64_t c = ((uint64_t)key << 32) | (uint32_t)~(uint32_t)i;
        if (key > kth) {
            ck[atomicAdd(&cgt, 1)] = c;
        } else if (key == kth) {
            if (rank < need) ck[K - need + rank] = c;
            rank++;
        }
    }
    __syncthreads();
    // (3) the reference's order
    bitonic_desc(ck);
    // (4) exp(v - max) in f32, their f64 sum in order, probabilities
    const float mx = key_value((uint32_t)(ck[0] >> 32));
    if (tid < K) ev[tid] = expf_rounded(key_value((uint32_t)(ck[tid] >> 32)) - mx);
    __syncthreads();
    if (tid == 0) {
        double s = 0.0;
        for (int i = 0; i < K; i++) s += (double)ev[i];
        dsum = s;
    }
    __syncthreads();
    float pv = tid < K ? (float)((double)ev[tid] / dsum) : 0.0f;
    int n = K;
    if (p.top_p < 1.0f) {
        __syncthreads();
        if (tid < K) ev[tid] = pv;
        __syncthreads();
        if (tid == 0) {
            float acc = 0.0f;
            int keep = K;
            for (int i = 0; i < K; i++) {
                acc += ev[i];
                if (acc >= p.top_p) {
                    keep = i + 1;
                    break;
                }
            }
            float s2 = 0.0f;
            for (int i = 0; i < keep; i++) s2 += ev[i];
            keep_s = keep;
            ssum = s2;
        }
        __syncthreads();
        n = keep_s;
        pv = pv / ssum;
    }
    const size_t base = (size_t)row * cap;
    const uint32_t tk = ~(uint32_t)ck[tid];
    if (tid < n) {
        tok[base + tid] = tk;
        pr[base + tid] = pv;
    }
    if (tid == 0) n_out[row] = n;
    // (5) the same pairs in token order
    __syncthreads();
    ck[tid] = tid < n ? ((uint64_t)(0xFFFFFFFFu - tk) << 32) | __float_as_uint(pv) : 0;
    __syncthreads();
    bitonic_desc(ck);
    if (tid < n) {
        tok_id[base + tid] = 0xFFFFFFFFu - (uint32_t)(ck[tid] >> 32);
        pr_id[base + tid] = __uint_as_float((uint32_t)ck[tid]);
    }
}

// sampler::draw over n pairs (src/sampler.rs:93-103)
__device__ uint32_t draw_pairs(const uint32_t* tok, const float* pr, int n, uint64_t& rng) {
    float s = 0.0f;
    for (int i = 0; i < n; i++) s += pr[i];
    float u = (float)rng_uniform(rng) * s;
    for (int i = 0; i < n; i++) {
        if (u < pr[i]) return tok[i];
        u -= pr[i];
    }
    return n > 0 ? tok[n - 1] : 0;
}

// probability of token t in a row's token-ordered pairs (0 if absent)
__device__ float lookup(const uint32_t* tok_id, const float* pr_id, int n, uint32_t t) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (tok_id[mid] < t)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo < n && tok_id[lo] == t ? pr_id[lo] : 0.0f;
}

// One thread per row: sampler::sample of each sampled row's distribution
// into out[row * out_stride + out_off]; greedy rows keep what the argmax
// wrote there.
__global__ void k_draw(int rows, const SampleParams* __restrict__ prm, const uint32_t* __restrict__ tok,
                       const float* __restrict__ pr, const int* __restrict__ n, uint64_t* __restrict__ rng,
                       uint32_t* __restrict__ out, int out_stride, int out_off, int cap) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= rows || prm[r].temperature <= 0.0f || sample_wide(prm[r])) return;
    uint64_t s = rng[r];
    out[(size_t)r * out_stride + out_off] = draw_pairs(tok + (size_t)r * cap, pr + (size_t)r * cap, n[r], s);
    rng[r] = s;
}

// One thread per sequence: Engine::execute's verify of proposals d1..dk
// (vtok[s*(k+1) + 1 + j]) against target rows s*(k+1) + j, for sampled
// sequences (src/engine.rs:575-610) and greedy ones (:570-574, with the
// argmax of each verify row in am).
__global__ void k_accept_sampled(int n_seqs, int k, const SampleParams* __restrict__ prm,
                                 const uint32_t* __restrict__ vtok, const uint32_t* __restrict__ am,
                                 const uint32_t* __restrict__ p_tok, const float* __restrict__ p_pr,
                                 const uint32_t* __restrict__ p_tok_id, const float* __restrict__ p_pr_id,
                                 const int* __restrict__ p_n, const uint32_t* __restrict__ q_tok_id,
                                 const float* __restrict__ q_pr_id, const int* __restrict__ q_n,
                                 uint64_t* __restrict__ rng, uint32_t* __restrict__ out_tokens,
                                 int32_t* __restrict__ out_count, int32_t* __restrict__ out_accepted, int cap) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n_seqs || sample_wide(prm[s])) return;  // k_accept_wide
    const int K1 = k + 1;
    const bool greedy = prm[s].temperature <= 0.0f;
    uint64_t st = rng[s];
    int ne = 0, accepted = 0;
    uint32_t* out = out_tokens + (size_t)s * K1;
    for (int j = 0; j < k; j++) {
        const int row = s * K1 + j;
        const uint32_t d = vtok[(size_t)s * K1 + 1 + j];
        bool take_d;
        uint32_t t = 0;
        if (greedy) {
            t = am[row];
            take_d = t == d;
        } else {
            const size_t pb = (size_t)row * cap, qb = ((size_t)j * n_seqs + s) * cap;
            const int pn = p_n[row], qn = q_n[j * n_seqs + s];
            const float px = lookup(p_tok_id + pb, p_pr_id + pb, pn, d);
            const float qx = lookup(q_tok_id + qb, q_pr_id + qb, qn, d);
            take_d = qx > 0.0f && rng_uniform(st) < (double)fminf(px / qx, 1.0f);
            if (!take_d) {
                // the part of p that q under-covers, in token order
                float rs = 0.0f;
                int rc = 0;
                for (int i = 0; i < pn; i++) {
                    const float a = p_pr_id[pb + i], b = lookup(q_tok_id + qb, q_pr_id + qb, qn, p_tok_id[pb + i]);
                    if (a > b) {
                        rs += a - b;
                        rc++;
                    }
                }
                if (rc > 0) {
                    float u = (float)rng_uniform(st) * rs;
                    bool done = false;
                    for (int i = 0; i < pn && !done; i++) {
                        const float a = p_pr_id[pb + i], b = lookup(q_tok_id + qb, q_pr_id + qb, qn, p_tok_id[pb + i]);
                        if (a > b) {
                            t = p_tok_id[pb + i];  // the last residual token if u never falls below
                            if (u < a - b)
                                done = true;
                            else
                                u -= a - b;
                        }
                    }
                } else {
                    // dense_pairs(p): its positive entries in token order
                    float ps = 0.0f;
                    for (int i = 0; i < pn; i++)
                        if (p_pr_id[pb + i] > 0.0f) ps += p_pr_id[pb + i];
                    float u = (float)rng_uniform(st) * ps;
                    bool done = false;
                    for (int i = 0; i < pn && !done; i++) {
                        const float a = p_pr_id[pb + i];
                        if (a > 0.0f) {
                            t = p_tok_id[pb + i];
                            if (u < a)
                                done = true;
                            else
                                u -= a;
                        }
                    }
                }
            }
        }
        if (take_d) {
            out[ne++] = d;
            accepted++;
        } else {
            out[ne++] = t;
            break;
        }
    }
    if (accepted == k) {
        const int row = s * K1 + k;
        if (greedy) {
            out[ne++] = am[row];
        } else {
            const size_t pb = (size_t)row * cap;
            out[ne++] = draw_pairs(p_tok + pb, p_pr + pb, p_n[row], st);
        }
    }
    out_count[s] = ne;
    out_accepted[s] = accepted;
    rng[s] = st;
}

// ---------------------------------------------------------------------------
// Wide distributions: top_k = 0 (no limit) or above kSampleCap. A row holds up
// to `cap` (the vocabulary) pairs, in the reference's order, plus a dense
// token-indexed copy of the probabilities (0 where a token is not kept) for
// the acceptance's lookups and residual. The work over the vocabulary runs on
// one workgroup per 1024 tokens and row: the keys, a stable LSD radix sort
// (four 8-bit passes), the exponentials and the final probabilities. The
// reference's sums and walks are sequential (f64 softmax sum, f32 top-p
// prefix, f32 draw sums); one workgroup per row or sequence runs them with
// seq_scan, which has the sequential loop's bits.
// Bound: the latency of eight dependent launches. 49,152 tokens, 4 rows: 2664
// us for the whole distribution on one workgroup a row (its tiles of the sort
// one after the other, its sums one lane each), 8008 us for the acceptance;
// now 140 us (sort 4 x 14, sums 71) and 200 us.
// ---------------------------------------------------------------------------
constexpr int kWideTile = 1024;  // tokens per workgroup

// A wide row's scratch: keys and tokens (two of each, the sort's ping-pong), the four passes'
// digit counts [pass][tile][256], and the softmax sum, the top-p sum and whether it applies.
struct WideRow {
    uint32_t *k0, *v0, *k1, *v1, *hist;
    double* dsum;
    float* s2;
    int* cut;
};
__device__ __forceinline__ WideRow wide_row(const SampleRows& d, int row) {
    uint32_t* p = d.scratch + (size_t)row * wide_scratch_words(d.cap);
    WideRow w;
    w.k0 = p;
    w.v0 = p + d.cap;
    w.k1 = p + 2 * (size_t)d.cap;
    w.v1 = p + 3 * (size_t)d.cap;
    w.hist = p + 4 * (size_t)d.cap;
    uint32_t* t = p + wide_scratch_words(d.cap) - 64;
    w.dsum = (double*)t;
    w.s2 = (float*)(t + 2);
    w.cut = (int*)(t + 3);
    return w;
}

// The complemented keys of a tile (ascending: value descending), its tokens, the first pass's
// digit counts; the later passes' counts and the dense copy cleared.
__global__ __launch_bounds__(kWideTile) void k_wide_keys(const float* __restrict__ logits, int vocab, int rows_per_seq,
                                                         const SampleParams* __restrict__ prm, SampleRows d) {
    __shared__ uint32_t hist[256];
    const int row = blockIdx.y, tid = threadIdx.x, i = blockIdx.x * kWideTile + tid, tiles = gridDim.x;
    const SampleParams p = prm[row / rows_per_seq];
    if (!sample_wide(p)) return;  // greedy rows and small top_k rows: k_dist
    const WideRow w = wide_row(d, row);
    const float t = p.temperature > 1e-5f ? p.temperature : 1e-5f;
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    if (i < vocab) {
        const uint32_t key = ~total_key(logits[(size_t)row * vocab + i] / t);
        w.k0[i] = key;
        w.v0[i] = (uint32_t)i;
        d.dense[(size_t)row * d.cap + i] = 0.0f;
        atomicAdd(&hist[key & 255u], 1u);
    }
    __syncthreads();
    if (tid < 256) {
        w.hist[(size_t)blockIdx.x * 256 + tid] = hist[tid];
#pragma unroll
        for (int pass = 1; pass < 4; pass++) w.hist[((size_t)pass * tiles + blockIdx.x) * 256 + tid] = 0;
    }
}

// One 8-bit pass of the stable LSD radix sort, one workgroup per tile of 1024: a digit's place is
// the count of smaller digits, plus its count in earlier tiles, plus its rank in the tile (wave
// ballots keep element order). The elements are counted for the next pass where they land.
__global__ __launch_bounds__(kWideTile) void k_wide_sort(int vocab, int pass, int rows_per_seq,
                                                         const SampleParams* __restrict__ prm, SampleRows d) {
    __shared__ uint32_t tot[4][256], bel[4][256], wsum[4];
    __shared__ uint32_t wcnt[kWideTile / 64][256];
    const int row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, tiles = gridDim.x;
    if (!sample_wide(prm[row / rows_per_seq])) return;
    const WideRow w = wide_row(d, row);
    const uint32_t *ki = pass & 1 ? w.k1 : w.k0, *vi = pass & 1 ? w.v1 : w.v0;
    uint32_t *ko = pass & 1 ? w.k0 : w.k1, *vo = pass & 1 ? w.v0 : w.v1;
    const uint32_t* hist = w.hist + (size_t)pass * tiles * 256;
    const int i = blockIdx.x * kWideTile + tid, shift = 8 * pass;
    const bool valid = i < vocab;
    const uint32_t key = valid ? ki[i] : 0u, val = valid ? vi[i] : 0u;
#pragma unroll
    for (int z = 0; z < 4; z++) (&wcnt[0][0])[z * kWideTile + tid] = 0;
    {
        // each quarter of the workgroup sums a quarter of the tiles' counts
        const int dg = tid & 255, part = tid >> 8;
        uint32_t all = 0, below = 0;
#pragma unroll 8
        for (int t = part; t < tiles; t += 4) {
            const uint32_t c = hist[(size_t)t * 256 + dg];
            all += c;
            below += t < (int)blockIdx.x ? c : 0u;
        }
        tot[part][dg] = all;
        bel[part][dg] = below;
    }
    __syncthreads();
    uint32_t excl = 0, mine = 0;
    if (tid < 256) {
        mine = tot[0][tid] + tot[1][tid] + tot[2][tid] + tot[3][tid];
        uint32_t inc = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = __shfl_up(inc, o, 64);
            if (lane >= o) inc += v;
        }
        if (lane == 63) wsum[wave] = inc;
        excl = inc - mine;
    }
    // this tile's ranks meanwhile
    const uint32_t dgt = (key >> shift) & 255u;
    uint64_t same = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
        const uint64_t bb = __ballot((dgt >> b) & 1u);
        same &= ((dgt >> b) & 1u) ? bb : ~bb;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1));
    if (valid && rank == 0) wcnt[wave][dgt] = __popcll(same);
    __syncthreads();
    if (tid < 256) {
        uint32_t run = excl + bel[0][tid] + bel[1][tid] + bel[2][tid] + bel[3][tid];
        for (int v = 0; v < wave; v++) run += wsum[v];
#pragma unroll
        for (int v = 0; v < kWideTile / 64; v++) {
            const uint32_t c = wcnt[v][tid];
            wcnt[v][tid] = run;
            run += c;
        }
    }
    __syncthreads();
    if (valid) {
        const uint32_t dst = wcnt[wave][dgt] + rank;
        ko[dst] = key;
        vo[dst] = val;
        if (pass < 3)
            atomicAdd(&w.hist[((size_t)(pass + 1) * tiles + dst / kWideTile) * 256 + ((key >> (shift + 8)) & 255u)], 1u);
    }
}

// exp(v - max) of the sorted row's first K values
__global__ __launch_bounds__(kWideTile) void k_wide_exp(int vocab, int rows_per_seq,
                                                        const SampleParams* __restrict__ prm, SampleRows d) {
    const int row = blockIdx.y, i = blockIdx.x * kWideTile + threadIdx.x;
    const SampleParams p = prm[row / rows_per_seq];
    if (!sample_wide(p)) return;
    const WideRow w = wide_row(d, row);
    const int K = p.top_k == 0 ? vocab : min(p.top_k, vocab);
    if (i < K) d.pr[(size_t)row * d.cap + i] = expf_rounded(key_value(~w.k0[i]) - key_value(~w.k0[0]));
}

// The f64 sum of a row's exponentials and its top-p prefix. The reference then sums the kept
// probabilities again from the start: the prefix's own sum.
__global__ __launch_bounds__(1024) void k_wide_sums(int vocab, int rows_per_seq, const SampleParams* __restrict__ prm,
                                                    SampleRows d) {
    __shared__ SeqShared<double> sd;
    __shared__ SeqShared<float> sf;
    const int row = blockIdx.x;
    const SampleParams p = prm[row / rows_per_seq];
    if (!sample_wide(p)) return;
    const WideRow w = wide_row(d, row);
    const int K = p.top_k == 0 ? vocab : min(p.top_k, vocab);
    const float* e = d.pr + (size_t)row * d.cap;
    double sum = 0.0;
    seq_scan<SEQ_SUM, 8, double>(K, sum, 0.0, [&](int i) { return e[i]; }, sd);
    int n = K;
    float acc = 0.0f;
    const bool cut = p.top_p < 1.0f;
    if (cut) {
        auto prob = [&](int i) { return (float)((double)e[i] / sum); };
        if (p.top_p > 0.0f) {
            const int at = seq_scan<SEQ_REACH, 4, float>(K, acc, p.top_p, prob, sf);
            n = at < K ? at + 1 : K;
        } else {
            acc = prob(0);
            if (acc >= p.top_p) n = 1;  // (a NaN reaches no limit, and stays one)
        }
    }
    if (threadIdx.x == 0) {
        *w.dsum = sum;
        *w.s2 = acc;
        *w.cut = cut;
        d.n[row] = n;
    }
}

// The kept pairs in the reference's order and the dense copy
__global__ __launch_bounds__(kWideTile) void k_wide_pairs(int rows_per_seq, const SampleParams* __restrict__ prm,
                                                          SampleRows d) {
    const int row = blockIdx.y, i = blockIdx.x * kWideTile + threadIdx.x;
    if (!sample_wide(prm[row / rows_per_seq]) || i >= d.n[row]) return;
    const WideRow w = wide_row(d, row);
    const size_t at = (size_t)row * d.cap;
    float v = (float)((double)d.pr[at + i] / *w.dsum);
    if (*w.cut) v = v / *w.s2;
    const uint32_t t = w.v0[i];
    d.pr[at + i] = v;
    d.tok[at + i] = t;
    d.dense[at + t] = v;
}

// sampler::draw over a wide row's n pairs, on the workgroup; every thread ends with the token
// and the advanced generator.
__device__ uint32_t draw_wide(const uint32_t* tok, const float* pr, int n, uint64_t& rng, SeqShared<float>& sh) {
    auto value = [&](int i) { return pr[i]; };
    float s = 0.0f;
    seq_scan<SEQ_SUM, 4, float>(n, s, 0.0f, value, sh);
    float u = (float)rng_uniform(rng) * s;
    const int at = seq_scan<SEQ_WALK, 4, float>(n, u, 0.0f, value, sh);
    return n > 0 ? tok[min(at, n - 1)] : 0;
}

// One workgroup per row: sampler::sample of each wide sampled row into
// out[row * out_stride + out_off].
__global__ __launch_bounds__(1024) void k_draw_wide(int rows, const SampleParams* __restrict__ prm, SampleRows d,
                                                    uint64_t* __restrict__ rng, uint32_t* __restrict__ out,
                                                    int out_stride, int out_off) {
    __shared__ SeqShared<float> sh;
    const int r = blockIdx.x;
    const SampleParams p = prm[r];
    if (!sample_wide(p)) return;
    uint64_t s = rng[r];
    const size_t base = (size_t)r * d.cap;
    const uint32_t t = draw_wide(d.tok + base, d.pr + base, d.n[r], s, sh);
    if (threadIdx.x == 0) {
        out[(size_t)r * out_stride + out_off] = t;
        rng[r] = s;
    }
}

// One workgroup per sequence: k_accept_sampled's rule for sequences whose
// distributions are wide (dense lookups; the residual max(0, p - q) and the
// dense pairs of p in token order over the whole vocabulary). Every thread
// follows the same generator.
__global__ __launch_bounds__(1024) void k_accept_wide(int n_seqs, int k, int vocab, const SampleParams* __restrict__ prm,
                                                      const uint32_t* __restrict__ vtok,
                                                      const uint32_t* __restrict__ am, SampleRows p, SampleRows q,
                                                      uint64_t* __restrict__ rng, uint32_t* __restrict__ out_tokens,
                                                      int32_t* __restrict__ out_count,
                                                      int32_t* __restrict__ out_accepted) {
    __shared__ SeqShared<float> sh;
    const int sq = blockIdx.x;
    const SampleParams pp = prm[sq];
    if (!sample_wide(pp)) return;
    const int K1 = k + 1;
    uint64_t st = rng[sq];
    int ne = 0, accepted = 0;
    uint32_t* out = out_tokens + (size_t)sq * K1;
    // a draw from the terms in token order: u walks them down; the token whose term exceeds what
    // is left of u, or the last token with a positive term (0 when there is none)
    auto draw = [&](auto term) -> uint32_t {
        float s = 0.0f;
        seq_scan<SEQ_SUM, 4, float>(vocab, s, 0.0f, term, sh);
        float u = (float)rng_uniform(st) * s;
        const int at = seq_scan<SEQ_WALK, 4, float>(vocab, u, 0.0f, term, sh);
        if (at < vocab) return (uint32_t)at;
        __syncthreads();
        if (threadIdx.x == 0) sh.start = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < vocab; i += blockDim.x)
            if (term(i) > 0.0f) atomicMax(&sh.start, i);
        __syncthreads();
        return (uint32_t)sh.start;
    };
    for (int j = 0; j < k; j++) {
        const int row = sq * K1 + j;
        const uint32_t dtok = vtok[(size_t)sq * K1 + 1 + j];
        const float* pd = p.dense + (size_t)row * p.cap;
        const float* qd = q.dense + ((size_t)j * n_seqs + sq) * q.cap;
        const float px = pd[dtok], qx = qd[dtok];
        if (qx > 0.0f && rng_uniform(st) < (double)fminf(px / qx, 1.0f)) {
            if (threadIdx.x == 0) out[ne] = dtok;
            ne++;
            accepted++;
            continue;
        }
        // the part of p that q under-covers, in token order, where there is one
        int any = 0;
        for (int i = threadIdx.x; i < vocab; i += blockDim.x) any |= pd[i] > qd[i];
        any = __syncthreads_or(any);
        uint32_t t;
        if (any)
            t = draw([&](int i) { return pd[i] > qd[i] ? pd[i] - qd[i] : 0.0f; });
        else
            t = draw([&](int i) { return pd[i] > 0.0f ? pd[i] : 0.0f; });  // p's positive entries
        if (threadIdx.x == 0) out[ne] = t;
        ne++;
        break;
    }
    if (accepted == k) {
        const int row = sq * K1 + k;
        const size_t pb = (size_t)row * p.cap;
        const uint32_t t = draw_wide(p.tok + pb, p.pr + pb, p.n[row], st, sh);
        if (threadIdx.x == 0) out[ne] = t;
        ne++;
    }
    if (threadIdx.x == 0) {
        out_count[sq] = ne;
        out_accepted[sq] = accepted;
        rng[sq] = st;
    }
}

void launch_dist(hipStream_t st, const float* logits, int rows, int vocab, int rows_per_seq, const SampleParams* prm,
                 SampleRows& out) {
    if (rows <= 0) return;
    hipLaunchKernelGGL(k_dist, dim3(rows), dim3(kSampleCap), 0, st, logits, vocab, rows_per_seq, prm, out.tok, out.pr,
                       out.tok_id, out.pr_id, out.n, out.cap);
    if (!out.dense) return;
    const dim3 grid((vocab + kWideTile - 1) / kWideTile, rows), block(kWideTile);
    hipLaunchKernelGGL(k_wide_keys, grid, block, 0, st, logits, vocab, rows_per_seq, prm, out);
    for (int pass = 0; pass < 4; pass++)
        hipLaunchKernelGGL(k_wide_sort, grid, block, 0, st, vocab, pass, rows_per_seq, prm, out);
    hipLaunchKernelGGL(k_wide_exp, grid, block, 0, st, vocab, rows_per_seq, prm, out);
    hipLaunchKernelGGL(k_wide_sums, dim3(rows), dim3(1024), 0, st, vocab, rows_per_seq, prm, out);
    hipLaunchKernelGGL(k_wide_pairs, grid, block, 0, st, rows_per_seq, prm, out);
}

void launch_draw(hipStream_t st, int rows, const SampleParams* prm, const SampleRows& d, uint64_t* rng, uint32_t* out,
                 int out_stride, int out_off) {
    if (rows <= 0) return;
    hipLaunchKernelGGL(k_draw, dim3((rows + 63) / 64), dim3(64), 0, st, rows, prm, d.tok, d.pr, d.n, rng, out,
                       out_stride, out_off, d.cap);
    if (d.dense) hipLaunchKernelGGL(k_draw_wide, dim3(rows), dim3(1024), 0, st, rows, prm, d, rng, out, out_stride,
                                    out_off);
}

void launch_accept_sampled(hipStream_t st, int n_seqs, int k, const SampleParams* prm, const uint32_t* vtok,
                           const uint32_t* am, const SampleRows& p, const SampleRows& q, uint64_t* rng,
                           uint32_t* out_tokens, int32_t* out_count, int32_t* out_accepted) {
    hipLaunchKernelGGL(k_accept_sampled, dim3((n_seqs + 63) / 64), dim3(64), 0, st, n_seqs, k, prm, vtok, am, p.tok,
                       p.pr, p.tok_id, p.pr_id, p.n, q.tok_id, q.pr_id, q.n, rng, out_tokens, out_count,
                       out_accepted, p.cap);
    if (p.dense)
        hipLaunchKernelGGL(k_accept_wide, dim3(n_seqs), dim3(1024), 0, st, n_seqs, k, p.vocab, prm, vtok, am, p, q, rng,
                           out_tokens, out_count, out_accepted);
}

}  // namespace fg
