// Which products run on the tiled GEMM (gemm_tiles.h), and on which tile.
#include "internal.h"

#include <algorithm>

namespace fg {

template <int KIND>
void run_mm(hipStream_t st, int epi, int cfg, const GemvArgs& a, hipEvent_t e0, hipEvent_t e1);
extern template void run_mm<BF16>(hipStream_t, int, int, const GemvArgs&, hipEvent_t, hipEvent_t);
extern template void run_mm<INT8>(hipStream_t, int, int, const GemvArgs&, hipEvent_t, hipEvent_t);
extern template void run_mm<INT4>(hipStream_t, int, int, const GemvArgs&, hipEvent_t, hipEvent_t);

// The tile shapes (run_mm_epi's cases): row tiles, 64-column waves, K shares; the time of a stage in
// us on a full chip, for a CU's only workgroup and (four waves: two of them fit a CU) for two, by
// which a product's shape is chosen.
// Fitted to 137 products of 48 to 1024 rows (int4, int8 and bf16, 576 to 49152 outputs, 576 to 14336
// inputs): the shape with the least modelled time was within 6% of the best measured one on all but
// seven, and within 12% on those that were measured.
static const struct {
    int rt, nwn, nwk;
    float one, two;
} kTiles[] = {
    {8, 4, 1, 2.2f, 3.9f},  {5, 4, 1, 1.8f, 2.75f}, {8, 4, 2, 3.9f, 0.0f},  {5, 2, 2, 2.0f, 2.75f}, {4, 2, 2, 1.75f, 2.35f},
    {5, 2, 4, 3.1f, 0.0f},  {4, 2, 4, 2.65f, 0.0f}, {3, 2, 4, 2.25f, 0.0f}, {2, 2, 4, 1.85f, 0.0f},
};

// What a lone product costs on the tiles and on k_gemm, in us, beyond what both pay (the packing of its
// inputs, the launches): per weight kind, a stage of each tile shape (kTiles' order) for a CU's only
// workgroup and for two of four waves, and k_gemm's time for a k-block pair of each wave by row tiles
// (2: one, two and three workgroups on a CU, 3: one and two, 4, 5, and 5 of 128 columns). A least
// squares fit to 3500 products of 33 to 1024 rows, each run on k_gemm and on all nine shapes (37 sizes,
// 576 to 49152 outputs, 576 to 14336 inputs); predicted over measured was 0.93 to 1.08 for nine in ten
// on the tiles and 0.88 to 1.12 on k_gemm. With store_on_gemm none of them is over 3% slower than on
// k_gemm; by tile counts alone 138 were, up to 1.22 times (bf16 4096 x 4096 at 320 rows: 33.9 against
// 39.8 us, int4 5120 x 960 at 224: 15.6 against 18.8).
struct Costs {
    float one[9], two[9];   // k_mm, a stage
    float two_rt[3], three_rt[2], four_rt, five_rt, five_rt128;  // k_gemm, a pair of k-blocks
    float round, alone;     // a round of tiles; a round of k_gemm's with one workgroup on a CU
    float out, split, split_out;  // per million outputs; k_gemm's split of K, and per million partial sums
    float weights, spread;  // k_gemm, per MB of weights; again for each of up to 8 XCDs that read them
    float gain;             // the tiles are taken where their time is below gain times k_gemm's
};
static const Costs kCosts[] = {
    // BF16
    {{1.32f, 0.92f, 2.58f, 1.07f, 0.88f, 2.0f, 1.66f, 1.35f, 0.96f},
     {2.15f, 1.44f, 0, 1.7f, 1.43f},
     {0.94f, 1.94f, 2.65f}, {1.08f, 3.92f}, 1.76f, 2.21f, 1.94f,
     0.31f, 1.05f, 2.9f, 3.54f, 2.76f, 0.033f, 0.036f, 0.96f},
    // INT8
    {{1.97f, 1.28f, 2.83f, 1.4f, 1.07f, 2.2f, 1.82f, 1.52f, 1.16f},
     {2.68f, 1.82f, 0, 2.03f, 1.68f},
     {1.54f, 3.09f, 4.4f}, {1.85f, 5.07f}, 2.55f, 3.01f, 2.59f,
     1.68f, 1.33f, 2.95f, 4.02f, 2.65f, 0.002f, 0.043f, 0.98f},
    // INT4
    {{1.79f, 1.34f, 2.95f, 1.49f, 1.23f, 2.33f, 1.96f, 1.66f, 1.29f},
     {2.65f, 1.96f, 0, 2.15f, 1.82f},
     {1.48f, 2.89f, 4.07f}, {1.74f, 4.54f}, 2.39f, 2.89f, 2.57f,
     1.31f, 1.05f, 2.77f, 4.17f, 2.21f, 0.0f, 0.061f, 0.98f},
};

// workgroups of a tile shape and its stages
static int tile_count(int tile, int N, int rt) {
    const auto& c = kTiles[tile];
    return ((rt + c.rt - 1) / c.rt) * ((N + 64 * c.nwn - 1) / (64 * c.nwn));
}
static float tile_stages(int tile, int KB) { return (float)((KB / 2 + kTiles[tile].nwk - 1) / kTiles[tile].nwk); }
// the time of n workgroups of t stages (one, two: a stage's) and `round` for each round of them
static float tile_time(int tile, int n, float stages, float one, float two, float round) {
    if (kTiles[tile].nwn * kTiles[tile].nwk == 8) return (float)((n + 255) / 256) * (round + stages * one);
    const int rest = n % 512;
    float t = (float)(n / 512) * (round + stages * two);
    if (rest) t += round + stages * (rest > 256 ? two : one);
    return t;
}

static float gemm_time(const Costs& c, const GemmShape& g, int kind, int N, int KB, int m) {
    const int cg = (N + 64 * g.cs - 1) / (64 * g.cs), per_cu = (cg * g.groups * g.ks + 255) / 256;
    const float pairs = (float)(KB / 2) / (float)(g.ks * (8 / g.cs));
    const int most = g.rtw == 2 ? 3 : g.rtw == 3 ? 2 : 1;  // workgroups that fit a CU
    auto round = [&](int r) {
        const float pair = g.rtw == 2   ? c.two_rt[r - 1]
                           : g.rtw == 3 ? c.three_rt[r - 1]
                           : g.rtw == 4 ? c.four_rt
                           : g.cs == 2  ? c.five_rt128
                                        : c.five_rt;
        return pairs * pair + (r == 1 ? c.alone : 0.0f);
    };
    float t = (float)(per_cu / most) * round(most);
    if (per_cu % most) t += round(per_cu % most);
    const float mout = (float)m * (float)N * 1e-6f;
    t += g.ks > 1 ? c.split + c.split_out * mout * (float)g.ks : c.out * mout;
    const float mb = (float)N * (float)KB * 32e-6f * (kind == BF16 ? 2.0f : kind == INT8 ? 1.125f : 0.625f);
    return t + mb * (c.weights + (cg % 8 ? c.spread * (float)std::min(g.groups, 8) : 0.0f));
}

void mm_tile_size(int tile, int* row_tiles, int* col_waves, int* k_shares) {
    *row_tiles = kTiles[tile].rt;
    *col_waves = kTiles[tile].nwn;
    *k_shares = kTiles[tile].nwk;
}

// Whether k_gemm is the faster for a forward's product with its epilogue: 3171 products of two-layer
// models (33 to 4096 rows, eleven models of 576 to 4096 wide, all kinds), each on k_gemm and on the tiles.
// q/k/v and gate/up (1629 of them) gain wherever the tiles are enough: 0.84, 0.80 and 0.82 of k_gemm's time
// in the mean for q/k/v (bf16, int8, int4), 0.69, 0.69 and 0.71 for gate/up, none over 4% slower. Of o and
// down, 47 were over 5% slower, up to 1.33 times; what they are is below, and with it one is, by 5.2%.
static bool resid_on_gemm(int kind, int tile, int n, const GemmShape& g, int N) {
    // k_gemm's tiles of four or five row tiles, one full round of the chip without a split (4096 x 14336 at 256
    // to 320 rows: 1.28 to 1.33 times as long on the tiles in bf16, 1.17 to 1.25 in int4, 1.11 in int8)
    const int wgs = (N + 64 * g.cs - 1) / (64 * g.cs) * g.groups;
    if (g.rtw >= 4 && g.ks == 1 && wgs > 192 && wgs <= 256) return true;
    if (kind != BF16) return false;
    // bf16, whose weights take twice the loads and no conversion to hide them: two-row tiles (2048 x 8192 at
    // 320 to 512 rows 1.25 to 1.31 times, 1536 wide even, narrower ones down to 0.71), three-row tiles in
    // more than one round (2560 x 6912 at 1024 rows 1.25, 3072 x 8192 at 832 1.22, 4096 x 14336 at 704
    // even), and four waves just past a round (2560 x 2560 at 1024 rows 1.08)
    const auto& c = kTiles[tile];
    if (c.rt == 2) return N >= 1536;
    if (c.rt == 3) return n > 256;
    return c.nwn * c.nwk == 4 && n > 256 && n <= 320;
}

// Whether k_gemm is the faster for a lone product.
static bool store_on_gemm(int kind, int tile, int n, const GemmShape& g, int N, int KB, int m, int rt) {
    const int cg = (N + 64 * g.cs - 1) / (64 * g.cs), wgs = cg * g.groups;
    // Up to 64 rows only the widest products come here, and all of them gain (49152 x 576 at 33 rows, int8:
    // 23.5 against 18.8 us).
    if (rt < 5) return false;
    // Past 1024 rows (211 products up to 32768, each on both) activations no longer stay in the L2s, which
    // the model does not know, and the tiles win, but for bf16 on k_gemm's two-row tiles up to 4096 rows
    // (960 x 576 at 2048: 22.2 against 26.4 us; at 16384 114.5 against 94.7). Seven of the bf16 products
    // are over 3% slower on the tiles, up to 1.10 times, none of int8 and four of int4, up to 1.07.
    if (rt > 64) return kind == BF16 && g.rtw == 2 && m <= 4096 && (KB <= 32 || (KB <= 64 && cg % 8 == 0));
    // Where k_gemm does better than its model: its two-row tiles, three workgroups on a CU, on short K
    // (3072 x 576 at 832 rows, int4: 23.9 against 27.1), for bf16 up to 2048 inputs when an XCD keeps its
    // column groups (3072 x 2048 at 832 rows: 36.0 against 43.0); and for bf16 one full round of its
    // largest tiles without a split (16384 x 2048 at 160 rows: 32.8 against 36.6).
    if (g.rtw == 2 && (KB < 32 || (kind == BF16 && KB <= 64 && cg % 8 == 0))) return true;
    if (kind == BF16 && g.rtw >= 4 && g.ks == 1 && wgs > 192 && wgs <= 256) return true;
    const Costs& c = kCosts[kind == BF16 ? 0 : kind == INT8 ? 1 : 2];
    const float tiles = tile_time(tile, n, tile_stages(tile, KB), c.one[tile], c.two[tile], c.round) +
                        c.out * (float)m * (float)N * 1e-6f;
    return tiles >= c.gain * gemm_time(c, g, kind, N, KB, m);
}

int mm_tile(int epi, int kind, int N, int KB, int m, int p_total, size_t kpart_cap) {
    const int rt = (p_total + 3) / 4;
    if (rt < 3) return -1;
    int tile = -1;
    float best = 0.0f;
    for (int i = 0; i < (int)(sizeof(kTiles) / sizeof(kTiles[0])); i++) {
        const float start = 5.0f;  // first loads, epilogue
        const float t = tile_time(i, tile_count(i, N, rt), tile_stages(i, KB), kTiles[i].one, kTiles[i].two, start);
        if (tile < 0 || t < best) {
            tile = i;
            best = t;
        }
    }
    // k_gemm splits K finer and wins where the tiles leave CUs idle. Its time, then the tiles', in us:
    // 2048 x 8192 at 256 rows (128 tiles) 42 against 59, at 320 (160) 69 against 61; 6144 x 2048 at 160
    // (240 of two row tiles) even, 22.4 against 21.9, at 192 (192 of three) 32.2 against 25.3; and on
    // short K with two row tiles 960 x 576 at 1024 rows 14.5 against 16.2.
    const int n = tile_count(tile, N, rt);
    if (kTiles[tile].rt == 2 ? n < 150 || m < 256 || KB < 32 : n < 180) return -1;
    if (epi != EPI_RESID && epi != EPI_STORE) return tile;
    const GemmShape g = gemm_shape(N / 16, KB, N, m, p_total, kpart_cap);
    const bool other = epi == EPI_RESID ? resid_on_gemm(kind, tile, n, g, N)
                                        : store_on_gemm(kind, tile, n, g, N, KB, m, rt);
    return other ? -1 : tile;
}

int launch_mm(hipStream_t st, int epi, const DMat& w, const GemvArgs& a, hipEvent_t e0, hipEvent_t e1) {
    const int tile = mm_tile(epi, w.kind, a.N, a.KB, a.m, a.p_total, a.kpart ? a.kpart_cap : 0);
    if (tile < 0) return 0;
    if (w.kind == INT4)
        run_mm<INT4>(st, epi, tile, a, e0, e1);
    else if (w.kind == INT8)
        run_mm<INT8>(st, epi, tile, a, e0, e1);
    else
        run_mm<BF16>(st, epi, tile, a, e0, e1);
    return 1;
}

}  // namespace fg
