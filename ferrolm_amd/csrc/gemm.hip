// Which products run on the tiled GEMM (gemm_tiles.h), and on which tile.
#include "internal.h"

namespace fg {

template <int KIND>
void run_mm(hipStream_t st, int epi, int cfg, const GemvArgs& a, hipEvent_t e0, hipEvent_t e1);
extern template void run_mm<BF16>(hipStream_t, int, int, const GemvArgs&, hipEvent_t, hipEvent_t);
extern template void run_mm<INT8>(hipStream_t, int, int, const GemvArgs&, hipEvent_t, hipEvent_t);
extern template void run_mm<INT4>(hipStream_t, int, int, const GemvArgs&, hipEvent_t, hipEvent_t);

// The tile shapes (run_mm_epi's cases): row tiles, 64-column waves, K shares; the time of a stage in
// us on a full chip, for a CU's only workgroup and (four waves: two of them fit a CU) for two.
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

int launch_mm(hipStream_t st, int epi, const DMat& w, const GemvArgs& a, hipEvent_t e0, hipEvent_t e1) {
    const int rt = (a.p_total + 3) / 4;
    if (rt < 3) return 0;
    int cfg = -1, tiles = 0;
    float best = 0.0f;
    for (int i = 0; i < (int)(sizeof(kTiles) / sizeof(kTiles[0])); i++) {
        const auto& c = kTiles[i];
        const int n = ((rt + c.rt - 1) / c.rt) * ((a.N + 64 * c.nwn - 1) / (64 * c.nwn));
        const float start = 5.0f, stages = (float)((a.KB / 2 + c.nwk - 1) / c.nwk);  // start: first loads, epilogue
        float t;
        if (c.nwn * c.nwk == 8) {
            t = (float)((n + 255) / 256) * (start + stages * c.one);
        } else {
            const int rest = n % 512;
            t = (float)(n / 512) * (start + stages * c.two);
            if (rest) t += start + stages * (rest > 256 ? c.two : c.one);
        }
        if (cfg < 0 || t < best) {
            cfg = i;
            best = t;
            tiles = n;
        }
    }
    // k_gemm splits K finer and wins where the tiles leave CUs idle. Its time, then the tiles', in us:
    // 2048 x 8192 at 256 rows (128 tiles) 42 against 59, at 320 (160) 69 against 61; 6144 x 2048 at 160
    // (240 of two row tiles) even, 22.4 against 21.9, at 192 (192 of three) 32.2 against 25.3; and on
    // short K with two row tiles 960 x 576 at 1024 rows 14.5 against 16.2.
    if (kTiles[cfg].rt == 2 ? tiles < 150 || a.m < 256 || a.KB < 32 : tiles < 180) return 0;
    if (w.kind == INT4)
        run_mm<INT4>(st, epi, cfg, a, e0, e1);
    else if (w.kind == INT8)
        run_mm<INT8>(st, epi, cfg, a, e0, e1);
    else
        run_mm<BF16>(st, epi, cfg, a, e0, e1);
    return 1;
}

}  // namespace fg
