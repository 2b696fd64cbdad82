"""The tiled GEMM at the edges of its tiles: products for each tile shape (which
one a product takes is asserted), with outputs that are not a multiple of 64 or
128, rows that are not one of 16, an input of 5 k-blocks (padded to 8, so some
shares of K have one stage and some none left), of 35 (padded to 36: a last stage
that is not full) and of 65; outputs into a buffer aligned to a float only; and
forwards, one of them with every projection and so every epilogue on the tiles.

A product's rows are held as two bf16 pieces (2^-17 of each input) and summed in
f32, so |y - exact| <= 2e-5 * sum|x||w| as in the other products' tests."""
import ctypes as C

import numpy as np
import pytest

import oracle
from ferrolm_amd import gpu
from ferrolm_amd.weights import BF16, INT4, INT8, Config, Matrix

from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu

# (outputs, inputs, rows), and the tile that the product takes: row tiles, 64-column waves, K shares
# (None: not the same one for every weight kind)
SHAPES = [(10016, 160, 1000), (16448, 160, 400), (9440, 160, 517), (16448, 160, 200), (16448, 160, 83),
          (11456, 160, 129), (6560, 160, 200), (11456, 160, 67), (1856, 1120, 300),
          (16448, 1120, 200), (11456, 1120, 129), (6560, 1120, 200),
          (16448, 160, 129), (8416, 160, 129), (1856, 2080, 300), (11456, 1120, 83), (9440, 1120, 517)]
TILES = [(8, 4, 1), (5, 4, 1), (8, 4, 2), (5, 2, 2), None,
         (5, 2, 4), (4, 2, 4), None, None,
         (5, 2, 2), (5, 2, 4), (4, 2, 4),
         (4, 2, 2), (3, 2, 4), (2, 2, 4), (3, 2, 4), (8, 4, 2)]


def _matrix(kind, n, k, rng):
    w = (0.1 * rng.standard_normal((n, k))).astype(np.float32)
    if kind == BF16:
        return Matrix(BF16, n, k, bf16=(w.view(np.uint32) >> 16).astype(np.uint16))
    return oracle.quantize(kind, w)


@pytest.mark.parametrize("kind", [BF16, INT8, INT4], ids=["bf16", "int8", "int4"])
@pytest.mark.parametrize("n,k,m", SHAPES)
def test_products_of_every_tile_shape(ctx, kind, n, k, m):
    tile = TILES[SHAPES.index((n, k, m))]
    assert tile is None or gpu.mm_tile(kind, n, k, m) == tile
    rng = np.random.default_rng(n + k + m)
    w = _matrix(kind, n, k, rng)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[:, ::7] *= 20.0
    b = rng.standard_normal(n).astype(np.float32)
    y = gpu.Mat(ctx, w).matmul(x, b)
    deq = w.to_f32().astype(np.float64)
    scale = np.abs(x).astype(np.float64) @ np.abs(deq).T
    assert np.all(np.abs(y - (x.astype(np.float64) @ deq.T + b)) <= 2e-5 * scale + 1e-6)


@pytest.mark.parametrize("kind", [INT8, INT4], ids=["int8", "int4"])
@pytest.mark.parametrize("n,k,m", [(1856, 1120, 300), (16448, 1120, 200), (11456, 1120, 129), (6560, 1120, 200)])
def test_an_overflow_in_the_last_inputs_stays_an_infinity(ctx, kind, n, k, m):
    """35 k-blocks make 18 pairs: with four shares of K the last stage has work for two only, and what the
    others hold of the last pair must not reach the sum (a zero times an infinity)."""
    rng = np.random.default_rng(n + k + m)
    w = (0.1 * rng.standard_normal((n, k))).astype(np.float32)
    sign = np.where(np.arange(n) % 3, 1.0, -1.0).astype(np.float32)
    w[:, k - 5] = sign  # the largest of its group: the largest codes
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[m // 2, k - 5] = 3e38
    y = gpu.Mat(ctx, oracle.quantize(kind, w)).matmul(x)
    assert np.array_equal(y[m // 2], sign * np.float32(np.inf))
    assert np.isfinite(np.delete(y, m // 2, axis=0)).all()


def test_output_aligned_to_a_float(ctx):
    hip = Hip()
    rng = np.random.default_rng(1)
    n, k, m = 6560, 160, 200
    w = gpu.Mat(ctx, _matrix(INT4, n, k, rng))
    xh = rng.standard_normal((m, k)).astype(np.float32)
    x, y = hip.alloc(xh.nbytes), hip.alloc(4 * (m * n + 8))
    got = []
    try:
        hip.put(x, xh)
        for off in (0, 1):
            hip.put(y, np.full(m * n + 8, 7.0, np.float32))
            gpu.check(gpu.lib().fg_matmul_device(ctx.h, w.h, x, m, C.c_void_p(y.value + 4 * off)))
            ctx.sync()
            got.append(hip.get(y, m * n + 8))
    finally:
        hip.free(x, y)
    assert np.array_equal(got[0][:m * n], got[1][1:m * n + 1])
    assert got[1][0] == 7.0 and np.all(got[1][m * n + 1:] == 7.0)


# hidden, intermediate, heads of 32, kv heads, vocab, rows
WIDE = (1056, 4256, 33, 11, 6560, 600)  # 33 and 133 k-blocks; the head's rows on one tile, the rest as the rule has it
EVERY = (1440, 1440, 45, 15, 2080, 517)  # 45 k-blocks (padded to 48) everywhere, rows past a tile


def test_every_projection_takes_the_tiles():
    h, i, heads, kv, vocab, n = EVERY
    for kind in (BF16, INT8, INT4):
        for use, out, inp in (("qkv", (heads + 2 * kv) * 32, h), ("resid", h, heads * 32), ("gate_up", 2 * i, h),
                              ("resid", h, i)):
            assert gpu.mm_tile(kind, out, inp, n, use)[0], (kind, use, out, inp)
    assert gpu.mm_tile(BF16, vocab, h, n, "head")[0]


@pytest.mark.parametrize("kind", [BF16, INT8, INT4], ids=["bf16", "int8", "int4"])
@pytest.mark.parametrize("dims", [WIDE, EVERY], ids=["wide", "every"])
def test_forward_on_the_tiles_matches_oracle(ctx, kind, dims):
    """Two layers: q/k/v with a bias, o, gate/up, down (its padding after the last output's k-block too) and the
    lm_head, logits, hidden states and cache slots within 1e-4 of the oracle."""
    from ferrolm_amd.synth import quantize_model, random_model
    h, i, heads, kv_heads, vocab, n = dims
    cfg = Config(vocab=vocab, hidden=h, intermediate=i, layers=2, heads=heads, kv_heads=kv_heads, head_dim=32,
                 rms_eps=1e-5, max_position=1024, qkv_bias=True)
    hm = quantize_model(random_model(cfg, seed=7, std=0.03), kind)
    prompt = [int(t) for t in np.random.default_rng(8).integers(0, cfg.vocab, n)]
    blocks = (n + 15) // 16
    table = [(i * 7) % blocks for i in range(blocks)]
    m, kv = gpu.Model(ctx, hm), gpu.KvCache(ctx, cfg, blocks)
    out = gpu.forward(ctx, m, kv, [(prompt, 0, table, gpu.LOGITS_ALL)], hidden=True)
    om = oracle.Model(hm)
    okv = om.kv(blocks)
    ol, oh = om.forward(okv, [(prompt, 0, table, 2)], hidden=True)
    assert np.abs(out.logits - ol).max() < 1e-4 * np.abs(ol).max()
    rel = np.linalg.norm(out.hidden - oh, axis=-1) / np.linalg.norm(oh, axis=-1)
    assert rel.max() < 1e-4, rel.max()
    top2 = np.sort(ol, axis=1)[:, -2:]
    clear = top2[:, 1] - top2[:, 0] > 2e-4 * np.abs(ol).max()
    assert clear.mean() > 0.9 and np.array_equal(out.argmax[clear], ol.argmax(axis=1)[clear])
    for li in range(cfg.layers):
        for g, o in zip(kv.layer(li), okv.layer(li)):
            assert np.abs(g - o).max() <= 1e-4 * np.abs(o).max()
