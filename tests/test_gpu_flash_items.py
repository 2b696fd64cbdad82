"""The flash attention items at the edges of their rule and of their parts: 64
rows and one fewer, 96 parts x kv heads (256 at head dim 128) and fewer, rows
that end an item, a
block of 64 (32 at head dim 128) positions and a part of 64, 128 or 256, or are
one short or over, after cached positions, and beside a chunk too short
to fill an item. All logits, the hidden states and the cache slots against the
oracle, with the bound of the other prefill tests."""
import numpy as np
import pytest

import oracle
from ferrolm_amd import gpu
from ferrolm_amd.synth import random_model
from ferrolm_amd.weights import Config

pytestmark = pytest.mark.gpu

# (heads, kv_heads, head_dim, [(cached positions, new rows) per sequence])
CASES = [(8, 8, 64, [(0, 63)]), (96, 96, 64, [(0, 64)]), (96, 96, 64, [(0, 63)]), (32, 32, 64, [(0, 64)]), (32, 32, 64, [(0, 65)]), (32, 32, 64, [(1, 127), (63, 129)]),
         (9, 3, 64, [(0, 211)]), (9, 3, 64, [(0, 240)]), (9, 3, 64, [(77, 401)]), (27, 9, 64, [(250, 261)]),
         (4, 4, 64, [(0, 640), (500, 577)]), (15, 5, 64, [(0, 20), (40, 20), (3, 41), (256, 60)]),
         (64, 64, 64, [(0, 300), (200, 5)]), (16, 16, 64, [(0, 255), (200, 1)]),
         (16, 4, 128, [(0, 96)]), (64, 16, 128, [(0, 176)]), (64, 16, 128, [(0, 160)]), (16, 4, 128, [(31, 130), (0, 16)]), (32, 8, 128, [(0, 257)]), (8, 8, 128, [(129, 191)])]


@pytest.mark.parametrize("heads,kv_heads,hd,seqs", CASES)
def test_prefill_at_the_edges(ctx, heads, kv_heads, hd, seqs):
    cfg = Config(vocab=96, hidden=heads * hd, intermediate=128, layers=1, heads=heads, kv_heads=kv_heads,
                 head_dim=hd, rms_eps=1e-5, rope_theta=10000.0, max_position=2048)
    hm = random_model(cfg, seed=5, std=0.03)
    rng = np.random.default_rng(6)
    tables, at = [], 0
    for pos, n in seqs:
        need = (pos + n + 15) // 16
        tables.append([int(x) for x in at + rng.permutation(need)])
        at += need
    toks = [[int(x) for x in rng.integers(0, 96, pos + n)] for pos, n in seqs]
    m, om = gpu.Model(ctx, hm), oracle.Model(hm)
    kv, okv = gpu.KvCache(ctx, cfg, at), om.kv(at)
    for i, (pos, _) in enumerate(seqs):
        if pos:
            gpu.forward(ctx, m, kv, [(toks[i][:pos], 0, tables[i], gpu.LOGITS_LAST)])
            om.forward(okv, [(toks[i][:pos], 0, tables[i], 1)])
    out = gpu.forward(ctx, m, kv, [(toks[i][pos:], pos, tables[i], gpu.LOGITS_ALL) for i, (pos, _) in enumerate(seqs)],
                      hidden=True)
    ol, oh = om.forward(okv, [(toks[i][pos:], pos, tables[i], 2) for i, (pos, _) in enumerate(seqs)], hidden=True)
    assert np.abs(out.logits - ol).max() < 1e-4 * np.abs(ol).max()
    assert (np.linalg.norm(out.hidden - oh, axis=-1) / np.linalg.norm(oh, axis=-1)).max() < 1e-4
    for g, o in zip(kv.layer(0), okv.layer(0)):
        assert np.abs(g - o).max() <= 1e-4 * np.abs(o).max()
