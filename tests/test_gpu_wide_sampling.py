"""Wide distributions (top_k 0 or above 1024) over logits chosen to reach every
branch of the sort and of the sequential sums: a vocabulary of one tile, of a
tile and a bit and of several; equal logits, runs of equal logits, steps of
powers of two (sums full of rounding ties), one dominant token, exponentials
down to the smallest, and ordinary noise. Tokens and generator states equal the
oracle's on the device's own logits."""
import numpy as np
import pytest

import oracle
from ferrolm_amd import gpu
from ferrolm_amd.gpu import SamplingParams
from ferrolm_amd.weights import Config, HostModel

pytestmark = pytest.mark.gpu

H = 32


def _columns(vocab, rng):
    """One logits row per input token: column t of the head (the embedding of t is a unit vector)."""
    i = np.arange(vocab)
    cols = [np.zeros(vocab), (i % 7).astype(float), -np.log(2.0) * (i % 24), np.where(i == vocab // 2, 30.0, 0.0),
            -60.0 * i / vocab, -90.0 * rng.random(vocab), 3.0 * rng.standard_normal(vocab),
            0.01 * rng.standard_normal(vocab), -np.log(2.0) * (i % 3), np.where(i % 5, -200.0, 1.0)]
    w = np.zeros((vocab, H), np.float32)
    w[:, :len(cols)] = np.stack(cols, axis=1)
    return w, len(cols)


@pytest.mark.parametrize("vocab", [32, 1024, 1056, 9216])
def test_wide_draws_equal_the_oracle(ctx, vocab):
    rng = np.random.default_rng(vocab)
    head, n = _columns(vocab, rng)
    bf = lambda a: (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)
    embed = np.zeros((vocab, H), np.float32)
    embed[np.arange(H), np.arange(H)] = 1.0
    cfg = Config(vocab=vocab, hidden=H, intermediate=64, layers=0, heads=2, kv_heads=1, head_dim=16,
                 max_position=64)
    hm = HostModel(cfg=cfg, embed=bf(embed), norm=np.full(H, 1 / np.sqrt(H), np.float32), layers=[], lm_head=bf(head))
    m = gpu.Model(ctx, hm)
    kv_cfg = Config(**{**cfg.__dict__, "layers": 1})
    toks = list(range(n))
    chunk = [(toks, 0, [0, 1], gpu.LOGITS_ALL)]
    lg = gpu.forward(ctx, m, gpu.KvCache(ctx, kv_cfg, 2), chunk).logits
    for seed, p in enumerate([SamplingParams(1.0, 1.0, 0), SamplingParams(0.7, 0.9, 0), SamplingParams(1.0, 0.999, 0),
                              SamplingParams(1.3, 1e-6, 0), SamplingParams(1.0, 0.0, 0),
                              SamplingParams(0.9, 0.8, max(1025, vocab - 5))]):
        for rep in range(6):
            st = np.array([gpu.rng_init(100 * seed + 20 * rep + j) for j in range(n)], np.uint64)
            got = gpu.forward_sampled(ctx, m, gpu.KvCache(ctx, kv_cfg, 2), chunk, [p] * n, st)
            for j in range(n):
                r = oracle.Rng(100 * seed + 20 * rep + j)
                assert int(got[j]) == oracle.sample(lg[j], (p.temperature, p.top_p, p.top_k), r), (j, p, rep)
                assert int(st[j]) == r.state


def _special(vocab, rng, nan):
    """Head columns with values that overflow to infinities at temperature 0.5 (3e38 / 0.5); with nan, also two
    rows whose logits are NaN for every token (an infinite weight that meets a zero input)."""
    base = rng.standard_normal(vocab)
    cols = [base.copy() for _ in range(6)]
    cols[0][vocab // 2] = 3e38
    cols[1][::3] = -3e38
    cols[2][[7, vocab - 3]] = 3e38, -3e38
    cols[3][[9, vocab // 3]] = 3e38
    cols[4][:] = -3e38
    w = np.zeros((vocab, H), np.float32)
    w[:, :len(cols)] = np.stack(cols, axis=1)
    if nan:
        w[[5, vocab - 40], H - 1] = np.inf, -np.inf
    return w, len(cols)


@pytest.mark.parametrize("vocab", [1056, 9216])
@pytest.mark.parametrize("nan", [False, True], ids=["inf", "nan"])
def test_wide_draws_with_infinite_and_nan_logits(ctx, vocab, nan):
    rng = np.random.default_rng(vocab)
    head, n = _special(vocab, rng, nan)
    bf = lambda a: (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)
    embed = np.zeros((vocab, H), np.float32)
    embed[np.arange(H), np.arange(H)] = 1.0
    cfg = Config(vocab=vocab, hidden=H, intermediate=64, layers=0, heads=2, kv_heads=1, head_dim=16,
                 max_position=64)
    hm = HostModel(cfg=cfg, embed=bf(embed), norm=np.full(H, 1 / np.sqrt(H), np.float32), layers=[], lm_head=bf(head))
    m = gpu.Model(ctx, hm)
    kv_cfg = Config(**{**cfg.__dict__, "layers": 1})
    chunk = [(list(range(n)), 0, [0, 1], gpu.LOGITS_ALL)]
    lg = gpu.forward(ctx, m, gpu.KvCache(ctx, kv_cfg, 2), chunk).logits
    assert np.isnan(lg).sum() == (2 * n if nan else 0)
    with np.errstate(over="ignore"):
        assert np.isposinf(lg[0] / np.float32(0.5)).any() and np.isneginf(lg[1] / np.float32(0.5)).any()
    for seed, p in enumerate([SamplingParams(0.5, 1.0, 0), SamplingParams(0.5, 0.9, 0), SamplingParams(0.5, 0.0, 0),
                              SamplingParams(1.0, 0.9, 0), SamplingParams(0.5, 0.95, vocab - 7)]):
        for rep in range(3):
            st = np.array([gpu.rng_init(100 * seed + 20 * rep + j) for j in range(n)], np.uint64)
            got = gpu.forward_sampled(ctx, m, gpu.KvCache(ctx, kv_cfg, 2), chunk, [p] * n, st)
            for j in range(n):
                r = oracle.Rng(100 * seed + 20 * rep + j)
                assert int(got[j]) == oracle.sample(lg[j], (p.temperature, p.top_p, p.top_k), r), (j, p, rep)
                assert int(st[j]) == r.state
