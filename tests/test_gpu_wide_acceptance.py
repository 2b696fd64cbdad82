"""Sampled speculative steps over wide distributions (top_k 0 or above 1024) of
several tiles of the sequential sums (9216 tokens; a tile is 4096 terms), on
models without layers, so that a row's logits are a chosen column of the head:
a residual that lies late, a draft equal to the target (nothing left over), flat
and tied distributions, one dominant last token, exponentials down to the
smallest; and generator states whose uniform is next to one where the residual
is drawn, so that a walk ends at or past its last term. Tokens, accepted counts
and generator states equal the oracle's on the device's own logits."""
import numpy as np
import pytest

import oracle
from ferrolm_amd import gpu
from ferrolm_amd.gpu import SamplingParams
from ferrolm_amd.weights import Config, HostModel

pytestmark = pytest.mark.gpu

V, H, CASES = 9216, 64, 8


def _heads(rng):
    i = np.arange(V)
    noise = lambda s: s * rng.standard_normal(V)
    base, flat, ln2 = noise(3.0), np.zeros(V), np.log(2.0)
    p = [base, -0.002 * (V - i), base, flat, np.where(i % 3, -200.0, 1.0), -ln2 * (i % 24),
         np.where(i == V - 1, 12.0, 0.0), -90.0 * rng.random(V)]
    q = [base + noise(0.7), -0.002 * i, base, noise(0.05), flat, -ln2 * ((i + 3) % 24),
         np.where(i == 0, 9.0, 0.0), flat]
    return p, q


def _model(ctx, columns):
    """Token t's logits are column t % CASES: its embedding is a unit vector, and the norm (1/8, a power of
    two) leaves one product per logit, the same in every path."""
    bf = lambda a: (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)
    cfg = Config(vocab=V, hidden=H, intermediate=64, layers=0, heads=2, kv_heads=1, head_dim=32, max_position=64)
    embed, head = np.zeros((V, H), np.float32), np.zeros((V, H), np.float32)
    embed[np.arange(V), np.arange(V) % CASES] = 1.0
    head[:, :CASES] = np.stack(columns, axis=1)
    hm = HostModel(cfg=cfg, embed=bf(embed), norm=np.full(H, 0.125, np.float32), layers=[], lm_head=bf(head))
    kv_cfg = Config(**{**cfg.__dict__, "layers": 1})
    m = gpu.Model(ctx, hm)
    rows = gpu.forward(ctx, m, gpu.KvCache(ctx, kv_cfg, 2), [(list(range(CASES)), 0, [0, 1], gpu.LOGITS_ALL)]).logits
    return m, kv_cfg, rows


class _Rows:
    """The device's logits, where the oracle's step asks a model for its own."""

    def __init__(self, cfg, rows):
        self.cfg, self.rows = cfg, rows

    def forward(self, kv, chunks):
        (tok, _, _, mode), = chunks
        return self.rows[[t % CASES for t in (tok if mode == 2 else tok[-1:])]]


def _state_before(uniform53, draws):
    """The generator state whose draws-th uniform is uniform53 / 2^53."""
    mask = (1 << 64) - 1
    s = ((uniform53 << 11) | 0x400) * pow(0x2545F4914F6CDD1D, -1, 1 << 64) & mask
    for _ in range(draws):  # undo x ^= x >> 12; x ^= x << 25; x ^= x >> 27
        for step, right in ((27, True), (25, False), (12, True)):
            t = s
            for _ in range(64 // step + 1):
                t = s ^ ((t >> step) if right else (t << step) & mask)
            s = t
    return s


def test_state_before_is_the_inverse():
    r = oracle.Rng(state=_state_before((1 << 53) - 3, 3))
    r.uniform(), r.uniform()
    assert r.uniform() == 1.0 - 3 * 2.0**-53


@pytest.mark.parametrize("params", [SamplingParams(1.0, 1.0, 0), SamplingParams(0.7, 0.9, 0),
                                    SamplingParams(1.2, 0.97, 3000), SamplingParams(1.0, 0.999, 0)],
                         ids=["all", "p0.9", "k3000", "p0.999"])
def test_steps_equal_the_oracle(ctx, params):
    rng = np.random.default_rng(17)
    p, q = _heads(rng)
    tm, kv_cfg, prow = _model(ctx, p)
    dm, _, qrow = _model(ctx, q)
    target, draft = _Rows(tm.cfg, prow), _Rows(dm.cfg, qrow)
    prm = (params.temperature, params.top_p, params.top_k)
    states = [[gpu.rng_init(1000 * rep + j) for j in range(CASES)] for rep in range(6)]
    # the third uniform of a step with one proposal draws its residual
    states += [[_state_before((1 << 53) - 1 - 7 * CASES * rep - j, 3) for j in range(CASES)] for rep in range(4)]
    accepted = proposed = 0
    for rep, st in enumerate(states):
        k = 3 if rep < 6 else 1
        tkv, dkv = gpu.KvCache(ctx, kv_cfg, CASES), gpu.KvCache(ctx, kv_cfg, CASES)
        block = lambda j: np.array([j], np.uint32)
        seqs = [gpu.SpecSeq(tail=np.array([j], np.uint32), draft_pos=0, pos=0, blocks=block(j), draft_blocks=block(j))
                for j in range(CASES)]
        got_st = np.array(st, np.uint64)
        toks, acc = gpu.spec_step(ctx, tm, tkv, dm, dkv, seqs, k, params=[params] * CASES, rng=got_st)
        for j in range(CASES):
            r = oracle.Rng(state=st[j])
            new, a, _, _ = oracle.spec_step_sampled(target, None, draft, None, [j], 0, 0, [j], [j], k, prm, r)
            assert toks[j].tolist() == new and int(acc[j]) == a and int(got_st[j]) == r.state, (rep, j)
            accepted += a
            proposed += k
    assert 0 < accepted < proposed
