"""A new cache is clear when fg_kv_create returns: rows written right after it
stay (the clear of a large cache takes milliseconds on the device, and one that
was still running could go over them)."""
import numpy as np
import pytest

from ferrolm_amd import gpu
from ferrolm_amd.weights import Config

pytestmark = pytest.mark.gpu


def test_rows_written_right_after_creation_stay(ctx):
    cfg = Config(vocab=512, hidden=128, intermediate=256, layers=256, heads=4, kv_heads=4, head_dim=128)
    rng = np.random.default_rng(3)
    for _ in range(3):
        kv = gpu.KvCache(ctx, cfg, 1024)  # 2 x 8 GiB: each clear takes over a millisecond
        n = 1024 * 16 * 4 * 128
        k, v = rng.standard_normal((2, n)).astype(np.float32)
        kv.set_layer(255, k, v)  # the part that a clear reaches last
        got = kv.layer(255)
        assert np.array_equal(got[0], k) and np.array_equal(got[1], v)
        assert not kv.layer(254)[1].any()
        kv.close()
