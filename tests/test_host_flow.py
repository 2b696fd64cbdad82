"""The library's host code on a HIP runtime of the CPU (fake_hip.cpp) that runs
queued work as late as a device may: memory is clear before a handle to it is
returned, and a failed call leaves nothing behind."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

# the fake's names come first in the library's symbol lookup
PRELUDE = """
import ctypes, sys
import numpy as np
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
from ferrolm_amd import gpu, host
from ferrolm_amd.weights import INT4, INT8, Config
fail = lambda name, nth=1: fake.fake_fail(name.encode(), nth)
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    """Runs code after PRELUDE in a process of its own, which has no other HIP runtime to find."""
    lib = tmp_path_factory.mktemp("hip") / "libfake_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-o", str(lib),
                    str(ROOT / "tests" / "fake_hip.cpp"), "-ldl", "-lpthread"], check=True, timeout=120)

    def go(code):
        env = dict(os.environ, FERRO_GPU_LIB=str(ROOT / "ferrolm_amd" / "libferro_gpu.so"))
        r = subprocess.run([sys.executable, "-c", PRELUDE + code, str(lib)], cwd=ROOT, env=env, capture_output=True,
                           text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr

    return go


def test_a_new_context_waits_for_its_counters_to_be_clear(run):
    """The split products' arrival counters: a clear left on the default stream would run beside the first
    launches on the context's stream, which does not wait for it."""
    run("""
c = gpu.Context(0)
assert fake.fake_pending_default() == 0
c.close()
""")


def test_no_clear_is_left_on_the_default_stream():
    """No source of the library clears memory on the default stream, where no launch waits for it."""
    for p in (ROOT / "ferrolm_amd" / "csrc").iterdir():
        assert "hipMemset(" not in p.read_text(), p


def test_a_new_cache_is_clear_for_every_context(run):
    """Rows that a second context writes to a cache just made stay: the clear does not run after them."""
    run("""
a, b = gpu.Context(0), gpu.Context(0)
cfg = Config(vocab=32, hidden=32, intermediate=32, layers=1, heads=2, kv_heads=2, head_dim=16)
kv = gpu.KvCache(a, cfg, 4)
k, v = np.random.default_rng(0).standard_normal((2, 4 * 16 * 2 * 16)).astype(np.float32)
kv.ctx = b
kv.set_layer(0, k, v)
a.sync()
got = kv.layer(0)
assert np.array_equal(got[0], k) and np.array_equal(got[1], v)
""")


@pytest.mark.parametrize("failing", ["kv = gpu.KvCache(c, cfg, 1 << 30)", "fail('hipMemsetAsync'); gpu.KvCache(c, cfg, 4)",
                                     "fail('hipStreamCreateWithFlags'); gpu.Context(0)",
                                     "fail('hipMalloc'); gpu.quantize(c, INT4, w)"])
def test_a_failed_call_leaves_no_error_for_the_next(run, failing):
    run(f"""
c = gpu.Context(0)
cfg = Config(vocab=32, hidden=32, intermediate=32, layers=1, heads=2, kv_heads=2, head_dim=128)
w = np.random.default_rng(0).standard_normal((32, 64)).astype(np.float32)
try:
    {failing}
    assert False
except gpu.FgError as e:
    assert "failed" in str(e)
got, want = gpu.quantize(c, INT4, w), host.quantize(INT4, w)
assert np.array_equal(got.q, want.q) and np.array_equal(got.s, want.s)
""")


SHAPES = [(32, 32), (64, 2048), (1056, 1024), (2080, 2080), (224, 32800)]  # the last two over 16 MB, in panels and whole


@pytest.mark.parametrize("refused", [None, ("hipHostMalloc", 1), ("hipStreamCreateWithFlags", 3),
                                     ("hipEventCreateWithFlags", 8)])
def test_quantizer_copies_with_and_without_staging(run, refused):
    """Every size class of host copy, whole or in panels through staging slots, and with the slots refused:
    codes and scales are the host quantizer's."""
    run(f"""
refused = {refused!r}
rng = np.random.default_rng(0)
for rows, cols in {SHAPES!r}:
    w = rng.standard_normal((rows, cols)).astype(np.float32)
    for imp in (None, rng.random(cols).astype(np.float32)):
        c = gpu.Context(0)
        if refused:
            fail(*refused)
        got, want = gpu.quantize(c, INT4, w, imp), host.quantize(INT4, w, imp)
        assert np.array_equal(got.q, want.q) and np.array_equal(got.s, want.s), (rows, cols, imp is None)
        if refused:
            fail(refused[0], 0)
        c.close()
""")


def test_a_small_quantizer_call_waits_once(run):
    """Its copies are queued one after the other and waited for together."""
    run("""
c = gpu.Context(0)
w = np.random.default_rng(0).standard_normal((64, 2048)).astype(np.float32)
for imp in (None, np.ones(2048, np.float32)):
    before = fake.fake_waits()
    gpu.quantize(c, INT8, w, imp)
    assert fake.fake_waits() == before + 1
""")


def test_the_search_takes_many_calibration_rows(run):
    """600,000 rows: more than one grid's worth of row groups."""
    run("""
c = gpu.Context(0)
gpu.awq_search(c, INT8, np.ones((32, 32), np.float32), np.ones((600_000, 32), np.float32))
assert 0 < fake.fake_widest() <= 65535
""")


@pytest.mark.parametrize("rows,cols,staged", [(1024, 1024, 0), (2048, 2016, 0), (2048, 2048, 1), (192, 32800, 0)])
def test_the_quantizer_takes_the_staging_slots_for_large_matrices_only(run, rows, cols, staged):
    """In panels from 16 MB on; whole (a panel of more than 4 MB) from 28 MB on: below, the runtime's own copies
    are faster."""
    run(f"""
c = gpu.Context(0)
gpu.quantize(c, INT4, np.ones(({rows}, {cols}), np.float32))
assert fake.fake_pinned() == {staged}
""")
