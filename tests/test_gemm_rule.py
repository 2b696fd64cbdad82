"""Which kernel a product takes, alone and as a forward's projection, without a
device: the tiled GEMM where it was measured faster than the other one, and not
where it was slower (the measurements stand beside the sizes)."""
import pytest

from ferrolm_amd import gpu
from ferrolm_amd.weights import BF16, INT4, INT8


# k_gemm's time, the tile's that the tile counts alone would choose
@pytest.mark.parametrize("kind,n,k,m", [
    (BF16, 4096, 4096, 256),    # 29.4, 34.5
    (BF16, 4096, 4096, 320),    # 33.9, 39.8
    (BF16, 2048, 2048, 400),    # 20.1, 23.0
    (BF16, 2048, 2048, 1024),   # 32.6, 36.2
    (BF16, 2048, 8192, 384),    # 51.3, 57.5
    (BF16, 16384, 2048, 160),   # 32.2, 36.5
    (BF16, 3584, 3584, 272),    # 27.4, 41.2
    (BF16, 3072, 2048, 832),    # 36.0, 43.0
    (INT4, 4096, 4096, 288),    # 38.2, 41.4
    (INT4, 2048, 2048, 320),    # 20.9, 22.8
    (INT4, 5120, 960, 224),     # 15.6, 18.8
    (INT4, 7168, 2560, 160),    # 1.22 times
    (INT4, 3072, 576, 832),     # 23.9, 27.1
    (INT8, 5120, 960, 240),     # 15.7, 18.1
    (INT8, 3072, 576, 512),     # 16.9, 18.5
    (INT8, 4096, 1024, 256),    # 1.10 times
    (BF16, 960, 576, 2048),     # 22.2, 26.4
    (BF16, 960, 960, 2048),     # 28.1, 32.0
])
def test_products_that_are_slower_on_the_tiles_stay_off_them(kind, n, k, m):
    assert gpu.mm_tile(kind, n, k, m) == (0, 0, 0)


@pytest.mark.parametrize("kind,n,k,m", [
    (INT4, 16384, 2048, 1024), (INT4, 6144, 2048, 1024), (INT4, 2048, 8192, 1024), (INT4, 28672, 4096, 80),
    (INT8, 16384, 2048, 160), (INT8, 2048, 2048, 576), (INT8, 960, 2560, 777), (BF16, 49152, 576, 33),
    (BF16, 6144, 2048, 512), (BF16, 2048, 8192, 1024), (INT8, 49152, 576, 33),
    # 572.9 to 419.7, 172.1 to 105.8, 863.1 to 657.7, 681.2 to 450.8, 307.2 to 204.6
    (BF16, 3072, 576, 32768), (BF16, 960, 2560, 6144), (BF16, 2048, 2048, 32768), (INT8, 3072, 576, 32768),
    (INT4, 960, 576, 32768)])
def test_products_that_gain_take_the_tiles(kind, n, k, m):
    assert gpu.mm_tile(kind, n, k, m)[0]


# o and down of a forward, their time on the tile over k_gemm's
@pytest.mark.parametrize("kind,n,k,m", [
    (BF16, 2048, 8192, 320),    # 1.31
    (BF16, 2048, 2048, 512),    # 1.10
    (BF16, 4096, 14336, 256),   # 1.33
    (BF16, 3072, 8192, 832),    # 1.22
    (BF16, 2560, 6912, 1024),   # 1.25
    (BF16, 2560, 2560, 1024),   # 1.08
    (INT8, 4096, 14336, 320),   # 1.11
    (INT4, 4096, 14336, 256),   # 1.25
    (INT4, 4096, 4096, 272),    # 1.06
])
def test_residual_products_that_are_slower_on_the_tiles_stay_off_them(kind, n, k, m):
    assert gpu.mm_tile(kind, n, k, m, "resid") == (0, 0, 0)


# a forward's products that gain, though some of them would not alone; the ratio again
@pytest.mark.parametrize("use,kind,n,k,m", [
    ("gate_up", BF16, 3072, 576, 1024),    # 17.4 us, 22.5 on k_gemm
    ("qkv", BF16, 3072, 2048, 832), ("resid", BF16, 576, 1536, 1024),  # 0.74
    ("resid", BF16, 960, 2560, 1024),      # 0.73
    ("resid", BF16, 2048, 8192, 1024),     # 0.89
    ("resid", INT4, 2048, 8192, 320),      # 0.83
    ("resid", INT8, 2048, 2048, 320),      # 0.84
    ("resid", INT4, 4096, 14336, 384),     # 0.65
    ("gate_up", INT4, 28672, 4096, 80), ("gate_up", INT8, 16384, 2048, 160), ("head", BF16, 128256, 4096, 80),
    ("qkv", INT4, 6144, 2048, 1024)])
def test_products_of_forwards_that_gain_take_the_tiles(use, kind, n, k, m):
    assert gpu.mm_tile(kind, n, k, m, use)[0]


def test_small_products_are_not_the_tiles():
    for kind in (BF16, INT8, INT4):
        for m in (1, 15, 16, 32):
            assert gpu.mm_tile(kind, 49152, 2048, m) == (0, 0, 0)
    with pytest.raises(gpu.FgError, match="bad argument"):
        gpu.mm_tile(INT4, 100, 2048, 64)
