"""The library's choice of tiles and K ranges (unok_gemm_nt_plan, a function of the sizes alone) at sizes
on both sides of its lines, where both sides were measured."""
import pytest

from uno_amd import _native as N
from uno_amd import kernels as K

F32_64, F32_32 = 7, 8


@pytest.fixture(autouse=True)
def _built():
    if not N.LIB_PATH.exists():
        pytest.skip("libunok.so not built")


def _f32(M, Nn, Kd, K2=0):
    return N.lib().unok_gemm_nt_plan(N.F32, M, Nn, Kd, K2, 1 if K2 else 0, N.int_array([Nn] if K2 else []))


# us on 64x64 / 32x32 tiles: the last figures of each line
@pytest.mark.parametrize("M,Nn,Kd,K2,tile", [
    (1334, 4096, 8, 0, F32_64),      # 11 / 42
    (3837, 1536, 64, 8, F32_64),     # 33 / 62
    (3502, 1536, 33, 32, F32_64),    # 29 / 69
    (407, 4096, 8, 8, F32_64),       # 9 / 16
    (4066, 1024, 256, 32, F32_64),   # 67 / 77
    (4096, 1536, 128, 0, F32_64),    # 40 / 50
    (4096, 1536, 256, 0, F32_32),    # 71 / 65
    (512, 4096, 128, 0, F32_32),     # 23 / 20
    (1024, 1536, 256, 0, F32_32),    # 40 / 20
    (2048, 768, 4096, 0, F32_32),    # 594 / 232
    (512, 768, 256, 8, F32_32),      # 33 / 8, the parity step's products
    (2000, 1536, 255, 0, F32_64),    # 46 / 72 (K no multiple of 4: element loads)
    (2000, 250, 9, 0, F32_64),       # 6.1 / 7.6
    (300, 770, 255, 0, F32_32),      # 33 / 9
    (2048, 256, 8, 0, F32_32),       # 6 / 6
    (8192, 2048, 256, 0, F32_64),    # from 2048 tiles on
])
def test_fp32_tiles(M, Nn, Kd, K2, tile):
    assert _f32(M, Nn, Kd, K2) == tile + 16


def _bf16(M, Nn, Kd, K2=0):
    return K.nt_plan(M, Nn, Kd, K2, (Nn,) if K2 else ())


SKINNY, REG = 4, 0


# us in one range / in the ranges taken: the last figures of each line
@pytest.mark.parametrize("M,Nn,Kd,tile,splits", [
    (8192, 64, 1024, SKINNY, 1),      # 9.4 / 14.0 in four
    (6000, 128, 1024, SKINNY, 1),     # 13.1 / 15.6 in two
    (15955, 32, 1024, SKINNY, 1),     # 9.6 / 13.0 in two
    (15955, 64, 2048, SKINNY, 1),     # 15.1 / 19.0 in two
    (4096, 192, 1024, SKINNY, 1),     # 15.8 / 17.2 in two
    (12000, 64, 12288, SKINNY, 1),    # 70 / 74 in two: the activations' bytes
    (16384, 64, 4096, SKINNY, 1),
    (777, 192, 128, REG, 1),          # 7.1 / 7.8 on 64-row tiles
    (8192, 192, 128, SKINNY, 1),
])
def test_skinny_products_in_one_range(M, Nn, Kd, tile, splits):
    assert _bf16(M, Nn, Kd) == (tile, splits)


@pytest.mark.parametrize("M,Nn,Kd", [(2048, 64, 4096),     # 24 / 14
                                     (777, 192, 12288),    # 112 / 21
                                     (17, 32, 2048),       # 14 / 7
                                     (6000, 64, 4096),     # 24 / 17
                                     (8192, 128, 12288)])  # 90 / 57
def test_skinny_products_in_ranges(M, Nn, Kd):
    tile, splits = _bf16(M, Nn, Kd)
    assert tile == SKINNY and splits > 1


@pytest.mark.parametrize("M,Nn,Kd", [(300, 4096, 12288), (485, 4096, 12288), (1196, 2048, 11008), (777, 4096, 4096),
                                     (64, 4096, 4096), (5, 512, 192), (3000, 24576, 4096)])
@pytest.mark.parametrize("K2", [32, 64, 128, 384])
def test_an_extension_leaves_the_ranges(M, Nn, Kd, K2):
    """The same K ranges with and without an extension, so that one of zeros changes no bit."""
    assert _bf16(M, Nn, Kd, K2)[1] == _bf16(M, Nn, Kd)[1]
