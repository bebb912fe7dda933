"""Plain products of 33 to 64 rows on tiles of 64 x 32 (`sliced_gemm_kernel`): walks of K of nine steps and more, with rows and columns that end
inside a tile."""
import pytest
import torch

from tests import test_gpu_sliced_tiles as sliced
from tests.test_gpu_sliced_tiles import chosen  # noqa: F401 (a fixture)

TALL = 6  # SLICES_64x32
SHAPES = [(64, 8192, 520), (50, 7008, 2048), (64, 7168, 2304), (48, 6432, 1000), (63, 8160, 1544), (33, 6400, 576)]


def test_the_sizes_here_reach_the_tile(chosen):  # noqa: F811
    assert all(chosen.plain(*shape) == TALL for shape in SHAPES)
    assert sliced.TILES[chosen.plain(33, 7008, 512) - 1] == sliced.TILES[chosen.plain(64, 8192, 512) - 1] == "32x64"


@pytest.mark.parametrize("shape", [(70, 4704, 688), (65, 5056, 568), (79, 4576, 664), (96, 5376, 832), (64, 7008, 3008), (64, 8224, 520), (64, 6368, 520),
                                   (32, 8192, 1024), (97, 4096, 2048)])
def test_products_that_stay_split_over_k(chosen, shape):  # noqa: F811
    """Timed on the GPU, the first three and the fifth: up to 8 % slower on tiles that walk K whole, from HBM or from L2. The others lie past the
    rule's lines."""
    assert chosen.plain(*shape) == 0


@pytest.mark.gpu
@sliced.DT
@pytest.mark.parametrize("bias", [False, True])
def test_plain_products(bias, dt, monkeypatch):
    monkeypatch.setitem(sliced.PLAIN, "64x32", SHAPES)
    sliced.test_plain_products("64x32", bias, dt)
