"""Which grouped products go to tiles of one workgroup per unit (`grouped_slices`), by what was timed on the GPU with uniform and with skewed routing."""
import pytest

from tests.test_gpu_sliced_tiles import TILES, chosen  # noqa: F401 (a fixture)


@pytest.mark.parametrize("groups,rows,n,k,tile", [
    (27, 173, 864, 2536, None), (49, 149, 512, 2584, None), (6, 172, 4192, 3248, None), (53, 61, 544, 1200, None),  # Zipf's routing: up to 1.53 times as long
    (7, 166, 2048, 2576, "128x128"), (6, 139, 2496, 672, "128x128"), (3, 1192, 960, 752, None),
    (30, 152, 736, 536, "192x128"), (8, 115, 2048, 8192, "128x128"), (8, 150, 2048, 8192, "192x128"),
])
def test_tiles_that_make_no_second_round(chosen, groups, rows, n, k, tile):  # noqa: F811
    way = chosen.grouped(groups * rows, groups, n, k)
    assert (TILES[way - 1] if way else None) == tile
