"""The size rules of the dispatch, at sizes where the variants on their two sides were measured to differ."""
import pytest

import routes


@pytest.mark.parametrize("rows,k,in_launch", [(1, 4096, True), (16, 7168, True), (1, 65536, True), (4096, 32, True), (8192, 8320, True), (16384, 288, False),
                                              (1, 131072, False), (16, 262144, False), (1, 1 << 20, False), (16384, 32, False),
                                              (65536, 32, False), (262144, 96, False), (65536, 1056, False),
                                              (64, 1 << 20, True), (1 << 20, 2048, False), ((1 << 20) - 1, 2048, False)])
def test_padding_of_tiled_mx_scales(rows, k, in_launch):
    """Padded in the quantiser's own launch up to four million elements in all or three million of padding; arrays without padding always (the grid is the same)
    as long as their elements can be counted with 31 bits."""
    assert routes.mx_padding_in_launch(rows, k) is in_launch
