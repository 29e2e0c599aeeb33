"""AUTO's line between the vector ALU and packed rows where a row is one group of words and results are many
(valu_ahead_of_rows in fastertnn_amd/csrc/ftnn_api.hip): either side of it, by type and layout; no scratch on either."""
import pytest

# (type, n, oh, ow, kernels, words)
LINES = [
    ((0, 161290, 1, 1, 31, 4), (0, 161291, 1, 1, 31, 4)), ((1, 312499, 1, 1, 16, 4), (1, 312500, 1, 1, 16, 4)), ((3, 400000, 1, 1, 15, 4), (3, 400000, 1, 1, 17, 4)),
    ((2, 1499, 1, 1, 1000, 4), (2, 1500, 1, 1, 1000, 4)), ((2, 1, 75, 99, 200, 4), (2, 1, 75, 100, 200, 4)), ((0, 1, 75, 99, 200, 4), (0, 1, 75, 100, 200, 4)),
    ((1, 1, 75, 99, 200, 4), (1, 1, 75, 100, 200, 4)), ((3, 1, 125, 259, 100, 4), (3, 1, 125, 260, 100, 4)), ((3, 16, 500, 500, 15, 4), (3, 16, 500, 500, 16, 4)),
]


@pytest.mark.parametrize("valu,rows", LINES)
def test_auto_line_of_many_results(valu, rows):
    import fastertnn_amd.lib as lib
    assert lib.mm_auto_engine(*valu) == lib.ENGINE_VALU
    assert lib.mm_auto_engine(*rows) == lib.ENGINE_MFMA_F4
    assert lib.mm_scratch_bytes(lib.ENGINE_AUTO, *valu) == lib.mm_scratch_bytes(lib.ENGINE_AUTO, *rows) == 0
