"""The tile shape that the GEMM estimate takes (host code, no device), where
the text's tiles would open a further round of tiles: 64 text rows beside video
tiles that fill the CUs to the last few. Each case names the shapes that were
measured within 8 % of the best one (tile index as in csrc/dit_gemm.hip)."""

import ctypes

import pytest

import awa_hip as A
from test_gpu_gemm_tiles import GemmStep


@pytest.mark.parametrize("split,rows,n,k,good", [
    (0, 3078, 2560, 2560, {1, 3}),  # 128 x 256: 250 + 10 tiles, 82 us against 59
    (0, 3078, 2560, 6912, {1, 3}),  # 184 / 136
    (0, 1000, 7680, 2560, {1}),     # 240 + 30 tiles, 81 / 58
    (0, 700, 13824, 2560, {3}),     # 256 x 192: 216 + 108 tiles, 92 / 66
    (0, 2048, 7680, 2560, {2}),     # 256 x 256: 240 + 30 tiles, 110 / 85
    (1, 3078, 2560, 6912, {1, 3, 4}),  # 431 / 339
    (1, 1000, 7680, 2560, {1, 3}),  # 175 / 136
    (1, 2048, 7680, 2560, {2}),     # 260 / 207
])
def test_text_tiles_count_as_a_round(split, rows, n, k, good):
    step = GemmStep(split=split, tile=-1, n=n, k=k)
    step.rows[0], step.rows[1] = rows, 64
    assert A.lib().awa_gemm_step_tile(ctypes.byref(step)) in good
