"""Bfloat16 heads of 64 columns whose tiles one wavefront walks (rows through LDS for both kinds of product), against the float64 oracle:
entry lists of every length around a block and around a piece of a list on either side, rows in one piece and split rows, with dropout,
heads that take one, two and four workgroups a tile.  (The same kernels in two and four parts: test_gpu_tile_parts.py; with a
score term: test_gpu_rel_pos.py.)  Dropout goes with the lists of the source side: a query row that one pair is left of has no gradient
in q and k but for the rounding of its bfloat16 result, 2^-9 of dO . o, which a bound by the gradients' size does not hold."""
import pytest
import test_gpu_tile_parts as tiles

CASES = [(n_tiles, flip, heads, 64, tiles.BF16, p, seg, 1, 1) for n_tiles, heads in ((400, 8), (200, 16), (640, 4))
         for flip, p, seg in ((False, 0.0, 256), (True, 0.0, 256), (False, 0.0, 32), (True, 0.25, 32))]


@pytest.mark.gpu
@pytest.mark.parametrize("n_tiles,flip,heads,d,dtype,p,seg,parts_dst,parts_src", CASES)
def test_rows_through_lds_match_the_oracle(n_tiles, flip, heads, d, dtype, p, seg, parts_dst, parts_src, monkeypatch):
    tiles.test_tiles_in_parts_match_the_oracle(n_tiles, flip, heads, d, dtype, p, seg, parts_dst, parts_src, monkeypatch)
