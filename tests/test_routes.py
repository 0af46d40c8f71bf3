"""Which kernel a call of given sizes takes (hf_route, at 256 CUs). CPU only: no kernel runs here; the tests of each
kernel use the same query for the sizes that they claim reach it."""

from __future__ import annotations

import pytest

from hyperflow_h3_flash_amd import _native


def up(m, n, r):
    return _native.library().hf_route(_native.ROUTE_UP_ROWS, m, n, 0, r)


def test_unknown_queries_and_sizes_are_zero():
    lib = _native.library()
    assert lib.hf_route(99, 4096, 4096, 4096, 64) == 0
    assert up(0, 4096, 64) == up(4096, 0, 64) == up(4096, 4096, 0) == up(37710, 7168, 264) == 0


# Measured against the kernels it replaces (us, tiles -> u in registers): where it is behind it is not taken. Ranks up to
# 64, outputs that the tiles leave in the Infinity Cache (50 -> 62, 51 -> 60, 23 -> 25, 38 -> 46, 54 -> 60); one tile of
# 128 columns (204 -> 254); narrow outputs at large ranks (25 -> 31, 26 -> 32, 24 -> 27, 22 -> 25); few steps (10.8 ->
# 12.7); 352 rows in blocks of 256.
@pytest.mark.parametrize("m,n,r", [
    (32768, 4096, 16), (131072, 1024, 32), (16384, 3072, 32), (14003, 7168, 16), (8192, 16384, 64), (3094835, 128, 64),
    (49152, 512, 200), (98304, 256, 256), (24576, 1024, 256), (98304, 256, 136), (1536, 8192, 192), (352, 19072, 64),
])
def test_up_projection_stays_on_tiles_where_they_are_ahead(m, n, r):
    assert up(m, n, r) == 0


@pytest.mark.parametrize("m,n,r", [
    (37710, 7168, 256), (37710, 7168, 64), (37710, 7168, 96), (41344, 2048, 256), (8192, 4096, 256),
    (2048, 4096, 64), (16384, 1024, 32), (65536, 192, 32), (130000, 512, 64), (131072, 192, 256),
])
def test_up_projection_keeps_u_in_registers_where_that_is_ahead(m, n, r):
    assert up(m, n, r) == 1


# Equal shares of a multiple of 8 steps, rows whole KiB apart (us, tiles -> in step -> spread): 125 -> 203 -> 124,
# 164 -> 217 -> 127, 130 -> 197 -> 117, 140 -> 171 -> 114.
@pytest.mark.parametrize("m,n,r", [(65536, 4096, 128), (32768, 8192, 192), (32768, 8192, 64), (130995, 2048, 64)])
def test_up_projection_spreads_workgroups_that_would_store_in_step(m, n, r):
    assert up(m, n, r) == 2


@pytest.mark.parametrize("m,n,r", [(65536 + 256, 4096, 128), (65536, 4096 + 64, 128), (32768, 3072, 128)])
def test_up_projection_leaves_other_shares_in_order(m, n, r):
    assert up(m, n, r) == 1


def rotate_lowrank(m, k, r):
    return _native.library().hf_route(_native.ROUTE_ROTATE_LOWRANK, m, 1, k, r)


# Each side of each line: 128 rows, 192 at up to 7 tiles of 1024, then 3.5 rounds (up to 5 tiles) or 2 of the workgroups
# that the CUs hold at once, while the projection alone would run by rows; up to 14 tiles.
@pytest.mark.parametrize("m,k,r,one", [
    (1, 3072, 64, 1), (128, 14336, 64, 1), (128, 14352, 64, 0), (129, 14336, 16, 0), (192, 7168, 64, 1),
    (192, 8192, 64, 0), (193, 8192, 8, 1), (384, 3072, 64, 1), (384, 3072, 72, 0), (298, 5120, 40, 1), (299, 5120, 40, 0),
    (204, 7168, 32, 1), (205, 7168, 32, 0), (332, 5120, 8, 1), (333, 5120, 8, 0), (385, 1024, 8, 0), (64, 5120, 0, 0),
])
def test_rotation_and_projection_in_one_launch(m, k, r, one):
    assert rotate_lowrank(m, k, r) == one


# One row of the 256 x 128 tiles and more than 128 MiB (26214.4 rows at K=5120), where those tiles run at all.
@pytest.mark.parametrize("m,k,n,streamed", [
    (256, 5120, 26216, 1), (256, 5120, 26208, 0), (257, 5120, 26216, 0), (129, 5120, 26216, 1), (128, 5120, 26216, 0),
    (256, 8192, 16392, 1), (256, 8192, 16384, 0), (256, 5120, 32768, 1), (256, 5120, 32776, 0),
])
def test_streamed_weight(m, k, n, streamed):
    assert _native.library().hf_route(_native.ROUTE_STREAM_WEIGHT, m, n, k, 32) == streamed
