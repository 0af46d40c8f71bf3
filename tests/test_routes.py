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


# Equal shares of a multiple of 8 steps, rows whole KiB apart (us, tiles -> in step -> spread): 125 -> 203 -> 124,
# 164 -> 217 -> 127, 130 -> 197 -> 117, 140 -> 171 -> 114.
@pytest.mark.parametrize("m,n,r", [(65536, 4096, 128), (32768, 8192, 192), (32768, 8192, 64), (130995, 2048, 64)])
def test_up_projection_spreads_workgroups_that_would_store_in_step(m, n, r):
    assert up(m, n, r) == 2


@pytest.mark.parametrize("m,n,r", [(65536 + 256, 4096, 128), (65536, 4096 + 64, 128), (32768, 3072, 128)])
def test_up_projection_leaves_other_shares_in_order(m, n, r):
    assert up(m, n, r) == 1
