"""The low-rank up projection of many rows (u in registers, columns in steps of 64: `lowrank_up_rows_kernel`) against
the other up kernels on the same inputs, bit for bit (every up kernel adds the ranks in the same order), and sampled
rows against the oracle's exactly rounded sums.

A zero bias sends the same call to the other kernels: it adds +0 to sums that start from +0, so it changes no bit.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch
from golden_utils import within_fp32_sum_bound

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.fail("no ROCm device visible")
    from hyperflow_h3_flash_amd import _native

    _native.library()


# Steps of (256 rows, 64 columns), 512 workgroups: a share within one block of rows (N = 28672: 448 steps a block), and
# shares that cross into the next; ragged last row blocks (one row, less and more than a wave's 64 rows of it); every
# count of 64-rank chunks, full and with a partial last one; the fewest steps of the route at several widths. Way 2 (equal
# shares of a multiple of 8 steps): a share that is a part of a row block's columns, all of them, and several blocks.
@pytest.mark.parametrize("m,n,r,way", [(2048, 4096, 8, 1), (1793, 4096, 64, 1), (8192, 4096, 72, 1),
                                       (6017, 4096, 128, 1), (6200, 4096, 136, 1), (32513, 1024, 192, 1),
                                       (1100, 28672, 200, 1), (27905, 2112, 256, 1), (50000, 192, 64, 1),
                                       (32640, 2048, 200, 2), (131072, 512, 256, 2), (262100, 512, 64, 2)])
def test_up_rows_is_bitwise_the_other_kernels(oracle_lib, m, n, r, way):
    from hyperflow_h3_flash_amd import _native
    from hyperflow_h3_flash_amd.int8 import lowrank_up

    assert _native.library().hf_route(_native.ROUTE_UP_ROWS, m, n, 0, r) == way
    gen = torch.Generator(device=DEV).manual_seed(m + n + r)
    u = torch.randn(m, r, device=DEV, generator=gen).to(torch.bfloat16)
    up = (torch.randn(n, r, device=DEV, generator=gen) * 0.1).to(torch.bfloat16)
    print(f"lowrank_up rows M={m} N={n} r={r}", flush=True)
    y = lowrank_up(u, up)
    want = lowrank_up(u, up, torch.zeros(n, device=DEV, dtype=torch.bfloat16))
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    rows = np.unique(np.concatenate([[0, 63, 64, 255, 256], np.arange(m - 2, m)]))
    at = torch.from_numpy(rows).to(DEV)
    bits = lambda t: t.cpu().contiguous().view(torch.int16).numpy().view(np.uint16)  # noqa: E731
    u_rows, up_bits = bits(u[at]), bits(up)
    f32 = oracle_lib.bf16_to_f32
    # an fp32 sum of r products in any order, rounded once
    assert within_fp32_sum_bound(f32(bits(y[at])), f32(oracle_lib.lowrank_up(u_rows, up_bits)), f32(u_rows),
                                 f32(up_bits))


@pytest.mark.parametrize("n", [4096, 4095, 4090, 4040])
def test_up_rows_writes_only_its_columns(n):
    """A padded output (row stride past N, whole lines) keeps its padding, also with a last step of fewer than 64
    columns, whole 8-column chunks or not; an output of ragged lines takes the other kernels: the same bits."""
    import ctypes

    from hyperflow_h3_flash_amd import _native

    m, ld, r = 2100, 4160, 64
    u = torch.randn(m, r, device=DEV).to(torch.bfloat16)
    up = torch.randn(n, r, device=DEV).to(torch.bfloat16)
    y = torch.full((m, ld), 7.0, device=DEV, dtype=torch.bfloat16)
    other = torch.full((m, ld + 8), 7.0, device=DEV, dtype=torch.bfloat16)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    lib = _native.library()
    assert lib.hf_route(_native.ROUTE_UP_ROWS, m, n, 0, r) == 1
    for out in (y, other):
        assert lib.hf_lowrank_up(u.data_ptr(), r, up.data_ptr(), r, r, None, out.data_ptr(), out.stride(0), m, n,
                                 stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(y[:, :n], other[:, :n])
    assert bool((y[:, n:] == 7.0).all()) and bool((other[:, n:] == 7.0).all())


def _padded(t, rows, cols):
    """A view of t's values inside a larger tensor of NaN (rows past the last and columns past each row's end)."""
    big = torch.full((t.shape[0] + rows, t.shape[1] + cols), float("nan"), device=DEV, dtype=torch.bfloat16)
    view = big[: t.shape[0], : t.shape[1]]
    view.copy_(t)
    return view


# Ranks that end inside a 64-rank chunk, or with it, rows that go on past the rank, and a ragged last row block: what lies
# past the rank, past the last row of u and past the last row of up is NaN and must not be read into the sums.
@pytest.mark.parametrize("m,n,r,pad_u,pad_up,way", [(2100, 4096, 8, 8, 56, 1), (2100, 4096, 64, 64, 8, 1),
                                                    (8191, 4096, 72, 8, 8, 1), (6017, 4096, 128, 72, 16, 1),
                                                    (6200, 4032, 136, 120, 8, 1), (7001, 4096, 192, 8, 64, 1),
                                                    (7001, 4096, 200, 56, 8, 1), (7001, 4096, 256, 8, 8, 1),
                                                    (32600, 2048, 200, 24, 40, 2)])
def test_up_rows_takes_rows_that_go_on_past_the_rank(m, n, r, pad_u, pad_up, way):
    import ctypes

    from hyperflow_h3_flash_amd import _native

    lib = _native.library()
    assert lib.hf_route(_native.ROUTE_UP_ROWS, m, n, 0, r) == way
    gen = torch.Generator(device=DEV).manual_seed(m + n + r)
    dense_u = torch.randn(m, r, device=DEV, generator=gen).to(torch.bfloat16)
    dense_up = (torch.randn(n, r, device=DEV, generator=gen) * 0.1).to(torch.bfloat16)
    u, up = _padded(dense_u, 64, pad_u), _padded(dense_up, 64, pad_up)
    zero = torch.zeros(n, device=DEV, dtype=torch.bfloat16)  # sends the call to the other kernels
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    print(f"lowrank_up rows padded M={m} N={n} r={r} ldu={u.stride(0)} ld_up={up.stride(0)}", flush=True)
    got = torch.empty(m, n, device=DEV, dtype=torch.bfloat16)
    want = torch.empty(m, n, device=DEV, dtype=torch.bfloat16)
    for out, a, b, bias in ((got, u, up, None), (want, dense_u, dense_up, zero.data_ptr())):
        assert lib.hf_lowrank_up(a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), r, bias, out.data_ptr(), n, m, n,
                                 stream) == 0
    torch.cuda.synchronize()
    assert not bool(torch.isnan(want).any())
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("m,n,r", [(2100, 4096, 64), (7001, 4096, 200)])
def test_up_rows_carries_infinities_and_nan(m, n, r):
    """Rows of u and of up with infinities, NaN, the largest values and -0: NaN where the other kernels give NaN, their
    bits elsewhere; rows without them are not touched."""
    from hyperflow_h3_flash_amd import _native
    from hyperflow_h3_flash_amd.int8 import lowrank_up

    assert _native.library().hf_route(_native.ROUTE_UP_ROWS, m, n, 0, r) == 1
    gen = torch.Generator(device=DEV).manual_seed(r)
    u = torch.randn(m, r, device=DEV, generator=gen).to(torch.bfloat16)
    up = (torch.randn(n, r, device=DEV, generator=gen) * 0.1).to(torch.bfloat16)
    big = torch.finfo(torch.bfloat16).max
    special = torch.tensor([float("inf"), -float("inf"), float("nan"), big, -big, 0.0, -0.0], device=DEV)
    for t, rows in ((u, [0, 63, 64, 255, 256, 1000, m - 1]), (up, [0, 31, 32, 63, 64, 2000, n - 1])):
        for i, row in enumerate(rows):
            t[row, (7 * i) % r] = special[i]
            t[row, r - 1 - i] = special[-1 - i]
    got = lowrank_up(u, up)
    want = lowrank_up(u, up, torch.zeros(n, device=DEV, dtype=torch.bfloat16))
    nan = torch.isnan(want)
    assert bool(nan.any()) and bool(torch.isinf(want).any()) and not bool(nan.all())
    assert torch.equal(torch.isnan(got), nan)
    assert torch.equal(got.view(torch.int16)[~nan], want.view(torch.int16)[~nan])
    # the largest values overflow to infinities of both signs too: rows of ordinary values only
    clean_rows, clean_cols = (u.abs() < 100).all(1), (up.abs() < 100).all(1)
    assert not bool(nan[clean_rows][:, clean_cols].any())
