"""The 256 x 128 tiles with the weight streamed past the caches (one row of tiles, a weight of more than 128 MiB): the
outputs of the same rows inside a taller product, whose tiles load the weight the ordinary way, bit for bit."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.fail("no ROCm device visible")
    from hyperflow_h3_flash_amd import _native

    _native.library()


# The fewest and the most rows of the route, ragged columns (the last tile 16 and 120 wide), K past a whole stage.
@pytest.mark.parametrize("m,k,n,r,act", [(129, 5136, 30736, 0, None), (200, 5376, 28280, 24, "gelu_tanh"),
                                         (256, 5120, 30720, 64, None)])
def test_streamed_weight_gives_the_bits_of_the_taller_product(m, k, n, r, act):
    from hyperflow_h3_flash_amd import _native
    from hyperflow_h3_flash_amd.int8 import int8_matmul

    route = _native.library().hf_route
    assert route(_native.ROUTE_STREAM_WEIGHT, m, n, k, r) == 1 and route(_native.ROUTE_STREAM_WEIGHT, 600, n, k, r) == 0
    gen = torch.Generator(device=DEV).manual_seed(m)
    rows = 600
    q = torch.randint(-127, 128, (rows, k), device=DEV, dtype=torch.int8, generator=gen)
    w = torch.randint(-127, 128, (n, k), device=DEV, dtype=torch.int8, generator=gen)
    sx = torch.rand(rows, device=DEV, generator=gen) * 0.01 + 0.001
    sw = torch.rand(n, device=DEV, generator=gen) * 0.01 + 0.001
    u = torch.randn(rows, r, device=DEV, generator=gen).to(torch.bfloat16) if r else None
    up = (torch.randn(n, r, device=DEV, generator=gen) * 0.1).to(torch.bfloat16) if r else None
    bias = torch.randn(n, device=DEV, generator=gen).to(torch.bfloat16)
    print(f"streamed weight M={m} K={k} N={n} r={r} {act}", flush=True)
    got = int8_matmul(q[:m], w, sx[:m], sw, u=u[:m] if r else None, up=up, bias=bias, activation=act)
    want = int8_matmul(q, w, sx, sw, u=u, up=up, bias=bias, activation=act)
    assert torch.equal(got.view(torch.int16), want[:m].view(torch.int16))
