"""Layers of 193 to 384 rows: the rotation and the row-wise low-rank projection in one launch where their workgroups
fit few rounds of the CUs, apart beyond; both give the bits of the composed calls (rotate_quant, lowrank_down,
int8_matmul)."""

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


# Both sides of the line: 3.5 rounds up to 5 tiles of 1024, 2 rounds past that (256 CUs holding 4 workgroups of 3 tiles,
# 2 of 5 to 7); a partial last tile, a rank that is no multiple of 8 workgroup ranks, ranks past 64, another group.
@pytest.mark.parametrize("m,k,r,group,one", [(384, 3072, 64, 256, 1), (384, 3072, 72, 64, 0), (384, 3072, 128, 256, 0),
                                             (298, 5120, 40, 256, 1), (299, 5120, 40, 256, 0), (193, 4864, 64, 256, 1),
                                             (204, 7168, 32, 1024, 1), (205, 7168, 32, 1024, 0), (193, 7168, 32, 16, 1)])
def test_row_launch_is_the_composed_layer(m, k, r, group, one):
    from hyperflow_h3_flash_amd import Int8RotLinear, _native
    from hyperflow_h3_flash_amd.int8 import int8_matmul, lowrank_down, rotate_quant

    assert _native.library().hf_route(_native.ROUTE_ROTATE_LOWRANK, m, 256, k, r) == one
    gen = torch.Generator(device=DEV).manual_seed(m + k + r)
    n = 256
    layer = Int8RotLinear(k, n, group, rank=r).to(DEV)
    x = torch.randn(m, k, device=DEV, generator=gen).to(torch.bfloat16)
    with torch.no_grad():
        layer.qweight.copy_(torch.randint(-127, 128, (n, k), device=DEV, dtype=torch.int8, generator=gen))
        layer.wscale.copy_(torch.rand(n, device=DEV, generator=gen) * 9e-3 + 1e-3)
        layer.down.weight.copy_(torch.randn(r, k, device=DEV, generator=gen) * 0.02)
        layer.up.weight.copy_(torch.randn(n, r, device=DEV, generator=gen) * 0.02)
        print(f"row launch M={m} K={k} r={r} G={group}", flush=True)
        got = layer(x)
        q, s = rotate_quant(x, group)
        want = int8_matmul(q, layer.qweight, s, layer.wscale, u=lowrank_down(x, layer.down.weight), up=layer.up.weight)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
