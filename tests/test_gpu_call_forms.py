"""`Int8RotLinear.forward` over the forms an input can take: contiguous bf16 goes to the kernels as it is and the output
is allocated in its final shape, everything else is first made contiguous bf16 rows. All forms of the same values give
the same bits, the output's shape and dtype follow the input's, and what was refused stays refused."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
K, N = 512, 320


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.fail("no ROCm device visible")
    from hyperflow_h3_flash_amd import _native

    _native.library()


def make_layer(rank=32, bias=True, activation=None):
    from hyperflow_h3_flash_amd import Int8RotLinear

    gen = torch.Generator(device=DEV).manual_seed(3)
    layer = Int8RotLinear(K, N, 256, rank=rank, bias=bias, activation=activation).to(DEV)
    with torch.no_grad():
        layer.qweight.copy_(torch.randint(-127, 128, (N, K), device=DEV, dtype=torch.int8, generator=gen))
        layer.wscale.copy_(torch.rand(N, device=DEV, generator=gen) * 9e-3 + 1e-3)
        for p in (layer.down.weight, layer.up.weight) if rank else ():
            p.copy_(torch.randn(p.shape, device=DEV, generator=gen) * 0.02)
        if bias:
            layer.bias.copy_(torch.randn(N, device=DEV, generator=gen) * 0.01)
    return layer


FORMS = {
    "rows": lambda x: x,
    "leading dims": lambda x: x.reshape(2, 3, -1, K),
    "transposed view": lambda x: x.t().contiguous().t(),
    "row stride past K": lambda x: torch.cat([x, x], 1)[:, :K],
    "every second row": lambda x: torch.stack([x, x], 1).reshape(-1, K)[::2],
    "fp32": lambda x: x.float(),
    "fp32 view": lambda x: x.float().t().contiguous().t(),
}


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("rank,bias,activation", [(32, True, None), (0, False, "swiglu")])
def test_every_form_of_an_input_gives_the_same_bits(form, rank, bias, activation):
    layer = make_layer(rank, bias, activation)
    x = torch.randn(42, K, device=DEV, generator=torch.Generator(device=DEV).manual_seed(1)).to(torch.bfloat16)
    with torch.no_grad():
        want = layer(x)
        v = FORMS[form](x)
        got = layer(v)
        layer.keep_input = True  # the codes in tensors of their own, then shared
        kept, again = layer(v), layer(v)
        layer.keep_input = False
        assert torch.equal(layer(v), kept) and torch.equal(again, kept)
    assert got.shape == (*v.shape[:-1], want.shape[-1]) and got.dtype == v.dtype and got.is_contiguous()
    assert torch.equal(got.reshape(want.shape).to(torch.bfloat16), want) and torch.equal(got, kept)


def test_one_row_and_no_rows():
    layer = make_layer()
    x = torch.randn(K, device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        one = layer(x)
        assert one.shape == (N,) and torch.equal(one, layer(x[None])[0])
        assert layer(x[None][:0]).shape == (0, N) and layer(torch.empty(2, 0, K, device=DEV)).shape == (2, 0, N)


def test_refused_inputs_stay_refused():
    layer = make_layer()
    x = torch.randn(4, K, device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        with pytest.raises(RuntimeError):
            layer(x[:, : K // 2])  # as many elements as two whole rows, but not rows
        with pytest.raises(ValueError, match="ALIGNMENT"):
            layer(torch.randn(4 * K + 1, device=DEV).to(torch.bfloat16)[1:].reshape(4, K))
        for name in ("qweight", "wscale", "bias"):
            moved = make_layer()
            setattr(moved, name, torch.nn.Parameter(getattr(moved, name).cpu(), requires_grad=False))
            with pytest.raises(ValueError, match="expected cuda"):
                moved(x)
        for name in ("down", "up"):
            moved = make_layer()
            getattr(moved, name).cpu()
            with pytest.raises(ValueError, match="expected cuda"):
                moved(x)
