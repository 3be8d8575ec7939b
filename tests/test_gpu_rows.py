"""Kernels that have a form of their own for steps of many rows: the router (csrc/experts.hip), heads before the attention
(csrc/attention_heads.hip), the activation of a stored product (csrc/elementwise.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from torchless_rs_amd.kernels import ops as o
    o.lib()
    return o


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,I", [(1, 1), (2, 1023), (2, 1024), (3, 1028), (2, 8192), (1, 1048580), (129, 2050)])
def test_the_activation_of_a_stored_product(ops, dtype, n, I):
    gu = torch.randn(n, 2 * I, generator=torch.Generator(device=DEV).manual_seed(I), device=DEV)
    out = torch.full((n, I), float("nan"), dtype=dtype, device=DEV)
    ops.act_mul(gu, out)
    gate, up = gu.double().split(I, dim=1)
    want = gate / (1.0 + torch.exp(-gate)) * up
    # the exponential, the division and two products: a few units of 2^-24; bfloat16 rounds the result once
    assert bool(((out.double() - want).abs() <= want.abs() * (1e-6 if dtype == torch.float32 else 2.0 ** -8) + 1e-30).all())
