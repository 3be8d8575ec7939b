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
@pytest.mark.parametrize("E,groups,keep,top,W", [(15, 0, 0, 2, 252), (16, 4, 2, 4, 512), (33, 11, 5, 9, 260), (64, 8, 1, 8, 132),
                                                 (64, 0, 0, 64, 4), (64, 64, 7, 7, 68), (65, 0, 0, 3, 64)])
def test_a_step_of_many_rows_routes_as_its_rows_do_in_small_steps(ops, dtype, E, groups, keep, top, W):
    """Rows by fours, with a last four that is not whole, give the bits of the kernel of a workgroup a row: scores of both kinds, ties (equal
    rows of the router), NaN and infinite rows, corrections, two largest, normalised weights, a shared expert's row."""
    n = 769
    g = torch.Generator(device=DEV).manual_seed(E * W + top)
    h = torch.randn(n, W, generator=g, device=DEV).to(dtype)
    h[3, 0], h[7, 0], h[9] = float("nan"), float("inf"), 0.0
    for shared in (False, True):
        wr = torch.randn(E + shared, W, generator=g, device=DEV) * W ** -0.5
        wr[E // 2] = wr[0]
        more = {"correction": torch.randn(E, generator=g, device=DEV), "bias": torch.randn(E, generator=g, device=DEV)}
        for logistic in (False, True):
            for kw in ({}, {"two_largest": True, "normalise_eps": 1e-6, **more}):
                def run(rows, at):
                    w = torch.full((rows.shape[0], E), -1.0, device=DEV)
                    c = torch.full((rows.shape[0], top), -1, dtype=torch.int32, device=DEV)
                    sw = torch.full((rows.shape[0],), -1.0, device=DEV) if shared else None
                    ops.route(rows, wr, groups, keep, top, w, c, logistic=logistic, shared_weight=sw, **kw)
                    return [t.view(torch.int32) for t in (w, c) + ((sw,) if shared else ())]
                many = run(h, 0)
                few = [torch.cat(t) for t in zip(*(run(h[i:i + 250], i) for i in range(0, n, 250)))]
                for a, b in zip(many, few):
                    assert torch.equal(a, b)


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
