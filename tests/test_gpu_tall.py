"""Products of more than 128 rows in tiles of the package's own (csrc/gemm_tall.hip, csrc/tile_loop.hpp) against float64, at the
edges of tiles, of K's stages and slices, and of the rule that chooses them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TILES = [(256, 256), (224, 256), (192, 256), (160, 256), (256, 128), (192, 128), (128, 128)]


@pytest.fixture(scope="module")
def ops():
    from torchless_rs_amd.kernels import ops as o
    o.lib()
    return o


def operands(M, N, K, apart=0):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a, w = torch.randn(M, K, generator=g, device=DEV).bfloat16(), torch.randn(N, K + apart, generator=g, device=DEV).bfloat16()[:, :K]
    return a, w, a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()


def bound(K, size):
    """A sum of K products in 32 bits, in any order, lies within K 2^-24 of the sum of the products' sizes; the worst of M N
    chains is a few dozen standard errors of a walk, sqrt(K) 2^-24 of it, below 8."""
    return 8 * K ** 0.5 * 2.0 ** -24 * size + 1e-30


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,apart", [(1, 4, 8, 0), (129, 64, 64, 8), (257, 772, 136, 0), (300, 260, 640, 0), (513, 128, 1096, 16)])
def test_tiles_and_slices(ops, tile, M, N, K, apart):
    a, w, want, size = operands(M, N, K, apart)
    stages = -(-K // 64)
    for S in (1, 2, 3, 5):
        if (S - 1) * -(-stages // S) >= stages:
            continue
        plan = ops.TallPlan(*tile, S, stagger=S == 1 and K % 64 == 0)
        out = torch.full((S, M, N), float("nan"), device=DEV)
        ops.gemm_tall_bf16(a, w, out if S > 1 else out[0], plan)
        assert bool(((out.double().sum(0) - want).abs() <= bound(K, size)).all())
    x = torch.randn(M, N, device=DEV)
    total = x.double() + want
    ops.gemm_tall_bf16(a, w, x, ops.TallPlan(*tile), accumulate=True)
    assert bool(((x.double() - total).abs() <= bound(K, size) + 2.0 ** -23 * total.abs()).all())


@pytest.mark.parametrize("tile", [(256, 256), (160, 256), (256, 128), (192, 128)])
@pytest.mark.parametrize("M,K,S", [(226, 4096, 8), (513, 640, 3), (300, 1344, 4)])
def test_a_slice_adds_its_stages_in_their_order(ops, tile, M, K, S):
    """A slice's sums have the bits of the product of its columns alone, however the rule would go through a K that is not cut; and stages in
    turn are refused where it is."""
    N, stages = 772, -(-K // 64)
    a, w, _, _ = operands(M, N, K)
    out = torch.full((S, M, N), float("nan"), device=DEV)
    ops.gemm_tall_bf16(a, w, out, ops.TallPlan(*tile, S))
    per = -(-stages // S)
    for s in range(S):
        k = slice(64 * per * s, min(K, 64 * per * (s + 1)))
        one = torch.empty(M, N, device=DEV)
        ops.gemm_tall_bf16(a[:, k].contiguous(), w[:, k], one, ops.TallPlan(*tile))
        assert torch.equal(out[s], one), s
    with pytest.raises(ops.KernelError, match="uncut"):
        ops.gemm_tall_bf16(a, w, out, ops.TallPlan(*tile, S, stagger=True))


@pytest.mark.parametrize("tile", [t for t in TILES if t[1] == 256])
@pytest.mark.parametrize("parts", [2, 4])
@pytest.mark.parametrize("M,N", [(17, 4100), (257, 2176), (1000, 772), (1025, 640)])
def test_last_tiles_in_parts(ops, tile, parts, M, N):
    """Whole tiles and parts write every sum once: halves by channels, quarters by rows too, the last of either cut short."""
    K = 192
    a, w, want, size = operands(M, N, K)
    tiles = -(-M // tile[0]) * -(-N // 256)
    for whole in (0, 8, tiles // 8 * 8):
        if whole <= tiles:
            x = torch.ones(M, N, device=DEV)
            ops.gemm_tall_bf16(a, w, x, ops.TallPlan(*tile, whole=whole, parts=parts), accumulate=True)
            assert bool(((x.double() - 1.0 - want).abs() <= bound(K, size) + 2.0 ** -23 * (want.abs() + 1.0)).all()), whole


@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "relu", ("swish_clamped", {"alpha": 1.702, "limit": 7.0, "shift": 1.0})])
@pytest.mark.parametrize("M,I,K,plan", [(129, 32, 64, (192, 128)), (300, 96, 264, (160, 256)), (520, 672, 128, (256, 256, 1, False, 8, 2)),
                                        (520, 672, 128, (192, 256, 1, False, 8, 4))])
def test_paired(ops, act, M, I, K, plan):
    """act(gate) * up of the sums, rounded to bfloat16 once (up to 2^-8 of itself); the sums' error and the exponential's, (8 + 1.5 |g|) 2^-24
    of the value, pass through functions whose slope is near 1 or below, times the other factor: 1e-5 of the sums' sizes covers both."""
    a, w, p, size = operands(M, 2 * I, K)
    a, p, size = a * K ** -0.5, p * K ** -0.5, size * K ** -0.5
    p = a.double() @ w.double().t()
    gate, up = p.view(M, I // 32, 2, 32).unbind(2)
    gate, up = gate.reshape(M, I), up.reshape(M, I)
    name = act if isinstance(act, str) else act[0]
    if name == "silu":
        want = torch.nn.functional.silu(gate) * up
    elif name == "gelu_tanh":
        want = torch.nn.functional.gelu(gate, approximate="tanh") * up
    elif name == "relu":
        want = torch.relu(gate) * up
    else:
        gate = gate.clamp(max=7.0)
        want = gate * torch.sigmoid(1.702 * gate) * (up.clamp(-7.0, 7.0) + 1.0)
    out = torch.full((M, I), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.gemm_tall_bf16(a, w, out, ops.TallPlan(*plan), silu_pair=True, pair_act=act)
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * (1.0 + size.max())).all())


def test_plans_fit_what_they_are_for(ops):
    """Every plan of the rule can be launched: K's slices all have stages, whole tiles are rounds of workgroups, partial sums are
    made only where they are welcome, nothing is planned up to MID_ROWS rows or for sizes the tiles do not take."""
    for N, K in ((28672, 4096), (4096, 14336), (5120, 14336), (18560, 4096), (64, 64), (12288, 4104), (4096, 4096), (2048, 8192), (65536, 16384)):
        for M in list(range(129, 700, 37)) + [1024, 1999, 2048, 4097, 16384]:
            for kind, sums in (("store", False), ("add", False), ("add", True), ("pair", False), ("act", False)):
                p = ops.tall_plan(M, N, K, 256, kind, sums)
                if p is None:
                    continue
                stages = -(-K // 64)
                assert (p.rows, p.channels) in TILES and (p.n_split == 1 or (sums and kind == "add"))
                assert (p.n_split - 1) * -(-stages // p.n_split) < stages and not (p.stagger and (K % 64 or p.n_split > 1 or p.parts))
                assert p.parts in (0, 2, 4) and p.whole % 256 == 0 and (p.parts or not p.whole)
    assert ops.tall_plan(128, 28672, 4096, 256, "pair") is None and ops.tall_plan(2048, 28672, 4100, 256, "pair") is None
    assert ops.tall_plan(2048, 28704, 4096, 256, "pair") is None and ops.tall_plan(2048, 4098, 4096, 256, "add") is None


def test_what_the_tiles_do_not_take_is_refused(ops):
    a, w = torch.zeros(200, 128, dtype=torch.bfloat16, device=DEV), torch.zeros(256, 128, dtype=torch.bfloat16, device=DEV)
    out = torch.zeros(200, 256, device=DEV)
    with pytest.raises(ops.KernelError, match="no tiles"):
        ops.gemm_tall_bf16(a, w, out, ops.TallPlan(64, 256))
    with pytest.raises(ops.KernelError, match="without a stage"):
        ops.gemm_tall_bf16(a, w, torch.zeros(3, 200, 256, device=DEV), ops.TallPlan(256, 256, 3))
    with pytest.raises(ops.KernelError, match="multiple of 8"):
        ops.gemm_tall_bf16(a, w, out, ops.TallPlan(256, 256, whole=1, parts=2))
    with pytest.raises(ops.KernelError, match="bfloat16 rows"):
        ops.gemm_tall_bf16(a, torch.zeros(128, 256, dtype=torch.bfloat16, device=DEV).t(), out, ops.TallPlan(256, 256))


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("act", ["relu2", "relu", "xielu", "gated", "plain_gated"])
@pytest.mark.parametrize("M,I,K,plan", [(129, 32, 64, (192, 128)), (300, 160, 264, (160, 256)), (520, 672, 128, (256, 256, 1, False, 8, 2)),
                                        (520, 672, 128, (192, 256, 1, False, 8, 4)), (257, 96, 128, (256, 128, 1, True))])
def test_an_experts_activation(ops, act, M, I, K, plan, weighted):
    """The activation on the sums, rounded to bfloat16 once, as in `test_paired`; gate and up rows lie apart.  The square's slope is twice
    its root: 1e-5 of the sums' sizes times the largest of them covers it."""
    gated = "gated" in act
    a, w, p, size = operands(M, 2 * I if gated else I, K)
    a = a * K ** -0.5
    p = a.double() @ w.double().t()
    top = float(p.abs().max())
    factor = torch.rand(M, device=DEV) if weighted else None
    kw = {}
    if gated:
        limit, alpha, shift = (0.75, 1.702, 1.0) if act == "gated" else (float("inf"), 1.0, 0.0)
        kw["terms"] = ops.GateTerms(3.0, alpha, shift, limit, True)
        g, u = p[:, :I].clamp(max=limit), p[:, I:].clamp(-limit, limit)
        want = g * torch.sigmoid(alpha * g) * (u + shift)
    else:
        kw["activation"] = act
        want = torch.relu(p) ** 2 if act == "relu2" else torch.relu(p)
        if act == "xielu":
            kw["constants"] = {"a": 0.8, "b": 0.9}
            want = torch.where(p > 0, 0.8 * p * p + 0.5 * p, 0.9 * (torch.expm1(p) - p) + 0.5 * p)
    if weighted:
        want = want * factor.double()[:, None]
    out = torch.full((M, I), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.gemm_tall_act(a, w, out, ops.TallPlan(*plan), row_weight=factor, **kw)
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * (1.0 + top) * (1.0 + top)).all())


@pytest.mark.parametrize("M,I,K,plan", [(513, 32768, 16384, (256, 256)), (130, 131072, 16384, (192, 128)), (130, 131072, 16384, (224, 256, 1, False, 512, 2))])
def test_gate_and_up_rows_that_lie_gigabytes_apart(ops, M, I, K, plan):
    """2^30 and 2^32 bytes between a gate row and its up row; the bound is `test_an_experts_activation`'s, checked at the ends and in the middle."""
    g = torch.Generator(device=DEV).manual_seed(I)
    a, w = (torch.randn(M, K, generator=g, device=DEV) * K ** -0.5).bfloat16(), torch.randn(2 * I, K, generator=g, device=DEV, dtype=torch.bfloat16)
    out = torch.full((M, I), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.gemm_tall_act(a, w, out, ops.TallPlan(*plan), terms=ops.GateTerms(3.0, 1.0, 0.0, float("inf"), True))
    for c in (0, I // 2 - 96, I - 96):
        p, u = a.double() @ w[c:c + 96].double().t(), a.double() @ w[I + c:I + c + 96].double().t()
        want = torch.nn.functional.silu(p) * u
        top = float(torch.maximum(p.abs(), u.abs()).max())
        assert bool(((out[:, c:c + 96].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * (1.0 + top) * (1.0 + top)).all())
    assert bool(torch.isfinite(out.float()).all())


@pytest.mark.parametrize("limit,alpha,shift", [(7.0, 1.702, 1.0), (float("inf"), 1.0, 0.0)])
@pytest.mark.parametrize("M,I,K,plan", [(129, 160, 136, (192, 128)), (520, 672, 128, (256, 256, 1, False, 8, 2)), (520, 672, 128, (192, 256, 1, False, 8, 4))])
def test_a_gated_epilogue_has_the_bits_of_the_activation(ops, M, I, K, plan, limit, alpha, shift):
    """As the activation's own kernel makes of the same sums stored, far from 0 too (pre-activations reach 20)."""
    a, w, _, _ = operands(M, 2 * I, K)
    a = (a.float() * 4.0 * K ** -0.5).bfloat16()
    terms, sw = ops.GateTerms(limit, alpha, shift, None, False), torch.rand(M, device=DEV)
    u, want, out = torch.empty(M, 2 * I, device=DEV), *(torch.empty(M, I, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.gemm_tall_bf16(a, w.contiguous(), u, ops.TallPlan(*plan[:2]))
    ops.expert_gated_act(u, None, 0, 0, I, terms, want, sw)
    ops.gemm_tall_act(a, w.contiguous(), out, ops.TallPlan(*plan), terms=terms, row_weight=sw)
    assert torch.equal(out, want)


def test_a_product_stored_in_bfloat16_is_the_librarys(ops):
    """Products above MID_ROWS rows may be stored in bfloat16, also where float32 ones go in tiles: each sum, within `bound`, rounded
    once to 8 bits."""
    M, N, K = 1000, 14340, 2048
    assert ops.tall_plan(M, N, K, 256, "store") is not None
    a, w, want, size = operands(M, N, K)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.gemm(a, w.contiguous(), out)
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 * bound(K, size)).all())


def test_the_paired_silu_far_from_zero(ops):
    """Gates down to -100 on sums that are exact (one product of each row counts): the exponential and reciprocal instructions are within
    (8 + 1.5 |g|) 2^-24 of the value, whose rounding to 8 bits, half a unit of the last, is up to 2^-8 of itself; below -87 the value is under 2^-119 of the up sum and
    may be 0."""
    M, I, K = 256, 512, 64
    g = torch.Generator(device=DEV).manual_seed(3)
    a = torch.zeros(M, K, dtype=torch.bfloat16, device=DEV)
    a[torch.arange(M, device=DEV), torch.arange(M, device=DEV) % K] = 1.0
    gate = (torch.rand(I, K, generator=g, device=DEV) * 140.0 - 100.0).bfloat16()
    gate[:4] = torch.tensor([-20.0, -60.0, -87.0, -88.0], device=DEV)[:, None].bfloat16()
    up = torch.randn(I, K, generator=g, device=DEV).bfloat16()
    w = torch.stack([gate.view(I // 32, 32, K), up.view(I // 32, 32, K)], dim=1).reshape(2 * I, K).contiguous()
    out = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.gemm_tall_bf16(a, w, out, ops.TallPlan(256, 256), silu_pair=True)
    p, u = a.double() @ gate.double().t(), a.double() @ up.double().t()
    want = p / (1.0 + torch.exp(-p)) * u
    bound = (2.0 ** -8 + (8.0 + 1.5 * p.abs()) * 2.0 ** -24) * want.abs() + torch.where(p < -87.0, 2.0 ** -118 * u.abs(), 0.0)
    assert bool(((out.double() - want).abs() <= bound).all())
