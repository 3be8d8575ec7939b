"""Products over each expert's own rows (csrc/gemm_grouped.hip) against float64, at the edges of its tiles: 224 positions,
256 channels (128 gated ones), stages of 64 k."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from torchless_rs_amd.kernels import ops as o
    o.lib()
    return o


def grouped(ops, chosen, E):
    n, top = chosen.shape
    off = torch.empty(E + 1, dtype=torch.int32, device=DEV)
    order, place = (torch.empty(n * top, dtype=torch.int32, device=DEV) for _ in range(2))
    ops.group_pairs(chosen, E, off, order, place)
    return off, order, place


def choose(n, E, top, seed, crowded):
    """`crowded`: a choice of every row lies with expert E - 1, and some experts have no row at all."""
    g = torch.Generator().manual_seed(seed)
    score = torch.rand(n, E, generator=g)
    if crowded:
        score[:, E - 1] += 2.0
        score[:, : E // 3] -= 2.0
    return score.topk(top).indices.int().to(DEV).contiguous()


@pytest.mark.parametrize("n,E,top,crowded", [(1, 1, 1, False), (7, 5, 3, True), (64, 16, 4, False), (500, 130, 2, True), (1025, 16, 4, True),
                                             (3000, 1024, 8, False)])
def test_group_pairs(ops, n, E, top, crowded):
    chosen = choose(n, E, top, n + E, crowded)
    off, order, place = grouped(ops, chosen, E)
    flat = chosen.view(-1).long()
    want = torch.argsort(flat, stable=True)
    assert torch.equal(order.long(), want)
    assert torch.equal(place.long()[want], torch.arange(n * top, device=DEV))
    assert torch.equal(off.long(), torch.cat([torch.zeros(1, dtype=torch.long, device=DEV), torch.bincount(flat, minlength=E).cumsum(0)]))


def test_pairs_of_numbers_that_are_no_experts_have_places(ops):
    """What goes by `order` and `place` stays in its buffers whatever the choice holds."""
    chosen = choose(300, 6, 3, 5, False)
    chosen[7, 1], chosen[8, 0], chosen[299, 2], chosen[0, 0] = -1, 6, 2 ** 31 - 1, -2 ** 31
    off, order, place = (torch.full((s,), -9, dtype=torch.int32, device=DEV) for s in (7, 900, 900))
    ops.group_pairs(chosen, 6, off, order, place)
    flat = chosen.clamp(0, 5).view(-1).long()
    want = torch.argsort(flat, stable=True)
    assert torch.equal(order.long(), want) and torch.equal(place.long()[want], torch.arange(900, device=DEV))
    assert off.tolist() == [0] + flat.bincount(minlength=6).cumsum(0).tolist()


CASES = [  # n, H, E, top, ff, shared, gated, on_input, crowded
    (1, 64, 4, 2, 64, 64, False, False, False), (33, 72, 6, 2, 40, 24, True, False, True), (160, 128, 2, 1, 256, 512, False, False, False),
    (161, 200, 3, 2, 264, 600, True, True, True), (320, 8, 5, 4, 8, 64, False, False, True), (700, 256, 16, 4, 136, 0, True, True, False),
    (1300, 192, 4, 2, 520, 720, False, False, True), (400, 320, 70, 3, 128, 192, True, False, True)]


@pytest.mark.parametrize("n,H,E,top,ff,shared,gated,on_input,crowded", CASES)
def test_experts_over_their_own_rows(ops, n, H, E, top, ff, shared, gated, on_input, crowded):
    """Both products and the sum over a row's experts.  The hidden activations are rounded to bfloat16 once (2^-9 of
    themselves, and a unit more for the float sums below it); the second product and the sum are float sums of K = ff and
    of `top` terms: at most (ff + top) 2^-24 of the sum of their terms' sizes."""
    g = torch.Generator(device=DEV).manual_seed(n + H)
    wide, slices = (2 if gated else 1), ops.shared_slices(ff, shared)
    sw = torch.rand(n, generator=g, device=DEV) + 0.5
    up = (torch.randn(wide * (E * ff + shared), H, generator=g, device=DEV) * H ** -0.5).bfloat16()
    down = (torch.randn(H, E * ff + shared, generator=g, device=DEV) * ff ** -0.5).bfloat16()
    y = torch.randn(n, H, generator=g, device=DEV).bfloat16()
    chosen = choose(n, E, top, 3 * n, crowded)
    weights = torch.rand(n, E, generator=g, device=DEV) + 0.1
    off, order, place = grouped(ops, chosen, E)
    terms = ops.GateTerms(1.5, 1.702, 1.0, 0.75, on_input) if gated else None
    act = {"terms": terms} if gated else {"activation": "relu2" if n % 2 else "relu"}

    def hidden(rows, w, s, limit):
        p = rows.double() @ w.double().T
        if not gated:
            return torch.relu(p) ** (2 if n % 2 else 1) * s
        a, u = p[:, : p.shape[1] // 2], p[:, p.shape[1] // 2:]
        if on_input:
            a, u = a * s, u * s
        a, u = a.clamp(max=limit), u.clamp(-limit, limit)
        return a * torch.sigmoid(1.702 * a) * (u + 1.0) * (1.0 if on_input else s)

    assert slices == -(-shared // ff) and slices <= ops.MOST_SLICES
    h = torch.zeros(n * (top + slices), ff, dtype=torch.bfloat16, device=DEV)
    ops.grouped_up(y, up, ff, shared, slices, off, order, top, weights, h, shared_weight=sw, **act)
    want = torch.zeros(n * (top + slices), ff, dtype=torch.float64, device=DEV)
    z_want, z_size = (torch.zeros(n * (top + slices), H, dtype=torch.float64, device=DEV) for _ in range(2))
    bounds = off.tolist()
    for e in range(E):
        at = slice(bounds[e], bounds[e + 1])
        rows = order[at].long() // top
        want[at] = hidden(y[rows], up[wide * e * ff: wide * (e + 1) * ff], weights[rows, e: e + 1].double(), 1.5)
        d = down[:, e * ff: (e + 1) * ff].double()
        z_want[at], z_size[at] = h[at].double() @ d.T, h[at].double().abs() @ d.abs().T
    if slices:                                               # what every row uses, cut in slices
        ones = torch.ones(n, 1, dtype=torch.float64, device=DEV)
        whole = hidden(y, up[wide * E * ff:], ones, 0.75) * sw[:, None].double()
        for j in range(slices):
            part = whole[:, j * ff: (j + 1) * ff]
            at, m = slice(n * (top + j), n * (top + j + 1)), part.shape[1]
            want[at, :m] = part
            d = down[:, E * ff + j * ff: E * ff + j * ff + m].double()
            z_want[at], z_size[at] = h[at, :m].double() @ d.T, h[at, :m].double().abs() @ d.abs().T
    assert float(((h.double() - want).abs() - want.abs() * 2.0 ** -8).max()) < 1e-4 * float(want.abs().max())
    z = torch.empty(n * (top + slices), H, device=DEV)
    ops.grouped_down(h, down, E, shared, slices, top, off, z)
    assert bool(((z.double() - z_want).abs() <= (ff + 8) * 2.0 ** -24 * z_size + 1e-30).all())
    out = torch.randn(n, H, generator=g, device=DEV)
    before = out.clone()
    ops.combine_pairs(z, place, out, True, slices)
    total = torch.zeros(n, H, device=DEV)
    for k in range(top):
        total += z[place.view(n, top)[:, k].long()]
    for j in range(slices):
        total += z[n * (top + j): n * (top + j + 1)]
    assert torch.equal(out, before + total)
    ops.combine_pairs(z, place, out, False, slices)
    assert torch.equal(out, total)


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("accumulate", [False, True])
def test_experts_of_sizes_that_are_no_multiples_of_eight(gated, accumulate):
    """Very many rows, an expert after the other by the library's products.  The hidden channels are rounded to bfloat16 once, the
    rest are sums of 32 bits."""
    from types import SimpleNamespace
    from torchless_rs_amd.parts import ffn_routed
    from torchless_rs_amd.parts.base import Workspace
    H, E, top, ff, shared, n = 64, 3, 2, 12, 10, 200
    part = ffn_routed.RoutedExperts(H, E, top, ff, shared_size=shared, gated=gated, activation="silu" if gated else "relu2")
    g = torch.Generator(device=DEV).manual_seed(7 + gated)
    part.load({k: (torch.randn(v.shape, generator=g, device=DEV) * v.shape[-1] ** -0.5).bfloat16() for k, v in part.weight_specs().items()},
              torch.bfloat16)
    ctx = SimpleNamespace(workspace=Workspace(torch.device(DEV)), dtype=torch.bfloat16, host={}, pending=None)
    y, x = torch.randn(n, H, generator=g, device=DEV).bfloat16(), torch.randn(n, H, generator=g, device=DEV)
    assert not part._serves(y) and part.many_rows(ctx, y)
    score = torch.softmax(y.double() @ part.router.double().T, dim=-1)
    picked = score.topk(top + 1)
    sure = picked.values[:, top - 1] > picked.values[:, top] * (1 + 1e-4)
    wt = torch.zeros_like(score).scatter_(1, picked.indices[:, :top], picked.values[:, :top])
    want = x.double().clone() if accumulate else torch.zeros(n, H, dtype=torch.float64, device=DEV)
    size = want.abs()
    up, down, at, wide = part.up.weight.double(), part.down.weight.double(), 0, 2 if gated else 1
    for e in range(E + 1):
        m = ff if e < E else shared
        z = y.double() @ up[wide * at: wide * (at + m)].T
        h = torch.nn.functional.silu(z[:, :m]) * z[:, m:] if gated else torch.relu(z) ** 2
        h = h * (wt[:, e: e + 1] if e < E else 1.0)
        want += h @ down[:, at: at + m].T
        size += h.abs() @ down[:, at: at + m].abs().T
        at += m
    if accumulate:
        part.forward(ctx, y, x)
    else:
        part.produce(ctx, y, x)
    # a hidden channel off by half a unit of its 8 bits, at most 2^-8 of itself, and the sums of 32 bits before and behind it
    assert bool(((x.double() - want).abs() <= (2.0 ** -8 + (H + 64) * 2.0 ** -24) * size + 1e-5)[sure].all())


def test_refused(ops):
    """Operands that the kernel does not take are an error, not a wrong result."""
    y = torch.zeros(4, 64, dtype=torch.bfloat16, device=DEV)
    up = torch.zeros(40, 64, dtype=torch.bfloat16, device=DEV)
    h = torch.empty(4, 24, dtype=torch.bfloat16, device=DEV)
    off, order = torch.zeros(3, dtype=torch.int32, device=DEV), torch.zeros(4, dtype=torch.int32, device=DEV)
    w = torch.zeros(4, 2, device=DEV)
    with pytest.raises(ops.KernelError):
        ops.grouped_up(y, up, 24, 0, 0, off, order, 1, w, h, activation="relu")         # two experts of 24 rows in 40
    with pytest.raises(ops.KernelError):
        ops.grouped_up(y, up[:, :20].contiguous(), 20, 0, 0, off, order, 1, w, h[:, :20].contiguous(), activation="relu")
    with pytest.raises(ops.KernelError):
        ops.grouped_up(y, up[:32], 16, 0, 0, off, order, 1, w, h[:, :16].contiguous(), activation="xielu")
    assert not ops.grouped_experts_serve(y, up, up, 12, 0)
    assert not ops.grouped_experts_serve(y.float(), up, up, 16, 0)


@pytest.mark.parametrize("n", [17, 40, 128])
def test_a_graph_of_a_routed_step(n):
    """Steps that a graph may hold: its replays follow the rows' own choices, and give the eager bits."""
    from types import SimpleNamespace
    from torchless_rs_amd.parts import ffn_routed
    from torchless_rs_amd.parts.base import Workspace
    H, E, top, ff = 128, 16, 4, 2304
    part = ffn_routed.RoutedExperts(H, E, top, ff, shared_size=ff + 128, activation="relu2")
    g = torch.Generator(device=DEV).manual_seed(n)
    part.load({k: (torch.randn(v.shape, generator=g, device=DEV) * v.shape[-1] ** -0.5).bfloat16() for k, v in part.weight_specs().items()},
              torch.bfloat16)

    def context():
        return SimpleNamespace(workspace=Workspace(torch.device(DEV)), dtype=torch.bfloat16, host={"fixed_launches": True}, pending=None)

    y, x, ctx = torch.empty(n, H, dtype=torch.bfloat16, device=DEV), torch.empty(n, H, device=DEV), context()
    inputs = [torch.randn(n, H, generator=g, device=DEV).bfloat16() for _ in range(4)]
    y.copy_(inputs[0])
    assert part.may_capture(n) and part.many_rows(ctx, y)
    part.produce(ctx, y, x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        part.produce(ctx, y, x)
    for t in inputs + inputs[:2]:
        y.copy_(t)
        graph.replay()
        torch.cuda.synchronize()
        out = torch.empty(n, H, device=DEV)
        part.produce(context(), t, out)
        assert torch.equal(out, x)
        s = torch.softmax(t.double() @ part.router.double().T, dim=-1)
        picked = s.topk(top + 1)
        sure = picked.values[:, top - 1] > picked.values[:, top] * (1 + 1e-4)
        wt = torch.zeros_like(s).scatter_(1, picked.indices[:, :top], picked.values[:, :top]).repeat_interleave(ff, dim=1)
        h = torch.relu(t.double() @ part.up.weight.double().T) ** 2
        h[:, :E * ff] *= wt
        want = h @ part.down.weight.double().T
        # the hidden channels are rounded to bfloat16: a thousand and more of them, so far below 2^-8 of a result's size
        assert float((out[sure].double() - want[sure]).norm() / want[sure].norm()) < 2.0 ** -8


@pytest.mark.parametrize("E,top,groups,keep,options", [
    (16, 4, 0, 0, {}), (16, 4, 4, 2, {}), (130, 3, 0, 0, {"logistic": True}), (24, 6, 4, 2, {"logistic": True, "correction": True, "two_largest": True}),
    (8, 8, 0, 0, {"normalise_eps": 0.0}), (5, 2, 0, 0, {"correction": True})])
@pytest.mark.parametrize("n", [9, 70])
def test_rows_whose_scores_are_not_numbers_choose_experts(ops, n, E, top, groups, keep, options):
    """NaN and infinite rows among others: every slot holds an expert and no expert twice, the row's NaN stays in its weights,
    and the other rows have the bits they have without them."""
    W = 64
    g = torch.Generator(device=DEV).manual_seed(n + E)
    y, router = (torch.randn(r, W, generator=g, device=DEV) for r in (n, E))
    if options.get("correction"):
        options = dict(options, correction=torch.randn(E, generator=g, device=DEV))
    bad = {1: float("nan"), 3: float("inf"), n - 1: -float("inf")}
    spoilt = y.clone()
    for row, value in bad.items():
        spoilt[row, row % W] = value
    spoilt[1] = float("nan")
    results = []
    for rows in (y, spoilt):
        weights, chosen = torch.empty(n, E, device=DEV), torch.full((n, top), -1, dtype=torch.int32, device=DEV)
        ops.route(rows, router, groups, keep, top, weights, chosen, **options)
        assert int(chosen.min()) >= 0 and int(chosen.max()) < E
        assert bool((chosen.sort(dim=1).values.diff(dim=1) > 0).all()) or top == 1
        results.append((weights, chosen))
    (weights, chosen), (w_spoilt, c_spoilt) = results
    well = [r for r in range(n) if r not in bad]
    assert torch.equal(weights[well], w_spoilt[well]) and torch.equal(chosen[well], c_spoilt[well])
    assert bool(w_spoilt[1][c_spoilt[1].long()].isnan().all())


@pytest.mark.parametrize("n", [20, 64, 200])
def test_a_routed_step_with_rows_that_are_not_numbers(n):
    """The rows beside one of NaN keep their bits; its own result is NaN."""
    from types import SimpleNamespace
    from torchless_rs_amd.parts import ffn_routed
    from torchless_rs_amd.parts.base import Workspace
    H, E, top, ff = 64, 16, 4, 3000
    part = ffn_routed.RoutedExperts(H, E, top, ff, shared_size=64, activation="relu2")
    g = torch.Generator(device=DEV).manual_seed(n)
    part.load({k: (torch.randn(v.shape, generator=g, device=DEV) * v.shape[-1] ** -0.5).bfloat16() for k, v in part.weight_specs().items()},
              torch.bfloat16)
    y = torch.randn(n, H, generator=g, device=DEV).bfloat16()
    spoilt = y.clone()
    spoilt[[2, n - 1]] = float("nan")
    out = []
    for rows in (y, spoilt):
        ctx = SimpleNamespace(workspace=Workspace(torch.device(DEV)), dtype=torch.bfloat16, host={}, pending=None)
        assert part.many_rows(ctx, rows)
        ctx.workspace.get("experts_chosen", (n, top), torch.int32).fill_(-1)
        ctx.workspace.get("experts_place", (n * top,), torch.int32).fill_(0)
        x = torch.empty(n, H, device=DEV)
        part._grouped(ctx, rows, x, False)
        out.append(x)
    well = [r for r in range(n) if r not in (2, n - 1)]
    # (which rows share a tile may change with the choices of two, which changes no row's order of sums)
    assert torch.equal(out[0][well], out[1][well])
    assert bool(out[1][[2, n - 1]].isnan().all())


@pytest.mark.parametrize("positions", [1, 31, 32, 33, 95, 97, 159, 161, 191, 193, 223, 224, 225, 449])
@pytest.mark.parametrize("H,ff", [(64, 256), (136, 264), (320, 24)])
@pytest.mark.parametrize("gated", [False, True])
def test_tiles_of_every_height(ops, positions, H, ff, gated):
    """An expert of `positions` rows between one of none and one of a single row: a tile is up to 224 positions high, in steps
    of 32, and K's end may lie inside a stage of 64 (136, 264, 24) or be the first stage's (64, 24).  The bounds are those
    of `test_experts_over_their_own_rows`."""
    E, n, wide = 3, positions + 1, 2 if gated else 1
    g = torch.Generator(device=DEV).manual_seed(positions + H)
    up = (torch.randn(wide * E * ff, H, generator=g, device=DEV) * H ** -0.5).bfloat16()
    down = (torch.randn(H, E * ff, generator=g, device=DEV) * ff ** -0.5).bfloat16()
    y = torch.randn(n, H, generator=g, device=DEV).bfloat16()
    chosen = torch.full((n, 1), 1, dtype=torch.int32, device=DEV)
    chosen[n // 2] = 2
    weights = torch.rand(n, E, generator=g, device=DEV) + 0.1
    off, order, place = grouped(ops, chosen, E)
    h = torch.empty(n, ff, dtype=torch.bfloat16, device=DEV)
    act = {"terms": ops.GateTerms(1.5, 1.702, 1.0, 0.75, True)} if gated else {"activation": "relu2"}
    ops.grouped_up(y, up, ff, 0, 0, off, order, 1, weights, h, **act)
    want, z_want, z_size = (torch.zeros(n, c, dtype=torch.float64, device=DEV) for c in (ff, H, H))
    for e, at in ((1, slice(0, positions)), (2, slice(positions, n))):
        rows = order[at].long()
        s = weights[rows, e: e + 1].double()
        p = y[rows].double() @ up[wide * e * ff: wide * (e + 1) * ff].double().T
        if gated:
            a, u = (p[:, :ff] * s).clamp(max=1.5), (p[:, ff:] * s).clamp(-1.5, 1.5)
            want[at] = a * torch.sigmoid(1.702 * a) * (u + 1.0)
        else:
            want[at] = torch.relu(p) ** 2 * s
        d = down[:, e * ff: (e + 1) * ff].double()
        z_want[at], z_size[at] = h[at].double() @ d.T, h[at].double().abs() @ d.abs().T
    assert float(((h.double() - want).abs() - want.abs() * 2.0 ** -8).max()) < 1e-4 * float(want.abs().max())
    z = torch.empty(n, H, device=DEV)
    ops.grouped_down(h, down, E, 0, 0, 1, off, z)
    assert bool(((z.double() - z_want).abs() <= (ff + 8) * 2.0 ** -24 * z_size + 1e-30).all())


@pytest.mark.parametrize("on_input", [False, True])
@pytest.mark.parametrize("n,shared", [(40, 0), (300, 304), (700, 0)])
def test_a_gated_experts_epilogue_has_the_bits_of_the_activation(ops, n, shared, on_input):
    """What a tile does with its sums is what the activation's own kernel makes of the same sums stored (K's stages in one order in
    both), far from 0 too: pre-activations reach 20 and the clamp is off for the experts."""
    H, E, top, ff = 136, 4, 2, 264
    slices = ops.shared_slices(ff, shared) if shared else 0
    g = torch.Generator(device=DEV).manual_seed(n)
    up = (torch.randn(2 * (E * ff + shared), H, generator=g, device=DEV) * 5.0 * H ** -0.5).bfloat16()
    y = torch.randn(n, H, generator=g, device=DEV).bfloat16()
    weights, sw = torch.rand(n, E, generator=g, device=DEV) + 0.5, torch.rand(n, generator=g, device=DEV)
    off, order, place = grouped(ops, choose(n, E, top, n, False), E)
    terms = ops.GateTerms(float("inf"), 1.702, 1.0, 7.0, on_input)
    h = torch.zeros(n * (top + slices), ff, dtype=torch.bfloat16, device=DEV)
    ops.grouped_up(y, up, ff, shared, slices, off, order, top, weights, h, terms=terms, shared_weight=sw)
    bounds = off.tolist()
    for e in range(E):
        rows = order[bounds[e]:bounds[e + 1]].long() // top
        u, want = torch.empty(len(rows), 2 * ff, device=DEV), torch.empty(len(rows), ff, dtype=torch.bfloat16, device=DEV)
        ops.gemm_tall_bf16(y[rows].contiguous(), up[2 * e * ff:2 * (e + 1) * ff], u, ops.TallPlan(224, 256))
        ops.expert_gated_act(u, weights[rows, e:e + 1].contiguous(), 1, ff, 0, terms, want)
        assert torch.equal(h[bounds[e]:bounds[e + 1]], want)
    if shared:
        u, want = torch.empty(n, 2 * shared, device=DEV), torch.empty(n, shared, dtype=torch.bfloat16, device=DEV)
        ops.gemm_tall_bf16(y, up[2 * E * ff:], u, ops.TallPlan(224, 256))
        ops.expert_gated_act(u, None, 0, 0, shared, terms, want, sw)
        mine = torch.cat([h[n * (top + j):n * (top + j + 1)] for j in range(slices)], dim=1)[:, :shared]
        assert torch.equal(mine, want)
