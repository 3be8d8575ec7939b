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
@pytest.mark.parametrize("dk,dv,rotary", [(64, 64, 64), (65, 40, 24), (128, 128, 64), (128, 96, 128), (200, 64, 130), (256, 256, 256), (96, 32, 0)])
def test_heads_of_many_rows_are_those_of_few(ops, dtype, dk, dv, rotary):
    """A wave that goes from head to head leaves what a wave a head leaves, against 64 bits and bit by bit."""
    nq, nkv, ng, n = 3, 2, 300, 2100
    g = torch.Generator(device=DEV).manual_seed(dk + rotary)
    width = nq * dk + nkv * (dk + dv) + ng
    proj = torch.randn(n, width, generator=g, device=DEV)
    pos = torch.randint(0, 5000, (n,), generator=g, device=DEV, dtype=torch.int32)
    inv = 10000.0 ** (-2.0 * torch.arange(rotary // 2, device=DEV) / max(rotary, 1)) if rotary else None
    qn, kn = (1.0 + 0.1 * torch.randn(dk, generator=g, device=DEV) for _ in range(2))
    bias = torch.randn(width, generator=g, device=DEV)
    for kw in ({}, {"q_norm": qn, "k_norm": kn, "bias": bias}, {"unit_norm": True, "v_factor": 0.5}):
        def run(rows, at):
            m = rows.shape[0]
            q, k, v = (torch.empty(m, h, d, dtype=dtype, device=DEV) for h, d in ((nq, dk), (nkv, dk), (nkv, dv)))
            gate = torch.empty(m, ng, device=DEV)
            ops.head_prepare(rows, at, ops.Rotation(inv, rotary), ops.HeadTerms(eps=1e-5, **kw), nq, nkv, dk, dv, ng, q, k, v, gate)
            return q, k, v, gate
        many = run(proj, pos)
        few = [torch.cat(t) for t in zip(*(run(proj[i:i + 30], pos[i:i + 30]) for i in range(0, 90, 30)))]
        for a, b in zip(many, few):
            assert torch.equal(a[:90], b)
        t = proj.double() + (kw["bias"].double() if "bias" in kw else 0.0)
        x = t[:, :(nq + nkv) * dk].view(n, nq + nkv, dk)
        if "q_norm" in kw:
            x = x / (x.square().mean(-1, keepdim=True) + 1e-5).sqrt()
            x = torch.cat([x[:, :nq] * qn.double(), x[:, nq:] * kn.double()], 1)
        half = rotary // 2
        if half:
            angle = (pos.float()[:, None] * inv).double()[:, None]
            u, w = x[..., :half], x[..., half:rotary]
            x = torch.cat([u * angle.cos() - w * angle.sin(), u * angle.sin() + w * angle.cos(), x[..., rotary:]], -1)
        if kw.get("unit_norm"):
            x = x / (x.square().mean(-1, keepdim=True) + 1e-5).sqrt()
        # float32: a few roundings of 2^-24 of the two products of a rotated channel; bfloat16: one of up to 2^-8 of the result
        tol = 4e-6 * (1.0 + x.abs().amax(-1, keepdim=True)) + (2.0 ** -8 * x.abs() if dtype == torch.bfloat16 else 0.0)
        assert bool(((torch.cat(many[:2], 1).double() - x).abs() <= tol).all())


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


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nq,nkv,d", [(1, 1, 8), (3, 1, 64), (32, 8, 128), (5, 5, 200), (40, 8, 256)])
def test_pairs_by_fours_are_those_one_by_one(ops, dtype, nq, nkv, d):
    """Rotation four pairs a thread, values four channels and their commit 16 bytes at a time leave the bits that buffers off 16 bytes get,
    for 70 sequences, of which some begin inside a page and end inside one."""
    g = torch.Generator(device=DEV).manual_seed(d)
    new = [1 + (7 * b) % 131 for b in range(70)]
    cached = [(29 * b) % 200 for b in range(70)]
    n, i32 = sum(new), lambda l: torch.tensor(l, dtype=torch.int32, device=DEV)
    off, cols = ops.aligned_columns(cached, new)
    seq = i32([b for b in range(70) for _ in range(new[b])])
    pos = i32([cached[b] + i for b in range(70) for i in range(new[b])])
    cu, after = i32([sum(new[:b]) for b in range(71)]), i32([c + m for c, m in zip(cached, new)])
    inv = 10000.0 ** (-2.0 * torch.arange(d // 2, device=DEV) / d)
    data = torch.randn(n, (nq + 2 * nkv) * d, generator=g, device=DEV)
    table = torch.randperm(70 * 6, generator=g, device=DEV).view(70, 6).int()

    def run(shift):
        def buf(fill, *shape, dt=dtype):
            size = 1
            for s in shape:
                size *= s
            return torch.full((size + shift,), fill, dtype=dt, device=DEV)[shift:].view(shape)
        qkv = buf(0.0, *data.shape, dt=torch.float32).copy_(data)
        q, k, vt, pages = buf(3.0, n, nq, d), buf(3.0, n, nkv, d), buf(7.0, nkv, d, cols), buf(5.0, 420, 2, nkv, 64, d)
        ops.rope_v_tiles(qkv, pos, inv, nq, nkv, d, q, k, vt, cu, i32(off), i32(cached), after)
        ops.kv_commit_tiles(k, vt, seq, pos, i32(off), i32(cached), after, table, 1 << 24, pages)
        return q, k, vt, pages
    for a, b in zip(run(0), run(1)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(4096, 2048), (4097, 2048), (4104, 2048), (9001, 1028), (16384, 2044), (5000, 1024), (4500, 64), (12345, 4), (3000, 2052),
                                 (2048, 4096), (4103, 132)])
def test_few_rows_by_many_outputs(ops, M, N, K, accumulate):
    """One to four rows: the bits of the same rows among eight, whose kernel adds in the same order, and float64 within the order's
    rounding: a sum in runs, groups and their sum is a chain of K / 64 + 16 additions, each off by 2^-24 of the sum of the sizes."""
    g = torch.Generator(device=DEV).manual_seed(N + K)
    a, w = torch.randn(8, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    start = torch.randn(8, N, generator=g, device=DEV) if accumulate else torch.full((8, N), float("nan"), device=DEV)
    few, many = start[:M].clone(), start.clone()
    ops.gemm_plain(a[:M].contiguous(), w, few, accumulate)
    ops.gemm_plain(a, w, many, accumulate)
    assert torch.equal(few, many[:M])
    want = a[:M].double() @ w.double().t() + (start[:M].double() if accumulate else 0.0)
    size = a[:M].double().abs() @ w.double().abs().t() + (start[:M].double().abs() if accumulate else 0.0)
    assert bool(((few.double() - want).abs() <= (K / 64 + 18) * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,H", [(1, 1), (1, 4096), (3, 1023), (2, 1028), (40, 2050), (300, 4100)])
def test_rows_of_the_table(ops, dtype, n, H):
    g = torch.Generator(device=DEV).manual_seed(H)
    table = torch.randn(50, H, generator=g, device=DEV).to(dtype)
    ids = torch.randint(0, 50, (n,), generator=g, device=DEV, dtype=torch.int32)
    out = torch.full((n, H), float("nan"), device=DEV)
    ops.embed(table, ids, out, 1.5)
    assert torch.equal(out, table[ids.long()].float() * 1.5)
