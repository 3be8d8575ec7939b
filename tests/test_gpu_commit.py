"""Keys and values that go into their pages with the rotation (`rope_v_tiles` with `commit`) against the commit behind the attention
(`kv_commit_tiles`), bit by bit, and which steps may."""
import types

import numpy as np
import pytest
import torch

DEV = "cuda:0"
PAGE = 64


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("ring", [5, 1 << 24])
@pytest.mark.parametrize("nq,nkv,d,rotary,odd", [(4, 2, 16, 16, 0), (6, 3, 80, 40, 0), (2, 1, 256, 256, 0), (32, 8, 128, 128, 0), (4, 2, 128, 128, 1), (3, 1, 66, 66, 0)])
def test_pages_written_with_the_rotation(dt, ring, nq, nkv, d, rotary, odd):
    """Sequences that start inside a page, on one, end on one; a cache whose first element is not aligned (`odd`)."""
    from torchless_rs_amd.kernels import ops
    cached, new = [0, 70, 64, 120, 5], [2, 4, 64, 200, 59]
    B, n = len(cached), sum(new)
    i32 = lambda l: torch.tensor(l, dtype=torch.int32, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(d)
    qkv = torch.randn(n, (nq + 2 * nkv) * d, generator=g, device=DEV)
    row_seq = i32([b for b in range(B) for _ in range(new[b])])
    row_pos = i32([cached[b] + i for b in range(B) for i in range(new[b])])
    cu, after = i32([sum(new[:b]) for b in range(B + 1)]), i32([c + m for c, m in zip(cached, new)])
    off, cols = ops.aligned_columns(cached, new)
    off, before = i32(off), i32(cached)
    rot = ops.Rotation(10000.0 ** (-2.0 * torch.arange(rotary // 2, device=DEV) / rotary), rotary)
    need = [-(-(c + m) // PAGE) for c, m in zip(cached, new)]
    n_pages = sum(need) + 2
    perm = torch.randperm(n_pages, generator=torch.Generator().manual_seed(5)).tolist()
    table = torch.zeros(B, max(need), dtype=torch.int32)
    for b in range(B):
        table[b, :need[b]] = torch.tensor([perm.pop() for _ in range(need[b])], dtype=torch.int32)
    table = table.to(DEV)

    def run(early):
        q, k = torch.full((n, nq, d), 5.0, dtype=dt, device=DEV), torch.full((n, nkv, d), 5.0, dtype=dt, device=DEV)
        vt = torch.full((nkv, d, cols), 7.0, dtype=dt, device=DEV)
        size = n_pages * 2 * nkv * PAGE * d
        pages = torch.full((size + odd,), 3.0, dtype=dt, device=DEV)[odd:].view(n_pages, 2, nkv, PAGE, d)
        ops.rope_v_tiles(qkv, row_pos, rot, nq, nkv, d, q, k, vt, cu, off, before, after, commit=(row_seq, table, ring, pages) if early else None)
        if not early:
            ops.kv_commit_tiles(k, vt, row_seq, row_pos, off, before, after, table, ring, pages)
        return q, k, vt, pages

    for a, b in zip(run(True), run(False)):
        assert torch.equal(a, b)


def test_which_steps_overwrite_nothing():
    from torchless_rs_amd.kernels import ops
    from torchless_rs_amd.kernels.page import NO_RING
    ctx = lambda lens, fixed: types.SimpleNamespace(host={"len_after": np.array(lens), "fixed_launches": fixed})
    assert ops.overwrite_nothing(ctx([1, 128], False), 2) and not ops.overwrite_nothing(ctx([1, 129], False), 2)
    assert ops.overwrite_nothing(ctx([10 ** 6], False), NO_RING) and ops.overwrite_nothing(ctx([10 ** 6], True), NO_RING)
    assert not ops.overwrite_nothing(ctx([1], True), NO_RING - 1)          # (the captured step's next lengths are not known)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("S", [2, 3, 5, 16])
@pytest.mark.parametrize("nq,nkv,d,rotary,odd", [(4, 2, 16, 16, 0), (6, 3, 80, 40, 0), (40, 8, 256, 256, 0), (32, 8, 128, 128, 0), (4, 2, 128, 128, 1), (3, 1, 66, 66, 0), (1, 1, 2, 2, 0), (2, 1, 2, 0, 0)])
def test_partial_sums_are_added_with_the_rotation(dt, S, nq, nkv, d, rotary, odd):
    """Partial sums of q|k|v against `add_partials` and the rotation of their sum, bit by bit; buffers off 16 bytes (`odd`)."""
    from torchless_rs_amd.kernels import ops
    cached, new = [0, 70, 64, 120, 5], [2, 4, 64, 100, 59]
    B, n, width = len(cached), sum(new), (nq + 2 * nkv) * d
    i32 = lambda l: torch.tensor(l, dtype=torch.int32, device=DEV)
    g = torch.Generator(device=DEV).manual_seed(S + d)
    parts = torch.empty(S * n * width + odd, device=DEV)[odd:].view(S, n, width)
    parts.copy_(torch.randn(S, n, width, generator=g, device=DEV))
    row_seq = i32([b for b in range(B) for _ in range(new[b])])
    row_pos = i32([cached[b] + i for b in range(B) for i in range(new[b])])
    cu, after = i32([sum(new[:b]) for b in range(B + 1)]), i32([c + m for c, m in zip(cached, new)])
    off, cols = ops.aligned_columns(cached, new)
    off, before = i32(off), i32(cached)
    rot = ops.Rotation(10000.0 ** (-2.0 * torch.arange(rotary // 2, device=DEV) / rotary), rotary)
    table = torch.randperm(B * 4, generator=g, device=DEV).view(B, 4).int()

    def run(qkv):
        q, k = torch.full((n, nq, d), 5.0, dtype=dt, device=DEV), torch.full((n, nkv, d), 5.0, dtype=dt, device=DEV)
        vt = torch.full((nkv, d, cols), 7.0, dtype=dt, device=DEV)
        pages = torch.full((B * 4, 2, nkv, PAGE, d), 3.0, dtype=dt, device=DEV)
        ops.rope_v_tiles(qkv, row_pos, rot, nq, nkv, d, q, k, vt, cu, off, before, after, commit=(row_seq, table, 1 << 24, pages))
        return q, k, vt, pages

    together = run(parts)
    total = torch.empty(n * width + odd, device=DEV)[odd:].view(n, width).copy_(parts[0])
    rest = torch.empty((S - 1) * n * width + odd, device=DEV)[odd:].view(S - 1, n, width).copy_(parts[1:])
    ops.add_partials(total, rest)
    for a, b in zip(together, run(total)):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,rows", [(1536, 4096, ()), (6144, 4160, (129, 192, 193, 256)), (4096, 4096, (129, 192)), (6144, 3072, ()), (6112, 4096, ())])
def test_which_prompts_leave_their_projection_in_partial_sums(N, K, rows):
    """129 to 256 rows: the sums of the slices against float64, each within the rounding of a chain of K / 32 products of 32 and the
    slices' sum (2^-24 of the sizes' sum an addition, 5 within an instruction); other rows and sizes go without."""
    from torchless_rs_amd.kernels import ops
    from torchless_rs_amd.parts.base import Workspace
    from torchless_rs_amd.parts.linear import Linear
    g = torch.Generator(device=DEV).manual_seed(N)
    lin = Linear(torch.randn(N, K, generator=g, device=DEV, dtype=torch.bfloat16))
    ctx = types.SimpleNamespace(workspace=Workspace(torch.device(DEV)))
    w = lin.weight.double()
    for M in (129, 192, 193, 256, 257):
        a = torch.randn(M, K, generator=g, device=DEV, dtype=torch.bfloat16)
        parts = lin.rotated_partial(a, ctx, "parts")
        assert (parts is not None) == (M in rows), M
        if parts is not None:
            S = parts.shape[0]
            want, size = a.double() @ w.t(), a.double().abs() @ w.abs().t()
            assert ((parts.double().sum(0) - want).abs() <= (K / 32 + 5 + S) * 2 ** -24 * size).all()

    class Own(Linear):
        def __call__(self, a, out, accumulate=False, factor=None):
            out.zero_()
    assert Own(lin.weight).rotated_partial(torch.ones(192, K, device=DEV, dtype=torch.bfloat16), ctx, "parts") is None


@pytest.mark.gpu
def test_a_projection_that_is_no_linear_serves_prompts(tmp_path):
    """A product of a caller's own that knows the parts of `Linear` which the mixer has asked for all along."""
    from torchless_rs_amd.engine import Engine, SeqInput, load_model
    from util import TOL, make_model_dir, prompts, rel_err
    model = load_model(make_model_dir(tmp_path, "A", torch.bfloat16), "bfloat16")
    ids = prompts(model.spec.vocab_size, [150], 3)[0]

    class Product:
        def __init__(self, real):
            self.real, self.weight, self.own_tiles, self.calls = real, real.weight, None, 0

        def own_kernels(self, n):
            return False

        def partial(self, a, ctx, name):
            return None

        def __call__(self, a, out):
            self.calls += 1
            self.real(a, out)

    def logits():
        eng = Engine(model, max_tokens=512, max_slots=2, use_graphs=False)
        return eng.step([SeqInput(eng.alloc(), ids, [149])]).clone()

    want = logits()
    mixers = [b.mixer for b in model.blocks]
    for m in mixers:
        m.qkv = Product(m.qkv)
    got = logits()
    assert all(m.qkv.calls == 1 for m in mixers)
    assert torch.isfinite(got).all() and rel_err(got, want.double()) < TOL["bfloat16"]
