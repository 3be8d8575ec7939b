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
