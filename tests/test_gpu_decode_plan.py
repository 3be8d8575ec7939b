"""A single-token step's keys in parts by the lengths of its sequences (attn_decode_plan_kernel, csrc/attention_bf16.hip): the plan
against its rule, and attention through it against float64."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PAGE = 64


@pytest.fixture(scope="module")
def ops():
    from torchless_rs_amd.kernels import ops as o
    o.lib()
    return o


def n_pages(p, window, keep, chunk):
    lo = max(0, p - window + 1) if window else 0
    if chunk:
        lo = max(lo, p // chunk * chunk)
    kept = min(-(-keep // PAGE), lo // PAGE) if window else 0
    return p // PAGE - lo // PAGE + 1 + kept


def part_pages(n, round_, rounds):
    """The rule: over the counts of rounds that hold every sequence, the smallest parts that fit, the count with the least rounds x
    pages (the fewest rounds of equal ones), at least as many pages as the merge of a part more is worth."""
    best = None
    least = next(q for q in range(1, 10 ** 6) if 20 * q * q >= 3 * max(n))
    for k in range(1, rounds + 1):
        if k * round_ < len(n):
            continue
        q = next(q for q in range(1, max(n) + 1) if sum(-(-x // q) for x in n) <= k * round_)
        q = max(q, least)
        if best is None or k * q < best[0]:
            best = (k * q, q)
    return best[1]


@pytest.mark.parametrize("lengths,round_,rounds", [([1, 1], 2, 1), ([64, 65, 130], 16, 1), ([1062, 1125, 1319, 1323, 2297, 2604, 3832, 8192], 64, 1),
                                                   ([4096] * 20, 64, 1), ([4096] * 22, 64, 3), ([131072, 1], 512, 1), (list(range(1, 6400, 100)), 64, 3),
                                                   ([17] * 512, 512, 1), ([9000] + [30] * 99, 100, 3), ([5000] * 65, 512, 2)])
@pytest.mark.parametrize("window,keep,chunk", [(0, 0, 0), (300, 0, 0), (4096, 100, 0), (0, 0, 256)])
def test_a_plan_covers_every_page_once_in_the_smallest_parts(ops, lengths, round_, rounds, window, keep, chunk):
    B, places = len(lengths), round_ * rounds
    pos = [x - 1 for x in lengths]
    plan = torch.full((places + 8, 4), -7, dtype=torch.int32, device=DEV)
    seqs = torch.full((B, 2), -7, dtype=torch.int32, device=DEV)
    row_pos = torch.tensor(pos, dtype=torch.int32, device=DEV)
    ops._check(ops.lib().tl_attn_decode_plan(ops._p(row_pos), B, window, keep, chunk, round_, rounds, ops._p(plan), ops._p(seqs), ops._stream()))
    plan, seqs = plan.tolist(), seqs.tolist()
    n = [n_pages(p, window, keep, chunk) for p in pos]
    Q = part_pages(n, round_, rounds)
    at = 0
    for b in range(B):
        parts = -(-n[b] // Q)
        assert seqs[b] == [at, parts]
        cuts = [s * n[b] // parts for s in range(parts + 1)]
        assert plan[at:at + parts] == [[4 * b + 2 * (s == 0) + (parts == 1), cuts[s], cuts[s + 1], pos[b]] for s in range(parts)]
        at += parts
    assert at <= places and all(e[0] == -1 for e in plan[at:places]) and plan[places:] == [[-7] * 4] * 8


@pytest.mark.parametrize("lengths,first,resident", [([64 * (i % 33) + 5 for i in range(64)], 32, 64), ([700] * 64, 32, 64), ([9, 1000], 1, 2),
                                                    (list(range(1, 5121, 10)), 32, 64), ([500, 40, 3000], 3, 3), ([100 * i + 1 for i in range(45)], 32, 64)])
@pytest.mark.parametrize("window,keep,chunk", [(0, 0, 0), (300, 0, 0), (4096, 100, 0), (0, 0, 256)])
def test_an_order_has_every_sequence_once_the_longest_beside_the_shortest(ops, lengths, first, resident, window, keep, chunk):
    B, pos = len(lengths), [x - 1 for x in lengths]
    plan = torch.full((B + 8, 4), -7, dtype=torch.int32, device=DEV)
    row_pos = torch.tensor(pos, dtype=torch.int32, device=DEV)
    ops._check(ops.lib().tl_attn_decode_order(ops._p(row_pos), B, window, keep, chunk, first, resident, ops._p(plan), ops._stream()))
    n = [n_pages(p, window, keep, chunk) for p in pos]
    ranks = sorted(range(B), key=lambda b: (-n[b], b))
    end = min(B, resident)
    want = ranks[:first] + ranks[first:end][::-1] + ranks[end:]
    assert plan.tolist() == [[4 * b + 3, 0, n[b], pos[b]] for b in want] + [[-7] * 4] * 8


def step(ops, lengths, nq, nkv, d, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    width = -(-max(lengths) // PAGE) + 1
    pages = torch.randn(len(lengths) * width, 2, nkv, PAGE, d, generator=g, device=DEV).bfloat16()
    table = torch.randperm(len(lengths) * width, generator=g, device=DEV).view(len(lengths), width).int()
    q = torch.randn(len(lengths), nq, d, generator=g, device=DEV).bfloat16()
    from torchless_rs_amd.parts.base import Workspace
    ctx = types.SimpleNamespace(n_rows=len(lengths), device=torch.device(DEV), host={}, workspace=Workspace(torch.device(DEV)), all_single=True,
                                row_pos=torch.tensor([x - 1 for x in lengths], dtype=torch.int32, device=DEV))
    return q, pages, table, ctx


def want(q, pages, table, lengths, scale, window=0, keep=0, chunk=0, logistic=False, bias=None, sinks=None, gate=None, slopes=None):
    B, nq, d = q.shape
    nkv = pages.shape[2]
    out, size = torch.empty(B, nq, d, dtype=torch.float64, device=DEV), torch.empty(B, nq, d, dtype=torch.float64, device=DEV)
    for b, L in enumerate(lengths):
        mine = pages[table[b].long()].double()
        k = mine[:, 0].transpose(0, 1).reshape(nkv, -1, d)[:, :L].repeat_interleave(nq // nkv, 0)
        v = mine[:, 1].reshape(-1, nkv, d, PAGE).permute(1, 0, 3, 2).reshape(nkv, -1, d)[:, :L].repeat_interleave(nq // nkv, 0)
        s = (k * q[b].double()[:, None]).sum(-1) * scale
        j, p = torch.arange(L, device=DEV), L - 1
        if slopes is not None:
            s = s - slopes.double()[:, None] * (p - j)
        ok = torch.ones(L, dtype=torch.bool, device=DEV)
        if window:
            ok &= (p - j < window) | (j < keep)
        if chunk:
            ok &= j // chunk == p // chunk
        if logistic:
            w = torch.sigmoid(s + bias.double()[:, None]) * ok
        else:
            s = s.masked_fill(~ok, float("-inf"))
            if sinks is not None:
                s = torch.cat([s, sinks.double()[:, None]], 1)
            w = torch.softmax(s, -1)[:, :L]
        if gate is not None:
            w = w * gate[b].double()[:, None]
        out[b], size[b] = (w[..., None] * v).sum(1), (w[..., None] * v.abs()).sum(1)
    return out, size


LENGTHS = [[1, 700], [64, 65, 1, 1500, 129], [2048] + [130] * 30, [3000, 1, 500, 2999] * 7]


@pytest.mark.parametrize("lengths", LENGTHS)
@pytest.mark.parametrize("nq,nkv,d", [(8, 2, 128), (32, 8, 64), (12, 3, 128), (4, 1, 256), (40, 2, 64)])
@pytest.mark.parametrize("window", [None, 300])
def test_attention_in_planned_parts(ops, lengths, nq, nkv, d, window):
    """The weights go to the second product with 8 bits and so does the result: up to 2^-8 of the sum of sizes and of itself."""
    q, pages, table, ctx = step(ops, lengths, nq, nkv, d)
    out = torch.full_like(q, float("nan"))
    planned = ops.decode_plan(ctx, nq, nkv, d, table.shape[1], window)
    if planned is None:                              # 28 or 31 sequences of these heads are more than half a round
        assert len(lengths) > 5
    assert planned is None or ops.decode_plan(ctx, nq, nkv, d, table.shape[1], window)[0] is planned[0]
    ops.attention(q, None, None, pages, table, table.shape[1], ctx, None, window, d ** -0.5, out)
    ref, size = want(q, pages, table, lengths, d ** -0.5, window or 0)
    assert bool(((out.double() - ref).abs() <= 2.0 ** -8 * (size + ref.abs()) + 1e-5).all())


@pytest.mark.parametrize("lengths", [[1, 4200], [64, 65, 1, 4500, 129], [4300] + [130] * 30])
@pytest.mark.parametrize("kind", ["sinks", "logistic", "kept", "chunk"])
def test_attention_with_terms_in_planned_parts(ops, lengths, kind):
    nq, nkv, d = 8, 2, 128
    q, pages, table, ctx = step(ops, lengths, nq, nkv, d, 1)
    g = torch.Generator(device=DEV).manual_seed(2)
    kw, ref_kw = {"sinks": ({"sinks": torch.randn(nq, generator=g, device=DEV)},) * 2,
                  "logistic": ({"logistic": True, "score_bias": torch.randn(nq, generator=g, device=DEV) - 4.0},) * 2,
                  "kept": ({"window": 200, "keep_first": 70},) * 2, "chunk": ({"chunk": 192},) * 2}[kind]
    ref_kw = {{"score_bias": "bias", "keep_first": "keep"}.get(k, k): v for k, v in ref_kw.items()}
    gate = torch.rand(len(lengths), nq, generator=g, device=DEV) if kind in ("sinks", "logistic") else None
    out = torch.full_like(q, float("nan"))
    ring = 1 << 20 if kind == "kept" else table.shape[1]
    ops.attention_scored(q, None, None, pages, nkv, d, table, ring, ctx, None, ops.ScoreTerms(d ** -0.5, **kw), gate, out)
    assert "decode_plans" in ctx.host
    ref, size = want(q, pages, table, lengths, d ** -0.5, gate=gate, **ref_kw)
    assert bool(((out.double() - ref).abs() <= 2.0 ** -8 * (size + ref.abs()) + 1e-5).all())


@pytest.mark.parametrize("nq,nkv,d,B", [(32, 8, 128, 64), (32, 8, 128, 128), (16, 16, 256, 32), (16, 8, 64, 64)])
def test_attention_in_an_order_has_the_bits_of_the_batch_s_own(ops, nq, nkv, d, B):
    lengths = [1 + (i * 613) % 900 for i in range(B)]
    q, pages, table, ctx = step(ops, lengths, nq, nkv, d)
    places, seqs = ops.decode_plan(ctx, nq, nkv, d, table.shape[1], None)
    assert seqs is None and tuple(places.shape) == (B, 4)
    out, own = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    ops.attention(q, None, None, pages, table, table.shape[1], ctx, None, None, d ** -0.5, out)
    part = torch.empty(B * nq * (d + 2), device=DEV)
    ops.attn_decode_bf16(q, pages, table, table.shape[1], ctx.row_pos, None, d ** -0.5, 1, part, own)
    assert torch.equal(out, own)


@pytest.mark.parametrize("kind", ["sinks", "logistic", "kept", "chunk", "slopes"])
def test_attention_with_terms_in_an_order(ops, monkeypatch, kind):
    """Whole sequences in an order with each of the terms, tables of more than 64 pages: the bits of the batch's own order, and float64's result at
    the weights' and the result's 8 bits."""
    nq, nkv, d, B = 16, 8, 64, 64
    lengths = [1 + (i * 613) % 900 for i in range(B)]
    lengths[5], lengths[40] = 4300, 2222
    q, pages, table, ctx = step(ops, lengths, nq, nkv, d, 3)
    g = torch.Generator(device=DEV).manual_seed(4)
    kw = {"sinks": {"sinks": torch.randn(nq, generator=g, device=DEV)}, "kept": {"window": 200, "keep_first": 70}, "chunk": {"chunk": 192},
          "logistic": {"logistic": True, "score_bias": torch.randn(nq, generator=g, device=DEV) - 4.0},
          "slopes": {"slopes": 0.02 * torch.rand(nq, generator=g, device=DEV)}}[kind]
    ref_kw = {{"score_bias": "bias", "keep_first": "keep"}.get(k, k): v for k, v in kw.items()}
    gate = torch.rand(B, nq, generator=g, device=DEV) if kind in ("sinks", "logistic") else None
    ring = 1 << 20 if kind == "kept" else table.shape[1]
    call = lambda out: ops.attention_scored(q, None, None, pages, nkv, d, table, ring, ctx, None, ops.ScoreTerms(d ** -0.5, **kw), gate, out)
    out, own = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
    call(out)
    assert [seqs for _, seqs in ctx.host["decode_plans"].values()] == [None]
    monkeypatch.setattr(ops, "decode_plan", lambda *a, **k: None)
    call(own)
    assert torch.equal(out, own)
    ref, size = want(q, pages, table, lengths, d ** -0.5, gate=gate, **ref_kw)
    assert bool(((out.double() - ref).abs() <= 2.0 ** -8 * (size + ref.abs()) + 1e-5).all())


def test_who_goes_without_a_plan(ops):
    assert ops.decode_places(32, 32, 8, 33, 256, 128) is None and ops.decode_places(48, 32, 8, 33, 256, 128) is None
    assert ops.decode_places(64, 32, 8, 33, 256, 128) == (32, 64) and ops.decode_places(64, 512, 512, 33, 256, 128) is None
    assert ops.decode_places(513, 4, 1, 33, 256, 128) is None
    assert ops.decode_rounds(1, 32, 8, 256, 128) is None and ops.decode_rounds(33, 32, 8, 256, 128) is None
    assert ops.decode_rounds(8, 32, 8, 256, 128) == (64, 1) and ops.decode_rounds(22, 32, 8, 256, 128) == (64, 3)
    assert ops.decode_rounds(513, 4, 1, 2048, 128) is None and ops.decode_rounds(4, 32, 32, 256, 256) == (8, 3)
    assert ops.decode_rounds(32, 32, 8, 256, 128) == (64, 3)
    q, pages, table, ctx = step(ops, [100, 70], 4, 2, 96)
    assert ops.decode_plan(ctx, 4, 2, 96, table.shape[1], None) is None and ops.decode_plan(ctx, 4, 2, 64, 2049, None) is None
    was = ops.decode_through_lds(False)
    try:
        assert ops.decode_plan(ctx, 4, 2, 64, 8, None) is None
    finally:
        ops.decode_through_lds(was)


@pytest.mark.parametrize("window", [None, 512])
def test_replayed_steps_are_planned_by_their_own_lengths(tmp_path, ops, window):
    """A captured step of two sequences over 11 pages makes its plan at every replay: the sequences change places in the batch and
    grow over page boundaries, with eager work and synchronisations between the replays, and every step has the bits of an
    engine that never captures, and float64's logits at the format's tolerance."""
    import plain_mistral as plain
    from torchless_rs_amd import write_random_model
    from torchless_rs_amd.engine import Engine, SeqInput, load_model
    from util import TOL, prompts, read_model_dir, rel_err
    cfg = {"architectures": ["MistralForCausalLM"], "model_type": "mistral", "hidden_size": 256, "num_hidden_layers": 2, "num_attention_heads": 4, "num_key_value_heads": 2, "head_dim": 64,
           "intermediate_size": 256, "vocab_size": 300, "rope_theta": 10000.0, "sliding_window": window, "rms_norm_eps": 1e-5,
           "max_position_embeddings": 4096, "tie_word_embeddings": False, "hidden_act": "silu"}
    mdir = write_random_model(str(tmp_path / "m"), cfg, seed=6, std=0.05, norm_std=0.1, dtype=torch.bfloat16)
    cfgd, w = read_model_dir(mdir)
    model = load_model(mdir, "bfloat16")
    ids = prompts(cfg["vocab_size"], [700, 700, 700], seed=9)
    at = [641, 20, 310]                                       # the first goes on inside its 11th page throughout
    engines = [Engine(model, max_tokens=64 * 48, max_slots=4, use_graphs=g) for g in (True, False)]
    for eng in engines:
        eng.slots_ = [eng.alloc() for _ in ids]
        eng.step([SeqInput(s, p[:n], []) for s, p, n in zip(eng.slots_, ids, at)])
    planned = 0
    for t in range(36):
        pair = [(0, 1), (1, 0), (0, 2), (2, 0)][t % 4]
        outs = []
        for eng in engines:
            outs.append(eng.step([SeqInput(eng.slots_[i], [ids[i][at[i]]], [0]) for i in pair]).clone())
            if t % 5 == 0:
                extra = eng.alloc()
                eng.step([SeqInput(extra, ids[1][:100 + t], [0])])
                eng.free(extra)
            torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[1]), t
        for row, i in enumerate(pair):
            if t % 9 == 0:
                assert rel_err(outs[0][row:row + 1], plain.forward(w, cfgd, ids[i][:at[i] + 1])[-1:]) < TOL["bfloat16"], (t, i)
            at[i] += 1
    for g in engines[0]._graphs.values():
        planned += g.graph is not None and any(name.startswith("attn_plan_") for name in g.workspace._bufs)
    assert planned and not engines[1]._graphs
    for eng in engines:
        eng.close()


def test_replayed_steps_are_ordered_by_their_own_lengths(tmp_path, ops):
    """A captured step of 64 sequences puts them in order at every replay: they change places in the batch and grow over page boundaries,
    with eager work and synchronisations between the replays, and every step has the bits of an engine that never captures, and
    float64's logits at the format's tolerance."""
    import plain_mistral as plain
    from torchless_rs_amd import write_random_model
    from torchless_rs_amd.engine import Engine, SeqInput, load_model
    from util import TOL, prompts, read_model_dir, rel_err
    cfg = {"architectures": ["MistralForCausalLM"], "model_type": "mistral", "hidden_size": 256, "num_hidden_layers": 2, "num_attention_heads": 8, "num_key_value_heads": 8, "head_dim": 64,
           "intermediate_size": 256, "vocab_size": 300, "rope_theta": 10000.0, "sliding_window": None, "rms_norm_eps": 1e-5,
           "max_position_embeddings": 4096, "tie_word_embeddings": False, "hidden_act": "silu"}
    mdir = write_random_model(str(tmp_path / "m"), cfg, seed=7, std=0.05, norm_std=0.1, dtype=torch.bfloat16)
    cfgd, w = read_model_dir(mdir)
    model = load_model(mdir, "bfloat16")
    B = 64
    ids = prompts(cfg["vocab_size"], [500] * B, seed=10)
    at = [460 if i == 3 else 1 + (i * 53) % 300 for i in range(B)]       # the longest goes on inside its 8th page
    engines = [Engine(model, max_tokens=64 * 8 * (B + 2), max_slots=B + 2, use_graphs=g) for g in (True, False)]
    for eng in engines:
        eng.slots_ = [eng.alloc() for _ in ids]
        eng.step([SeqInput(s, p[:n], []) for s, p, n in zip(eng.slots_, ids, at)])
    for t in range(20):
        batch = sorted(range(B), key=lambda i: (i * (2 * t + 1) + 11 * t) % B)
        outs = []
        for eng in engines:
            outs.append(eng.step([SeqInput(eng.slots_[i], [ids[i][at[i]]], [0]) for i in batch]).clone())
            if t % 4 == 0:
                extra = eng.alloc()
                eng.step([SeqInput(extra, ids[1][:100 + t], [0])])
                eng.free(extra)
            torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[1]), t
        for row, i in enumerate(batch):
            if t % 9 == 0 and row % 13 == 0:
                assert rel_err(outs[0][row:row + 1], plain.forward(w, cfgd, ids[i][:at[i] + 1])[-1:]) < TOL["bfloat16"], (t, i)
            at[i] += 1
    assert any(g.graph is not None and any(name.startswith("attn_plan_order") for name in g.workspace._bufs) for g in engines[0]._graphs.values())
    assert not engines[1]._graphs
    for eng in engines:
        eng.close()


@pytest.mark.parametrize("B,nq,nkv,d,splits", [(1, 32, 8, 128, 16), (1, 32, 8, 128, 2), (3, 40, 2, 64, 9), (2, 6, 6, 256, 5), (5, 17, 1, 128, 33), (8, 32, 8, 128, 8)])
def test_parts_merged_by_the_last_of_them_have_the_bits_of_a_merge_of_its_own(ops, B, nq, nkv, d, splits):
    lengths = [1 + (i * 977 + 700) % 2300 for i in range(B)]        # with fewer pages than parts among them
    q, pages, table, ctx = step(ops, lengths, nq, nkv, d, seed=3)
    part = torch.full((B * nq * splits * (d + 2),), float("nan"), device=DEV)
    apart, met = torch.zeros_like(q), torch.zeros_like(q)
    ops.attn_decode_bf16(q, pages, table, table.shape[1], ctx.row_pos, None, 0.1, splits, part, apart)
    arrived = ops.decode_counters(ctx, B, nq, nkv)
    for _ in range(4):                                               # the counters are left as they were found
        part.fill_(float("nan"))
        met.zero_()
        ops.attn_decode_bf16(q, pages, table, table.shape[1], ctx.row_pos, None, 0.1, splits, part, met, arrived)
        assert torch.equal(met, apart) and int(arrived.abs().max()) == 0


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("splits", [9, 16, 20, 36])
def test_merged_parts_have_those_bits_where_they_come_in_more_than_one_trip(ops, d, splits):
    """Many channels: a sum that one of the two ways rounds elsewhere changes a bfloat16 in some hundred thousand."""
    q, pages, table, ctx = step(ops, [2200 + i for i in range(64)], 64, 8, d, seed=splits)
    part = torch.full((64 * 64 * splits * (d + 2),), float("nan"), device=DEV)
    apart, met = torch.zeros_like(q), torch.zeros_like(q)
    ops.attn_decode_bf16(q, pages, table, table.shape[1], ctx.row_pos, None, 0.1, splits, part, apart)
    ops.attn_decode_bf16(q, pages, table, table.shape[1], ctx.row_pos, None, 0.1, splits, part, met, ops.decode_counters(ctx, 64, 64, 8))
    assert torch.equal(met, apart)


@pytest.mark.parametrize("sort", ["plain", "sinks", "logistic", "window"])
@pytest.mark.parametrize("nq,nkv,d", [(8, 2, 64), (8, 2, 128), (4, 2, 256), (34, 2, 128)])
def test_planned_parts_and_terms_merge_to_the_same_bits_both_ways(ops, monkeypatch, sort, nq, nkv, d):
    """Planned parts (counts that differ by sequence, one part among them) and uniform ones, with and without terms, merged by the last
    part and by the launch; one buffer of counters for two numbers of sequences, zero behind every launch."""
    from torchless_rs_amd.parts.base import Workspace
    g = torch.Generator(device=DEV).manual_seed(d)
    rand = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    kw = {"plain": None, "sinks": dict(sinks=rand(nq), slopes=rand(nq).abs() * 1e-3), "logistic": dict(logistic=True, score_bias=rand(nq)),
          "window": dict(window=500, keep_first=64)}[sort]
    terms = ops.ScoreTerms(0.1, **kw) if kw is not None else None
    spaces = {meet: Workspace(torch.device(DEV)) for meet in (True, False)}
    for lengths in ([6000, 1, 700, 2500, 64, 65, 1300], [900, 5000], [4100]):
        q, pages, table, ctx = step(ops, lengths, nq, nkv, d, seed=len(lengths))
        gate = torch.rand(len(lengths), nq, generator=g, device=DEV) if sort in ("sinks", "logistic") else None
        got = {}
        for meet, ws in spaces.items():
            monkeypatch.setattr(ops, "meeting_counters", lambda ctx, B, nq, nkv, *rest, _m=meet: ops.decode_counters(ctx, B, nq, nkv) if _m else None)
            ctx.workspace, ctx.host = ws, {}
            if sort != "plain":
                ways = [lambda out: ops.attention_scored(q, None, None, pages, nkv, d, table, 1 << 24, ctx, None, terms, gate, out)]
            else:
                ways = [lambda out: ops.attention(q, None, None, pages, table, 1 << 24, ctx, None, None, 0.1, out)]
            plan = ops.decode_plan(ctx, nq, nkv, d, table.shape[1], terms.window if terms else None, terms.keep_first if terms else 0)
            if plan is not None:
                assert plan[1] is not None and int(plan[1][:, 1].max()) > 1
                ways.append(lambda out: ops.attn_decode_planned(q, pages, table, 1 << 24, ctx, plan, terms.window if terms else None, 0.1, out, terms, gate))
            for way in ways:
                out = torch.zeros_like(q)
                way(out)
                got.setdefault(meet, []).append(out)
                if meet:
                    assert not bool(ops.decode_counters(ctx, len(lengths), nq, nkv).any())
        assert len(got[True]) == len(got[False]) == 1 + (len(lengths) > 1)
        for a, b in zip(got[True], got[False]):
            assert torch.equal(a, b) and bool(a.any())


def test_too_few_counters_are_refused(ops, monkeypatch):
    """By every way in, before anything is launched."""
    lengths = [900, 1400]
    q, pages, table, ctx = step(ops, lengths, 40, 2, 64)         # 20 heads a group: two times 16
    need = ops.decode_counters(ctx, 2, 40, 2).numel()
    assert need >= 2 * 2 * 2 * 4
    out, part = torch.zeros_like(q), torch.zeros(2 * 40 * 4 * 66, device=DEV)
    with pytest.raises(ops.KernelError, match="counters"):
        ops.attn_decode_bf16(q, pages, table, table.shape[1], ctx.row_pos, None, 0.1, 4, part, out,
                             torch.zeros(need - 1, dtype=torch.int32, device=DEV))
    q, pages, table, ctx = step(ops, lengths, 8, 2, 64)
    short = torch.zeros(ops.decode_counters(ctx, 2, 8, 2).numel() - 1, dtype=torch.int32, device=DEV)
    out = torch.zeros_like(q)
    plan = ops.decode_plan(ctx, 8, 2, 64, table.shape[1], None)
    assert plan is not None and plan[1] is not None
    terms = ops.ScoreTerms(0.125, sinks=torch.zeros(8, device=DEV))
    monkeypatch.setattr(ops, "decode_counters", lambda *a: short)
    for call in (lambda: ops.attn_decode_planned(q, pages, table, table.shape[1], ctx, plan, None, 0.1, out),
                 lambda: ops.attn_decode_planned(q, pages, table, table.shape[1], ctx, plan, None, 0.1, out, terms=terms),
                 lambda: ops.attention_scored(q, None, None, pages, 2, 64, table, table.shape[1], ctx, None, terms, None, out)):
        with pytest.raises(ops.KernelError, match="counters"):
            call()
    assert not bool(out.any()) and not bool(short.any())


@pytest.mark.parametrize("nq,nkv,B,meet", [(8, 8, 1, True), (8, 2, 1, True), (8, 2, 2, True), (10, 2, 1, False), (32, 2, 2, False),
                                           (8, 2, 60, True), (8, 2, 90, False), (8, 2, 300, False)])
def test_parts_meet_where_a_wave_has_one_head_and_all_run_at_a_time(ops, monkeypatch, nq, nkv, B, meet):
    """Uniform parts and planned ones; of 90 sequences in three rounds of places, and of 300 in two parts each, some wait for their places."""
    assert ops.compute_units(torch.device(DEV)) == 256
    real, asked = ops.decode_counters, []
    monkeypatch.setattr(ops, "decode_counters", lambda *a: (asked.append(a[1:]), real(*a))[1])
    lengths = [700] * B
    q, pages, table, ctx = step(ops, lengths, nq, nkv, 64)
    out = torch.zeros_like(q)
    ops.attention(q, None, None, pages, table, table.shape[1], ctx, None, None, 0.1, out)
    assert asked == [(B, nq, nkv)] * meet
    asked.clear()
    ops.attention_scored(q, None, None, pages, nkv, 64, table, table.shape[1], ctx, None, ops.ScoreTerms(0.1), None, out)
    splits = ops.decode_splits(B, nq, nkv, table.shape[1], 256, 64)
    assert asked == [(B, nq, nkv)] * (nq // nkv <= 4 and splits > 1 and splits * B * nkv <= 512)
    ref, size = want(q, pages, table, lengths, 0.1)
    assert bool(((out.double() - ref).abs() <= 2.0 ** -8 * (size + ref.abs()) + 1e-5).all())
