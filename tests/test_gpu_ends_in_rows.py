"""A step's last block over the rows alone whose logits are wanted (`ENDS_IN_ROWS` of engine/model.py) against all of its rows: logits
and everything that later steps read."""
import copy
import types

import pytest
import torch

from util import TOL, make_model_dir, prompts, rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def models(tmp_path, name, dtype):
    from torchless_rs_amd.engine import load_model
    if name in ("A", "B"):
        return load_model(make_model_dir(tmp_path, name, torch.bfloat16), dtype)
    import importlib
    t, plain = importlib.import_module(f"test_gpu_{name}"), importlib.import_module(f"plain_{name}")
    cfg = copy.deepcopy(t.CONFIGS["mixed"])
    return load_model(t.write_model(str(tmp_path / name), cfg, plain.random_weights(cfg, 7)), dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["A", "B", "nepisun", "giforax"])
def test_the_wanted_rows_alone_have_the_logits_of_all_rows(tmp_path, monkeypatch, name, dtype):
    """Prompts in pieces (no logits wanted, the last row's, several), then tokens: 17 rows, and more than a tile; each step three times
    over the same engines' lives, so that short ones come from a captured graph."""
    from torchless_rs_amd.engine import Engine, SeqInput
    from torchless_rs_amd.engine import model as m
    model = models(tmp_path, name, dtype)
    V = model.spec.vocab_size
    ids = prompts(V, [150, 40, 33], 3)
    engines = {all_rows: Engine(model, max_tokens=64 * 24, max_slots=4) for all_rows in (False, True)}
    narrow = []
    for block in model.blocks:
        if hasattr(block, "forward_rows"):
            real = block.forward_rows
            monkeypatch.setattr(block, "forward_rows", lambda *a, _r=real, **k: (narrow.append(1), _r(*a, **k))[1])
    for life in range(4):
        got = {}
        for all_rows, eng in engines.items():
            monkeypatch.setattr(m, "ENDS_IN_ROWS", 1 << 30 if all_rows else 16)
            slots = [eng.alloc() for _ in ids]
            out, before = [], len(narrow)
            steps = [[(0, 0, 17, [16])], [(0, 17, 60, []), (1, 0, 20, [])], [(0, 77, 73, [72]), (1, 20, 20, [19, 3]), (2, 0, 33, [32])]]
            for step in steps:
                out.append(eng.step([SeqInput(slots[s], ids[s][a:a + n], w) for s, a, n, w in step]).clone())
            for t in range(2):
                out.append(eng.step([SeqInput(s, [(5 * t + i) % V], [0]) for i, s in enumerate(slots)]).clone())
            got[all_rows] = out
            assert len(narrow) - before == (0 if all_rows else 3) or life > 1     # (a captured step runs once)
            for s in slots:
                eng.free(s)
        for a, b in zip(got[False], got[True]):
            assert a.shape == b.shape
            if a.numel():
                assert torch.isfinite(a).all() and rel_err(a, b.double()) < TOL[dtype]


def test_who_may_end_in_rows():
    from torchless_rs_amd.parts.base import rows_apart
    from torchless_rs_amd.parts.ffn import SwiGLU

    class Mixes(SwiGLU):
        def forward(self, ctx, y, x):
            x += y.sum(0)

    class Says(Mixes):
        row_wise = True

    plain = types.SimpleNamespace
    mk = lambda c: object.__new__(c)
    assert rows_apart(mk(SwiGLU)) and not rows_apart(mk(Mixes)) and rows_apart(mk(Says)) and not rows_apart(plain())
    patched = mk(SwiGLU)
    patched.forward = lambda *a: None
    assert not rows_apart(patched)


def test_who_gives_rows():
    from torchless_rs_amd.parts.attention import AttentionMixer
    from torchless_rs_amd.parts.attention_heads import HeadwiseAttentionMixer
    from torchless_rs_amd.parts.base import Mixer, gives_rows
    from torchless_rs_amd.parts.retention import RetentionMixer

    class Other(AttentionMixer):
        def forward(self, ctx, run, y, x):
            pass

    mk = lambda c: object.__new__(c)
    assert gives_rows(mk(AttentionMixer), "forward_rows") and not gives_rows(mk(AttentionMixer), "produce_rows")
    assert gives_rows(mk(HeadwiseAttentionMixer), "forward_rows") and gives_rows(mk(HeadwiseAttentionMixer), "produce_rows")
    assert not gives_rows(mk(Other), "forward_rows") and not gives_rows(mk(RetentionMixer), "forward_rows") and not gives_rows(mk(Mixer), "forward_rows")


@pytest.mark.parametrize("name,what", [("A", "hidden"), ("A", "hidden on the object"), ("A", "down"), ("A", "add_into on the product"), ("A", "o"),
                                       ("A", "norm"), ("giforax", "route"), ("giforax", "out norm"), ("giforax", "o")])
def test_ways_of_a_callers_own_run_over_all_rows(tmp_path, name, what):
    """A step of which one row is wanted, and in its last block a method or a product that is not the package's: it is handed every row."""
    from torchless_rs_amd.engine import Engine, SeqInput
    from torchless_rs_amd.parts.linear import Linear
    model = models(tmp_path, name, "bfloat16")
    block, rows = model.blocks[model.spec.schedule[-1].layer], []

    def derived(part, method, of):
        real = getattr(type(part), method)
        part.__class__ = type("Own", (type(part),), {method: lambda self, *a, **k: (rows.append(a[of].shape[0]), real(self, *a, **k))[1]})

    class Own(Linear):
        def __call__(self, a, *rest, **kw):
            rows.append(a.shape[0])
            Linear.__call__(self, a, *rest, **kw)

        def partial(self, *a):
            return None

        wide_partial = tall_partial = partial

    if what == "hidden":
        derived(block.ffn, "_hidden", 1)
    elif what == "hidden on the object":
        real = block.ffn._hidden
        block.ffn._hidden = lambda ctx, y: (rows.append(y.shape[0]), real(ctx, y))[1]
    elif what == "down":
        block.ffn.down = Own(block.ffn.down.weight)
    elif what == "add_into on the product":
        real_add = block.ffn.down.add_into
        block.ffn.down.add_into = lambda a, *rest: (rows.append(a.shape[0]), real_add(a, *rest))[1]
    elif what == "o":
        block.mixer.o = Own(block.mixer.o.weight)
    elif what == "norm":
        derived(block.ffn_norm, "forward", 1)
    elif what == "route":
        derived(block.ffn, "_route", 1)
    else:
        derived(block.ffn_out_norm, "add_to", 1)
    eng = Engine(model, max_tokens=512, max_slots=2, use_graphs=False)
    eng.step([SeqInput(eng.alloc(), prompts(model.spec.vocab_size, [40], 3)[0], [39])])
    assert rows == [40]


@pytest.mark.parametrize("n,want,alone", [(17, 2, True), (17, 3, False), (16, 1, False), (40, 0, True), (40, 5, True), (40, 6, False), (40, 39, False), (40, 40, False)])
def test_up_to_an_eighth_of_the_rows_end_alone(tmp_path, monkeypatch, n, want, alone):
    from torchless_rs_amd.engine import Engine, SeqInput
    model = models(tmp_path, "A", "bfloat16")
    block, narrow = model.blocks[model.spec.schedule[-1].layer], []
    real = block.forward_rows
    monkeypatch.setattr(block, "forward_rows", lambda *a, **k: (narrow.append(1), real(*a, **k))[1])
    eng = Engine(model, max_tokens=512, max_slots=2, use_graphs=False)
    eng.step([SeqInput(eng.alloc(), prompts(model.spec.vocab_size, [n], 3)[0], list(range(want)))])
    assert len(narrow) == alone


@pytest.mark.parametrize("derived", [False, True])
def test_a_last_norm_of_a_callers_own_reads_the_whole_stream(monkeypatch, derived):
    """The last feed-forward's product over 20 wanted rows comes in slices of K: a norm that knows nothing of them is handed their sum."""
    from torchless_rs_amd import config_from_dict
    from torchless_rs_amd.engine import Engine, SeqInput, model_from_tensors
    from torchless_rs_amd.engine import model as m
    from torchless_rs_amd.kernels import ops
    from torchless_rs_amd.models import model_spec_for
    cfg = config_from_dict(dict(architectures=["MistralForCausalLM"], num_hidden_layers=2, hidden_size=512, num_attention_heads=4, num_key_value_heads=2,
                                head_dim=128, intermediate_size=2048, vocab_size=1000, rope_theta=1e4, rms_norm_eps=1e-5))
    g = torch.Generator(device=DEV).manual_seed(2)
    specs = model_spec_for(cfg).weight_specs()
    w = {k: torch.ones(v.shape, device=DEV) if len(v.shape) == 1 else torch.randn(tuple(v.shape), generator=g, device=DEV) * v.shape[-1] ** -0.5
         for k, v in specs.items()}
    model = model_from_tensors(cfg, {k: t.bfloat16() for k, t in w.items()}, "bfloat16", DEV)
    norm = model.final_norm
    plain = lambda self, ctx, x, out: ops.rmsnorm(x, norm.weight, norm.eps, out)
    if derived:
        norm.__class__ = type("Own", (type(norm),), {"forward": plain})
    else:
        norm.forward = lambda ctx, x, out: plain(norm, ctx, x, out)
    got = []
    for line in (16, 1 << 30):
        monkeypatch.setattr(m, "ENDS_IN_ROWS", line)
        eng = Engine(model, max_tokens=512, max_slots=2, use_graphs=False)
        got.append(eng.step([SeqInput(eng.alloc(), prompts(1000, [200], 3)[0], list(range(0, 200, 10)))]).clone())
    assert torch.isfinite(got[0]).all() and rel_err(got[0], got[1].double()) < TOL["bfloat16"]


@pytest.mark.parametrize("H", [64, 1000, 4096, 8192])
@pytest.mark.parametrize("parts", [0, 1, 9])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_a_norm_of_some_rows_has_the_bits_of_adding_gathering_and_the_norm(H, parts, dt):
    from torchless_rs_amd.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(H + parts)
    n, rows = 37, torch.tensor([36, 0, 0, 17], dtype=torch.int32, device=DEV)
    x, w = torch.randn(n, H, generator=g, device=DEV), torch.randn(H, generator=g, device=DEV)
    p = torch.randn(parts, n, H, generator=g, device=DEV) if parts else None
    assert ops.rmsnorm_rows_ok(x, w, p) and not ops.rmsnorm_rows_ok(x[:, 1:], w, p) and not ops.rmsnorm_rows_ok(torch.zeros(2, 9000), w, None)
    out, keep, was = torch.zeros(4, H, dtype=dt, device=DEV), torch.zeros(4, H, device=DEV), x.clone()
    ops.rmsnorm(x, w, 1e-5, out, rows=rows, parts=p, keep=keep)
    assert torch.equal(x, was)
    if parts:
        ops.add_partials(x, p)
    xs, y = torch.zeros(4, H, device=DEV), torch.zeros(4, H, dtype=dt, device=DEV)
    ops.gather_rows(x, rows, xs)
    ops.rmsnorm(xs, w, 1e-5, y)
    assert torch.equal(keep, xs) and torch.equal(out, y)
    both = torch.stack([x, 2 * x])
    many = torch.zeros(2, 4, H, device=DEV)
    ops.gather_rows(both, rows, many)
    assert torch.equal(many, both[:, rows.long()])


def test_rows_are_gathered_of_one_matrix_or_several():
    """More dimensions than that were taken and all but the first matrices left out."""
    from torchless_rs_amd.kernels import ops
    rows = torch.tensor([2, 0], dtype=torch.int32, device=DEV)
    for shape in ((4,), (2, 3, 4, 8)):
        x = torch.zeros(shape, device=DEV)
        with pytest.raises(ops.KernelError, match="gather.x"):
            ops.gather_rows(x, rows, torch.zeros(shape[:-2] + (2, shape[-1]), device=DEV))
