"""Prompts through the many-row kernels (Model._prompt) are bitwise the 16-token passes they replace:
hidden states, logits, keys, values and Gated-DeltaNet states, at lengths that end inside a 16-token piece, a
64-token group and a 128-key chunk, from an empty cache and after cached tokens, on the small decoders and on
layers of the real sizes; and the prompt kernels alone, with workspaces that take several launches."""

import gc

import pytest
import torch

from skinny_mlx import kernels as K
from skinny_mlx import patch as P
from skinny_mlx.cache import make_prompt_cache
from skinny_mlx.model import PIECES_MIN, PROMPT_MIN, build_model
from skinny_mlx.spec import forward

pytestmark = pytest.mark.gpu


# the small decoders with Gated-DeltaNet heads enough for every linear to be patched (16 rows of b and a)
SMALL = {"tiny-dense": {}, "tiny-hybrid": dict(linear_num_heads=16),
         "tiny-qwen35": dict(linear_num_heads=16, linear_num_key_heads=8)}


def _model(preset):
    model = build_model(preset, **SMALL[preset])
    P.patch_model(model)
    return model


def _state(cache, t):
    sh = cache.shared
    out = [sh.k_all[:, :, :t], sh.vt_all[..., :t]]
    if sh.gdn is not None:
        out += [sh.gdn.state, sh.gdn.conv]
    return out


@pytest.mark.parametrize("preset", list(SMALL))
@pytest.mark.parametrize("t,before", [(17, 0), (33, 40), (63, 0), (80, 0), (129, 0), (143, 17), (333, 100)])
def test_prompt_equals_pieces(preset, t, before):
    model = _model(preset)
    assert not PIECES_MIN <= t < PROMPT_MIN and model._prompt_ok(model._ids([0]))
    ids = torch.randint(0, model.args.vocab_size, (before + t,), generator=torch.Generator().manual_seed(t)).tolist()
    c1, c2 = make_prompt_cache(model), make_prompt_cache(model)
    for c in (c1, c2):
        if before:
            forward(model, ids[:before], c)
    h1, l1 = forward(model, ids[before:], c1)
    assert getattr(c1, "_piece_step", None) is None
    h2 = model._pieces(model._ids(ids[before:]), c2)
    assert torch.equal(h1, h2) and torch.equal(l1, torch.cat([model.logits(h2[i:i + 16]) for i in range(0, t, 16)]))
    for a, b in zip(_state(c1, before + t), _state(c2, before + t)):
        assert torch.equal(a, b)
    # both caches go on alike
    assert c1.attention_offset() == c2.attention_offset() == before + t
    assert torch.equal(forward(model, [7], c1)[1], forward(model, [7], c2)[1])


@pytest.mark.parametrize("t", [64, 70, 79])
@pytest.mark.parametrize("preset", list(SMALL))
def test_a_block_of_four_pieces_equals_them(preset, t):
    """The lengths that Model.hidden leaves to the pieces, as one block."""
    model = _model(preset)
    ids = model._ids(torch.randint(0, model.args.vocab_size, (t,), generator=torch.Generator().manual_seed(t)).tolist())
    c1, c2 = make_prompt_cache(model), make_prompt_cache(model)
    assert torch.equal(model._prompt(ids, c1), model._pieces(ids, c2))
    for a, b in zip(_state(c1, t), _state(c2, t)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("t", [1024 + 9, 1024 + 40])
@pytest.mark.parametrize("preset", ["dense-36", "hybrid-36", "qwen35-4b"])
def test_a_whole_block_of_the_decoders_layers_equals_pieces(preset, t):
    """Four layers of the decoders at their own sizes (so with the tiles of their projections and the MLP's one-launch
    form), past the end of a 1024-token block: a tail run as a step, and a second block."""
    model = build_model(preset, num_hidden_layers=4, vocab_size=1024)
    P.patch_model(model)
    ids = model._ids(torch.randint(0, 1024, (t,), generator=torch.Generator().manual_seed(t)).tolist())
    assert model._prompt_ok(ids)
    c1, c2 = make_prompt_cache(model), make_prompt_cache(model)
    assert torch.equal(model.hidden(ids, c1), model._pieces(ids, c2))
    for a, b in zip(_state(c1, t), _state(c2, t)):
        assert torch.equal(a, b)


def test_prompt_blocks_and_short_tail(monkeypatch):
    import skinny_mlx.model as M

    monkeypatch.setattr(M, "PROMPT_BLOCK", 96)
    model = _model("tiny-hybrid")
    ids = torch.randint(0, model.args.vocab_size, (96 + 96 + 9,), generator=torch.Generator().manual_seed(2)).tolist()
    c1, c2 = make_prompt_cache(model), make_prompt_cache(model)
    h1, _ = forward(model, ids, c1)
    assert torch.equal(h1, model._pieces(model._ids(ids), c2))
    for a, b in zip(_state(c1, len(ids)), _state(c2, len(ids))):
        assert torch.equal(a, b)


@pytest.mark.parametrize("skinny_range", [None, (99, 99)])  # unpatched; patched with the kernels switched off
def test_unpatched_linears_run_once_before_the_pieces_are_captured(skinny_range, monkeypatch):
    import skinny_mlx.graphs as G

    cached = []
    step = G.CapturedStep
    monkeypatch.setattr(G, "CapturedStep", lambda fn, cache, *a, **k: cached.append(cache.attention_offset()) or step(fn, cache, *a, **k))
    model = build_model("tiny-dense")
    if skinny_range:
        P.patch_model(model)
        monkeypatch.setattr(P, "SKINNY_RANGE", skinny_range)
    ids = list(range(70))
    c1, c2 = make_prompt_cache(model), make_prompt_cache(model)
    h = model.hidden(ids, c1)
    assert cached == [16] and torch.equal(h, torch.cat([model.hidden(ids[i:i + 16], c2) for i in range(0, 70, 16)]))


def test_unpatched_and_captured_inputs_keep_the_pieces():
    model = build_model("tiny-dense")
    ids = model._ids(list(range(100)))
    assert not model._prompt_ok(ids)
    P.patch_model(model)
    assert model._prompt_ok(ids) and not model._prompt_ok(ids.cpu())
    hybrid = build_model("tiny-hybrid")  # 2 rows of b and a: those linears stay unpatched
    P.patch_model(hybrid)
    assert not hybrid._prompt_ok(ids)


class _Wrapped(torch.nn.Module):
    """Any other module in the place of one of the model's: here it only hands through."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, *args):
        return self.inner(*args)


def _replace(model, where):
    layer = model.layers[-1]
    parent = {"o_proj": "self_attn", "q_proj": "self_attn", "down_proj": "mlp", "gate_proj": "mlp"}.get(where)
    owner = getattr(layer, parent) if parent else layer
    setattr(owner, where, _Wrapped(getattr(owner, where)))


@pytest.mark.parametrize("t", [20, 90])
@pytest.mark.parametrize("where", ["o_proj", "q_proj", "down_proj", "gate_proj", "mlp", "self_attn"])
def test_a_replaced_module_keeps_the_pieces(where, t):
    model = _model("tiny-dense")
    _replace(model, where)
    ids = torch.randint(0, model.args.vocab_size, (t,), generator=torch.Generator().manual_seed(t)).tolist()
    c1, c2 = make_prompt_cache(model), make_prompt_cache(model)
    assert not model._prompt_ok(model._ids(ids))
    h, _ = forward(model, ids, c1)
    assert torch.equal(h, torch.cat([model.hidden(ids[i:i + 16], c2) for i in range(0, t, 16)]))


@pytest.mark.parametrize("t", [20, 90])
def test_a_replaced_linear_of_another_library(t):
    model = _model("tiny-dense")
    down = torch.nn.Linear(512, 256, bias=False, device=model.device, dtype=torch.bfloat16)
    model.layers[0].mlp.down_proj = down
    ids = list(range(t))
    c1, c2 = make_prompt_cache(model), make_prompt_cache(model)
    with torch.no_grad():
        h = model.hidden(ids, c1)
        assert torch.equal(h, torch.cat([model.hidden(ids[i:i + 16], c2) for i in range(0, t, 16)]))


@pytest.mark.parametrize("how", ["hook", "pre-hook", "any module's hook", "forward", "class forward", "mixer"])
def test_hooks_and_replaced_methods_see_every_step(how, monkeypatch):
    """33 tokens: three passes, each through the hook or method of a layer's MLP (the mixer's for "mixer")."""
    from skinny_mlx.model import MLP

    model = _model("tiny-dense")
    layer, seen = model.layers[0], []
    mlp, handle = layer.mlp, None
    note = lambda *a: seen.append(1) if a[0] is mlp else None
    if how == "hook":
        mlp.register_forward_hook(note)
    elif how == "pre-hook":
        mlp.register_forward_pre_hook(note)
    elif how == "any module's hook":
        handle = torch.nn.modules.module.register_module_forward_hook(note)
    elif how == "forward":
        old = mlp.forward
        mlp.forward = lambda x: (seen.append(1), old(x))[1]
    elif how == "class forward":
        plain = MLP.forward
        monkeypatch.setattr(MLP, "forward", lambda self, x: (note(self), plain(self, x))[1])
    else:
        old = layer.mixer
        layer.mixer = lambda *a: (seen.append(1), old(*a))[1]
    try:
        model.hidden(list(range(33)), make_prompt_cache(model))
    finally:
        if handle is not None:
            handle.remove()
    assert len(seen) == 3


@pytest.mark.parametrize("t,block", [(18, False), (22, True), (32, True)])
def test_pieces_outside_the_skinny_range_keep_their_route(t, block, monkeypatch):
    """With the reference's range of 6 to 16 rows (its patch.py:22) a last piece of two tokens is multiplied
    unpatched, as a step of two is; whole pieces go through the kernels either way."""
    monkeypatch.setattr(P, "SKINNY_RANGE", (6, 16))
    model = _model("tiny-dense")
    ids = torch.randint(0, model.args.vocab_size, (t,), generator=torch.Generator().manual_seed(t)).tolist()
    assert model._prompt_ok(model._ids(ids)) == block
    c1, c2 = make_prompt_cache(model), make_prompt_cache(model)
    h = model.hidden(ids, c1)
    assert torch.equal(h, torch.cat([model.hidden(ids[i:i + 16], c2) for i in range(0, t, 16)]))


@pytest.mark.parametrize("preset,fuse_conv", [(p, True) for p in SMALL] + [("tiny-hybrid", False)])
def test_a_prompt_leaves_nothing_behind(preset, fuse_conv):
    """What is allocated after a prompt is what was before it (a fused projection's cached result would be 500 rows
    of q, k and v a layer)."""
    model = _model(preset)
    for layer in model.layers:
        if layer.is_linear:
            layer.linear_attn.fuse_conv = fuse_conv
    cache = make_prompt_cache(model)
    model.hidden(list(range(20)), cache)
    gc.collect()
    before = torch.cuda.memory_allocated()
    model.hidden([i % 999 for i in range(480)], cache)
    assert torch.cuda.memory_allocated() <= before


def test_a_dropped_result_is_still_returned():
    """Another thread's prompt may drop a projection's kept result between its computation and its return."""
    class Dropping(P._Projection):
        def __init__(self):
            self.forget()

        def __setattr__(self, name, value):
            object.__setattr__(self, name, None)

        def _compute(self, x):
            return x + 1

    x = torch.ones(4)
    assert torch.equal(Dropping().output(x), x + 1)


@pytest.mark.parametrize("preset,field,value", [("tiny-dense", "rope_theta", 5e5), ("tiny-qwen35", "rope_theta", 5e5),
                                                ("tiny-qwen35", "rope_dim", 32)])
def test_a_cache_of_another_rope_is_refused(preset, field, value):
    """A long input is refused as its 16-token steps are."""
    model = _model(preset)
    for t in (16, 100):
        cache = make_prompt_cache(model)
        setattr(cache.shared, field, value)
        with pytest.raises(ValueError, match="cache RoPE table"):
            forward(model, list(range(t)), cache)


@pytest.mark.parametrize("maxlen,past", [(1024, 0), (1024, 250), (8192, 4300), (17408, 16500)])  # one-, four- and eight-wave merges
@pytest.mark.parametrize("layout", ["dense", "general"])
def test_prompt_attention_equals_steps(dev, layout, maxlen, past):
    hq, hkv, d = (8, 2, 128) if layout == "dense" else (4, 1, 256)
    t = 150
    g = torch.Generator(device=dev).manual_seed(maxlen + past)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev).to(torch.bfloat16)
    cols = (hq + 2 * hkv) * d if layout == "dense" else (2 * hq + 2 * hkv) * d
    qkv, k0, v0, qn, kn = rnd(t, cols), rnd(hkv, maxlen, d), rnd(hkv, d, maxlen), rnd(d), rnd(d)
    pos = torch.tensor([past], dtype=torch.int32, device=dev)
    res = []
    for prompt in (True, False):
        k, vt = k0.clone(), v0.clone()
        if layout == "dense":
            table = K.rope_table(1e6, maxlen, dev)
            if prompt:
                o = K.attention_prompt(qkv, hq, hkv, d, qn, kn, 1e-6, table, pos, past + t, k, vt, d ** -0.5)
            else:
                ws = K.attn_workspace(hkv, maxlen, dev)
                o = torch.cat([K.attention_fused(qkv[i:i + 16], hq, hkv, d, qn, kn, 1e-6, table, pos + i, k, vt, d ** -0.5, ws)
                               for i in range(0, t, 16)])
        else:
            table = K.rope_table_dim(1e7, 64, maxlen, dev)
            args = (hq, hkv, d, 2 * d, 2 * hq * d, 2 * hq * d + hkv * d, d, qn, kn, 1e-6, 64, table)
            if prompt:
                o = K.attention_general_prompt(qkv, *args, pos, past + t, k, vt, d ** -0.5)
            else:
                ws = K.attn_general_workspace(hq, hkv, d, maxlen, dev)
                o = torch.cat([K.attention_general(qkv[i:i + 16], *args, pos + i, k, vt, d ** -0.5, ws)
                               for i in range(0, t, 16)])
        res.append((o, k, vt))
    for a, b in zip(*res):
        assert torch.equal(a, b)


def test_prompt_tokens_past_the_cache_are_dropped(dev):
    """A device position that leaves slots for 20 of 40 tokens (no caller of the package lets it): the others land
    nowhere, neither in the next head's rows nor behind the last head's. The RoPE table covers the positions."""
    hq, hkv, d, t, maxlen, guard = 8, 2, 128, 40, 512, 1 << 14
    past = maxlen - 20
    g = torch.Generator(device=dev).manual_seed(8)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev).to(torch.bfloat16)
    qkv, table = rnd(t, (hq + 2 * hkv) * d), K.rope_table(1e6, maxlen + 128, dev)
    k0, v0 = rnd(hkv * maxlen * d + guard), rnd(hkv * maxlen * d + guard)
    k, vt = k0.clone(), v0.clone()
    kc, vc = k[:-guard].view(hkv, maxlen, d), vt[:-guard].view(hkv, d, maxlen)
    pos = torch.tensor([past], dtype=torch.int32, device=dev)
    K.attention_prompt(qkv, hq, hkv, d, None, None, 1e-6, table, pos, maxlen, kc, vc, d ** -0.5)
    assert torch.equal(k[-guard:], k0[-guard:]) and torch.equal(vt[-guard:], v0[-guard:])
    assert torch.equal(kc[:, :past], k0[:-guard].view(hkv, maxlen, d)[:, :past])
    want = v0[:-guard].view(hkv, d, maxlen).clone()
    want[:, :, past:] = qkv[:20, (hq + hkv) * d:].view(20, hkv, d).permute(1, 2, 0)
    assert torch.equal(vc, want)


@pytest.mark.parametrize("past,token", [(0, 99), (100, 20), (250, 149), (120, 16)])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("layout", ["dense", "general"])
def test_an_infinite_value_reaches_no_token_before_its_step(dev, layout, bad, past, token):
    """A token whose values are no numbers: the rows of the pieces before it are what 16-token steps give."""
    hq, hkv, d, t, maxlen = (8, 2, 128, 150, 512) if layout == "dense" else (4, 1, 256, 150, 512)
    g = torch.Generator(device=dev).manual_seed(past)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev).to(torch.bfloat16)
    if layout == "dense":
        table, ws = K.rope_table(1e6, maxlen, dev), K.attn_workspace(hkv, maxlen, dev)
        lay, first, step = (), K.attention_prompt, K.attention_fused
        qkv = rnd(t, (hq + 2 * hkv) * d)
    else:
        table, ws = K.rope_table_dim(1e7, 64, maxlen, dev), K.attn_general_workspace(hq, hkv, d, maxlen, dev)
        lay, first, step = (d, hq * d, (hq + hkv) * d, None), K.attention_general_prompt, K.attention_general
        qkv = rnd(t, (hq + 2 * hkv) * d)
    qkv[token, (hq + hkv) * d:] = bad
    k0, v0 = rnd(hkv, maxlen, d), rnd(hkv, d, maxlen)
    pos = torch.tensor([past], dtype=torch.int32, device=dev)
    tail = () if layout == "dense" else (64,)
    k, vt = k0.clone(), v0.clone()
    out = first(qkv, hq, hkv, d, *lay, None, None, 1e-6, *tail, table, pos, past + t, k, vt, d ** -0.5)
    k2, vt2 = k0.clone(), v0.clone()
    ref = torch.cat([step(qkv[i:i + 16], hq, hkv, d, *lay, None, None, 1e-6, *tail, table, pos + i, k2, vt2, d ** -0.5, ws)
                     for i in range(0, t, 16)])
    piece = token // 16 * 16
    assert ref[:piece].isfinite().all() and torch.equal(out[:piece], ref[:piece])
    assert torch.equal(out.isnan(), ref.isnan())


def test_prompt_attention_in_several_launches(dev):
    """A workspace of one group of pieces (four) instead of all ten: three launches, the same bits."""
    from skinny_mlx import _lib

    hq, hkv, d, t, maxlen, past = 8, 2, 128, 150, 512, 130
    g = torch.Generator(device=dev).manual_seed(5)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev).to(torch.bfloat16)
    qkv, k0, v0 = rnd(t, (hq + 2 * hkv) * d), rnd(hkv, maxlen, d), rnd(hkv, d, maxlen)
    pos = torch.tensor([past], dtype=torch.int32, device=dev)
    table = K.rope_table(1e6, maxlen, dev)
    k, vt = k0.clone(), v0.clone()
    ref = K.attention_prompt(qkv, hq, hkv, d, None, None, 1e-6, table, pos, past + t, k, vt, d ** -0.5)
    L = _lib.lib()
    one = int(L.skinny_attn_prompt_workspace_bytes(t, hq, hkv, past + t))
    query = ((t * hq * d * 2) + 255) // 256 * 256
    ws = torch.empty(query + (one - query) * 4 // 10, dtype=torch.uint8, device=dev)
    out, k2, vt2 = torch.empty_like(ref), k0.clone(), v0.clone()
    _lib.check(L.skinny_attention_prompt_bf16(
        qkv.data_ptr(), qkv.stride(0), t, hq, hkv, d, None, None, 1e-6, table.data_ptr(), maxlen, pos.data_ptr(), past + t,
        k2.data_ptr(), vt2.data_ptr(), maxlen, d ** -0.5, ws.data_ptr(), ws.numel(), out.data_ptr(),
        _lib.stream_of(qkv)), "prompt")
    assert torch.equal(out, ref) and torch.equal(k2, k) and torch.equal(vt2, vt)


@pytest.mark.parametrize("h,hk", [(4, 4), (4, 2)])
@pytest.mark.parametrize("t", [17, 33, 130, 256, 257, 530])  # gates come in blocks of 256
def test_long_conv_and_recurrence_equal_blocks(dev, h, hk, t):
    c = 2 * hk * 128 + h * 128
    g = torch.Generator(device=dev).manual_seed(t + h)
    x = torch.randn((t, c), generator=g, device=dev).to(torch.bfloat16)
    ab = torch.randn((t, 2 * h), generator=g, device=dev).to(torch.bfloat16)
    w = torch.randn((c, 4), generator=g, device=dev).to(torch.bfloat16)
    A, dtb = torch.rand((h,), generator=g, device=dev), torch.rand((h,), generator=g, device=dev)
    conv0 = torch.randn((3, c), generator=g, device=dev).to(torch.bfloat16)
    s0 = torch.randn((h, 128, 128), generator=g, device=dev) * 0.1
    res = []
    for step in (t, 16):
        conv, s, xs, ys = conv0.clone(), s0.clone(), [], []
        rec = torch.empty((t, h, 128, 128), device=dev)
        for i in range(0, t, step):
            xs.append(K.gdn_conv_silu(x[i:i + step], conv, w, None))
            ys.append(K.gdn_recurrence(xs[-1], ab[i:i + step, :h], ab[i:i + step, h:], A, dtb, s,
                                       rec[i:i + step] if t % 2 else None, h, 128, 128, n_key_heads=hk))
        res.append((torch.cat(xs), torch.cat(ys), conv, s) + ((rec,) if t % 2 else ()))
    for a, b in zip(*res):
        assert torch.equal(a, b)
