"""What a user of this package has the GPU do, as timed cases: single projections, the MLP's gate|up,
the attention of a step, the Gated-DeltaNet mixer's input side, whole decode and verify steps, and
prompts. Sizes are the package's own decoders (model.PRESETS: dense-36, hybrid-36, qwen35-4b).

Token counts go from the one token of a decode step over the 2 to 16 of a verify step to prompts of
some hundred tokens; cached contexts from a hundred to tens of thousands of positions.

listed() and draw(rng) give cases as plain dicts; prepare(case, seed) what a program holds before the
call (packed weights, caches, a captured step); run(state) is one pass; exact(case, seed) the same
outputs in 64 bits by plain torch.
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "skinny-mlx_amd"))

DEV = "cuda:0"
BF16 = torch.bfloat16

# (K, N) of the decoders' plain projections: o_proj, down, fused q|k|v, the GDN out_proj, Qwen3.5's
# fused q|gate|k|v and down, the pruned draft head, the two full heads.
LINEARS = [(4096, 2560), (9728, 2560), (2560, 6144), (2048, 2560), (2560, 10240), (9216, 2560), (2560, 32768),
           (2560, 151936), (2560, 248320)]
HEADS = {151936, 248320}
GLUS = [(2560, 9728), (2560, 9216)]
# attention layouts: (query heads, kv heads, head dim, rotary dim, output gate)
LAYOUTS = {"dense": (32, 8, 128, 128, False), "qwen35": (16, 4, 256, 64, True)}
# Gated-DeltaNet mixers: (value heads, key heads, projection columns)
MIXERS = {"hybrid": (16, 16, 8224), "qwen35": (32, 16, 12352)}


def listed():
    return [
        # one decoded token through one projection, called by itself: the smallest call
        dict(name="linear_o_m1", op="linear", m=1, k=4096, n=2560),
        # the head of a verify step over 8 tokens: 221 MB of weights read once
        dict(name="linear_head_m8", op="linear", m=8, k=2560, n=151936),
        # a short prompt of an odd length through the fused q|k|v projection
        dict(name="linear_qkv_m77", op="linear", m=77, k=2560, n=6144),
        # a long prompt's down projection
        dict(name="linear_down_m1024", op="linear", m=1024, k=9728, n=2560),
        # a prompt's MLP front half: gate|up with SwiGLU
        dict(name="glu_m501", op="glu", m=501, k=2560, f=9728),
        # the attention of a verify step (12 layers of one captured step, each on its own cache)
        dict(name="attn_verify_m8", op="attn", layout="dense", m=8, past=2040, layers=12),
        # one token's attention over a long context
        dict(name="attn_long_m1", op="attn", layout="dense", m=1, past=32768, layers=4),
        # Qwen3.5's attention layout (256-dim heads, partial rotation, output gate), a 4-token verify
        dict(name="attn_qwen35_m4", op="attn", layout="qwen35", m=4, past=5003, layers=8),
        # the Gated-DeltaNet input side of a verify step: projection + conv, recurrence keeping every
        # token's state for the rollback, gated norm (8 layers of one captured step)
        dict(name="gdn_verify_m8", op="gdn", mixer="hybrid", m=8, layers=8),
        # a whole verify step of the dense decoder over 2048 cached tokens
        dict(name="step_dense_m8", op="step", preset="dense-36", m=8, past=2048, tree=False),
        # a whole decode step (one token) of the Qwen3.5-4B-shaped decoder
        dict(name="step_qwen35_m1", op="step", preset="qwen35-4b", m=1, past=512, tree=False),
        # a prompt through the hybrid decoder, from an empty cache to the logits
        dict(name="prompt_hybrid_t509", op="prompt", preset="hybrid-36", t=509),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    op = rng.choice(["linear", "linear", "glu", "attn", "attn", "gdn", "step", "prompt"])
    if op == "linear":
        k, n = rng.choice(LINEARS)
        return dict(op=op, m=_log_int(rng, 1, 64 if n in HEADS else 1024), k=k, n=n)
    if op == "glu":
        k, f = rng.choice(GLUS)
        return dict(op=op, m=_log_int(rng, 1, 1024), k=k, f=f)
    if op == "attn":
        return dict(op=op, layout=rng.choice(sorted(LAYOUTS)), m=_log_int(rng, 1, 16), past=_log_int(rng, 100, 32768),
                    layers=rng.randint(2, 6))
    if op == "gdn":
        return dict(op=op, mixer=rng.choice(sorted(MIXERS)), m=_log_int(rng, 1, 16), layers=rng.randint(4, 10))
    if op == "step":
        m = _log_int(rng, 1, 16)
        return dict(op=op, preset=rng.choice(["dense-36", "hybrid-36", "qwen35-4b"]), m=m,
                    past=_log_int(rng, 100, 3900), tree=m >= 4 and rng.random() < 0.4)
    return dict(op=op, preset=rng.choice(["dense-36", "hybrid-36", "qwen35-4b"]), t=_log_int(rng, 20, 500))


# --- inputs -------------------------------------------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _weights(n, k, g):
    """MLX W4 g64 weights with dequantised values of std ~1/sqrt(K), as a checkpoint's are."""
    w = torch.randint(-2 ** 31, 2 ** 31, (n, k // 8), dtype=torch.int32, generator=g, device=DEV)
    s = (torch.randn((n, k // 64), generator=g, device=DEV) / (3.7 * math.sqrt(k))).abs().to(BF16)
    b = (s.float() * -8.0 + torch.randn((n, k // 64), generator=g, device=DEV) * 0.02 / math.sqrt(k)).to(BF16)
    return w, s, b


def _rows(m, k, g, std=1.0):
    return (torch.randn((m, k), generator=g, device=DEV) * std).to(BF16)


def _attn_inputs(case, seed):
    g = _gen(seed)
    hq, hkv, d, rd, gate = LAYOUTS[case["layout"]]
    m, past, layers = case["m"], case["past"], case["layers"]
    maxlen = -(-(past + m) // 256) * 256
    k = torch.randn((layers, hkv, maxlen, d), generator=g, device=DEV).to(BF16)
    vt = torch.randn((layers, hkv, d, maxlen), generator=g, device=DEV).to(BF16)
    cols = hq * d * (2 if gate else 1) + 2 * hkv * d
    qkv = [_rows(m, cols, g) for _ in range(layers)]
    qn = (torch.randn((layers, d), generator=g, device=DEV) * 0.02 + 1).to(BF16)
    kn = (torch.randn((layers, d), generator=g, device=DEV) * 0.02 + 1).to(BF16)
    return k, vt, qkv, qn, kn, maxlen


def _gdn_inputs(case, seed):
    g = _gen(seed)
    h, hk, n = MIXERS[case["mixer"]]
    c = 2 * hk * 128 + h * 128
    out = []
    for _ in range(case["layers"]):
        out.append(dict(
            x=_rows(case["m"], 2560, g), w=_weights(n, 2560, g),
            conv_w=((torch.rand((c, 4), generator=g, device=DEV) - 0.5)).to(BF16), conv=_rows(3, c, g),
            A_log=torch.log(torch.rand((h,), generator=g, device=DEV) * 15.0 + 1.0),
            dt_bias=torch.rand((h,), generator=g, device=DEV) * 2.0 - 1.0,
            norm=(torch.randn((128,), generator=g, device=DEV) * 0.02 + 1).to(BF16),
            state=torch.randn((h, 128, 128), generator=g, device=DEV) * 0.1))
    return out, h, hk, c


def _captured(fn):
    from skinny_mlx.graphs import capture_graph

    return capture_graph(fn)


def prepare(case, seed):
    op = case["op"]
    if op in ("linear", "glu"):
        from skinny_mlx import qmm as Q

        g = _gen(seed)
        n = case["n"] if op == "linear" else 2 * case["f"]
        w = _weights(n, case["k"], g)
        packed = (Q.repack_for_skinny if op == "linear" else Q.repack_gate_up)(*w)
        return dict(op=op, fn=Q.skinny_qmm if op == "linear" else Q.skinny_glu, x=_rows(case["m"], case["k"], g), w=packed)
    if op == "attn":
        from skinny_mlx import kernels as K

        hq, hkv, d, rd, gate = LAYOUTS[case["layout"]]
        k, vt, qkv, qn, kn, maxlen = _attn_inputs(case, seed)
        m, past, layers = case["m"], case["past"], case["layers"]
        pos = torch.tensor([past], dtype=torch.int32, device=DEV)
        if case["layout"] == "dense":
            table, ws = K.rope_table(1e6, maxlen, DEV), K.attn_workspace(hkv, maxlen, DEV)

            def layer(i):
                return K.attention_fused(qkv[i], hq, hkv, d, qn[i], kn[i], 1e-6, table, pos, k[i], vt[i], d ** -0.5, ws)
        else:
            table, ws = K.rope_table_dim(1e7, rd, maxlen, DEV), K.attn_general_workspace(hq, hkv, d, maxlen, DEV)

            def layer(i):
                return K.attention_general(qkv[i], hq, hkv, d, 2 * d, hq * 2 * d, hq * 2 * d + hkv * d, d, qn[i], kn[i],
                                           1e-6, rd, table, pos, k[i], vt[i], d ** -0.5, ws)
        torch.cuda.synchronize()
        graph, outs = _captured(lambda: [layer(i) for i in range(layers)])
        return dict(op=op, graph=graph, outs=outs + [k[:, :, past:past + m], vt[:, :, :, past:past + m]],
                    hold=(k, vt, qkv, qn, kn, pos, table, ws))
    if op == "gdn":
        from skinny_mlx import kernels as K
        from skinny_mlx import qmm as Q

        layers, h, hk, c = _gdn_inputs(case, seed)
        m, L = case["m"], case["layers"]
        states = torch.zeros((L, m, h, 128, 128), dtype=torch.float32, device=DEV)
        window = torch.zeros((L, m + 3, c), dtype=BF16, device=DEV)
        for l in layers:
            l["packed"] = Q.repack_for_skinny(*l.pop("w"))

        def layer(i):
            l = layers[i]
            y = Q.skinny_qmm_conv(l["x"], l["packed"], c, l["conv"], l["conv_w"], window[i])
            z, b, a = y[:, c:c + h * 128], y[:, c + h * 128:c + h * 128 + h], y[:, c + h * 128 + h:c + h * 128 + 2 * h]
            r = K.gdn_recurrence(y[:, :c], b, a, l["A_log"], l["dt_bias"], l["state"], states[i], h, 128, 128,
                                 n_key_heads=hk)
            return K.gated_rmsnorm(r, z, l["norm"], 1e-6)

        torch.cuda.synchronize()
        graph, outs = _captured(lambda: [layer(i) for i in range(L)])
        return dict(op=op, graph=graph, outs=outs + [l["state"] for l in layers] + [states, window],
                    hold=(layers, states, window))
    if op == "step":
        return _prepare_step(case, seed)
    from skinny_mlx.model import build_model
    from skinny_mlx.patch import patch_model

    model = build_model(case["preset"], device=DEV, seed=int(seed) & 0x7FFFFFFF)
    patch_model(model)
    ids = torch.randint(0, model.args.vocab_size, (case["t"],), generator=_gen(seed + 1), device=DEV).tolist()
    return dict(op=op, model=model, ids=ids)


def _prepare_step(case, seed):
    from skinny_mlx.cache import KVCache, make_prompt_cache
    from skinny_mlx.graphs import CapturedStep
    from skinny_mlx.model import build_model
    from skinny_mlx.patch import patch_model
    from skinny_mlx.rollback import HybridRollback
    from skinny_mlx.spec import forward
    from skinny_mlx.tree import DraftTree

    model = build_model(case["preset"], device=DEV, seed=int(seed) & 0x7FFFFFFF)
    patch_model(model)
    g = _gen(seed + 1)
    m, past = case["m"], case["past"]
    cache = make_prompt_cache(model)
    sh = cache.shared
    sh.k_all[:, :, :past].normal_(generator=g)
    sh.vt_all[..., :past].normal_(generator=g)
    if sh.gdn is not None:
        sh.gdn.state.normal_(0.0, 0.1, generator=g)
        sh.gdn.conv.normal_(generator=g)
    kv = [c for c in cache if isinstance(c, KVCache)]
    for c in kv:
        c.offset = past
    ids = torch.randint(0, model.args.vocab_size, (m,), generator=g, device=DEV, dtype=torch.int32)
    # a verify pass of a hybrid decoder records what its rollback needs, a decode step does not
    record = sh.gdn is not None and m > 1
    tree = DraftTree.from_branching((4, 2, 1), m, model.device) if case["tree"] else None
    if record:
        HybridRollback.for_model(model).record()
    step = CapturedStep(lambda: forward(model, ids, cache, tree), cache, m, recorded=m if record else None)
    model.recorder.recording = False
    return dict(op="step", step=step, kv=kv, m=m, gdn=sh.gdn, past=past, sh=sh, hold=(model, cache, ids, tree))


# --- one pass -----------------------------------------------------------------------------------

def run(state):
    op = state["op"]
    if op == "linear":
        return state["fn"](state["x"], state["w"])
    if op == "glu":
        return state["fn"](state["x"], state["w"], swiglu=True)
    if op in ("attn", "gdn"):
        state["graph"].replay()
        return state["outs"]
    if op == "step":
        hidden, logits = state["step"]()
        for c in state["kv"]:  # the next pass starts from the same cached length, as after a rejected draft
            c.trim(state["m"])
        p, m, sh = state["past"], state["m"], state["sh"]
        out = [hidden, logits, sh.k_all[:, :, p:p + m], sh.vt_all[..., p:p + m]]
        return out + ([sh.gdn.state, sh.gdn.conv] if state["gdn"] is not None else [])
    from skinny_mlx.cache import make_prompt_cache
    from skinny_mlx.spec import forward

    cache = make_prompt_cache(state["model"])
    hidden, logits = forward(state["model"], state["ids"], cache)
    t, sh = len(state["ids"]), cache.shared
    out = [hidden, logits, sh.k_all[:, :, :t], sh.vt_all[..., :t]]
    return out + ([sh.gdn.state, sh.gdn.conv] if sh.gdn is not None else [])


# --- what a pass cannot do without ---------------------------------------------------------------

def _w4_bytes(n, k):
    return n * k // 2 + 4 * n * (k // 64)


def _decoder_work(preset, tokens, past, prompt):
    """Bytes and flops of one forward over `tokens` new tokens after `past` cached ones."""
    from skinny_mlx.model import PRESETS

    a = PRESETS[preset]
    H, V, F = a.hidden_size, a.vocab_size, a.intermediate_size
    nbytes, flops = _w4_bytes(V, H) + tokens * (2 * H + 2 * V + 2 * H), 2 * tokens * V * H
    for i in range(a.num_hidden_layers):
        shapes = [(2 * F, H), (H, F)]
        if a.is_linear(i):
            h, hk = a.linear_num_heads, a.gdn_key_heads
            c = 2 * hk * 128 + h * 128
            shapes += [(c + h * 128 + 2 * h, H), (H, h * 128)]
            nbytes += 2 * h * 128 * 128 * 4 + 2 * 3 * c * 2
            if tokens > 1 and not prompt:
                nbytes += tokens * h * 128 * 128 * 4  # every token's state, for the rollback
            flops += tokens * h * 8 * 128 * 128
        else:
            hq, hkv, d = a.num_attention_heads, a.num_key_value_heads, a.head_dim
            shapes += [((hq * (2 if a.attn_output_gate else 1) + 2 * hkv) * d, H), (H, hq * d)]
            nbytes += 2 * hkv * d * 2 * (past + tokens)
            flops += 4 * hq * d * tokens * (past + (tokens + 1) // 2)
        for n, k in shapes:
            nbytes += _w4_bytes(n, k)
            flops += 2 * tokens * n * k
    return dict(bytes=nbytes, flops=flops)


def work(case):
    op = case["op"]
    if op in ("linear", "glu"):
        m, k = case["m"], case["k"]
        n = case["n"] if op == "linear" else 2 * case["f"]
        return dict(bytes=_w4_bytes(n, k) + 2 * m * k + 2 * m * (n if op == "linear" else n // 2), flops=2 * m * n * k)
    if op == "attn":
        hq, hkv, d, rd, gate = LAYOUTS[case["layout"]]
        m, past, L = case["m"], case["past"], case["layers"]
        cols = hq * d * (2 if gate else 1) + 2 * hkv * d
        return dict(bytes=L * (2 * hkv * d * 2 * (past + m) + 2 * m * cols + 2 * m * hq * d),
                    flops=L * 4 * hq * d * m * (past + m))
    if op == "gdn":
        h, hk, n = MIXERS[case["mixer"]]
        m, L, c = case["m"], case["layers"], 2 * hk * 128 + h * 128
        st = h * 128 * 128 * 4
        return dict(bytes=L * (_w4_bytes(n, 2560) + 2 * m * 2560 + (2 + m) * st + 2 * m * h * 128 + 2 * (m + 9) * c),
                    flops=L * (2 * m * n * 2560 + m * h * 8 * 128 * 128))
    if op == "step":
        return _decoder_work(case["preset"], case["m"], case["past"], False)
    return _decoder_work(case["preset"], case["t"], 0, True)


def tolerance(case):
    """About four times the distance two correct paths were measured at: the single layers against
    exact() (linear 0.0017, glu 0.0031, attention 0.0038, mixer 0.0051 relative in norm: bf16 outputs,
    and bf16 q, k, P, conv output and gate inside); whole decoders patched against unpatched (0.0015
    in hidden states, logits, keys and values, 0.0021 with single values 0.053 apart in the mixer states)."""
    return {"linear": dict(rel=0.007, max=0.04), "glu": dict(rel=0.0125, max=0.1), "attn": dict(rel=0.015, max=0.1),
            "gdn": dict(rel=0.02, max=0.2), "step": dict(rel=0.009, max=0.22), "prompt": dict(rel=0.009, max=0.22)}[case["op"]]


# --- the same in 64 bits --------------------------------------------------------------------------

def _dequant64(w, s, b, lo=0, hi=None):
    w, s, b = w[lo:hi], s[lo:hi], b[lo:hi]
    n, kp = w.shape
    q = torch.stack([(w >> (4 * i)) & 15 for i in range(8)], dim=-1).reshape(n, kp * 8).double()
    return q * s.double().repeat_interleave(64, 1) + b.double().repeat_interleave(64, 1)


def _matmul64(x, w, s, b):
    out = torch.empty((x.shape[0], w.shape[0]), dtype=torch.float64, device=x.device)
    for lo in range(0, w.shape[0], 16384):
        hi = min(lo + 16384, w.shape[0])
        out[:, lo:hi] = x.double() @ _dequant64(w, s, b, lo, hi).t().contiguous()
    return out


def _rms64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, pos, theta, rd):
    """Rotate-half RoPE over the first rd dims; x [T, heads, D], pos [T]."""
    half = rd // 2
    freq = theta ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / rd)
    ang = pos.double()[:, None] * freq
    c, s = ang.cos()[:, None, :], ang.sin()[:, None, :]
    a, b = x[..., :half], x[..., half:rd]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., rd:]], -1)


def exact(case, seed):
    op = case["op"]
    if op in ("linear", "glu"):
        g = _gen(seed)
        n = case["n"] if op == "linear" else 2 * case["f"]
        w = _weights(n, case["k"], g)
        y = _matmul64(_rows(case["m"], case["k"], g), *w)
        if op == "linear":
            return y
        gate, up = y[:, :case["f"]], y[:, case["f"]:]
        return gate * torch.sigmoid(gate) * up
    if op == "attn":
        hq, hkv, d, rd, gate = LAYOUTS[case["layout"]]
        k, vt, qkv, qn, kn, maxlen = _attn_inputs(case, seed)
        m, past = case["m"], case["past"]
        theta = 1e6 if case["layout"] == "dense" else 1e7
        pos = torch.arange(past, past + m, device=DEV)
        outs, new_k, new_v = [], [], []
        for i in range(case["layers"]):
            r = qkv[i].double()
            qs = 2 * d if gate else d
            q = r[:, :hq * qs].reshape(m, hq, qs)
            gt = q[..., d:] if gate else None
            kk, vv = r[:, hq * qs:].reshape(m, 2, hkv, d).unbind(1)
            q = _rope64(_rms64(q[..., :d], qn[i], 1e-6), pos, theta, rd)
            kk = _rope64(_rms64(kk, kn[i], 1e-6), pos, theta, rd)
            keys = torch.cat([k[i, :, :past].double(), kk.transpose(0, 1)], 1)            # [hkv, L, d]
            vals = torch.cat([vt[i, :, :, :past].double().transpose(1, 2), vv.transpose(0, 1)], 1)
            qg = q.reshape(m, hkv, hq // hkv, d).permute(1, 0, 2, 3).reshape(hkv, -1, d)
            sc = (qg @ keys.transpose(1, 2).contiguous()) * d ** -0.5
            t = torch.arange(m, device=DEV).repeat_interleave(hq // hkv)
            sc = sc.masked_fill(torch.arange(past + m, device=DEV)[None, :] > past + t[:, None], float("-inf"))
            o = (torch.softmax(sc, -1) @ vals).reshape(hkv, m, hq // hkv, d).permute(1, 0, 2, 3).reshape(m, hq, d)
            if gate:
                o = o * torch.sigmoid(gt)
            outs.append(o.reshape(m, hq * d))
            new_k.append(kk.transpose(0, 1))
            new_v.append(vv.permute(1, 2, 0))
        return outs + [torch.stack(new_k), torch.stack(new_v)]
    if op == "gdn":
        layers, h, hk, c = _gdn_inputs(case, seed)
        m = case["m"]
        outs, last, states, window = [], [], [], []
        for l in layers:
            y = _matmul64(l["x"], *l["w"])
            seq = torch.cat([l["conv"].double(), y[:, :c]])
            window.append(seq)
            cv = sum(seq[j:j + m] * l["conv_w"][:, j].double() for j in range(4))
            cv = cv * torch.sigmoid(cv)
            q, k = cv[:, :hk * 128].reshape(m, hk, 128), cv[:, hk * 128:2 * hk * 128].reshape(m, hk, 128)
            v = cv[:, 2 * hk * 128:].reshape(m, h, 128)
            q = q * torch.rsqrt(q.square().sum(-1, keepdim=True) + 1e-6) * 128 ** -0.5
            k = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + 1e-6)
            q, k = q.repeat_interleave(h // hk, 1), k.repeat_interleave(h // hk, 1)
            z = y[:, c:c + h * 128].reshape(m, h, 128)
            beta = torch.sigmoid(y[:, c + h * 128:c + h * 128 + h])
            a = y[:, c + h * 128 + h:c + h * 128 + 2 * h] + l["dt_bias"].double()
            decay = torch.exp(-torch.exp(l["A_log"].double()) * torch.nn.functional.softplus(a))
            s = l["state"].double()
            ys, ss = [], []
            for t in range(m):
                s = s * decay[t][:, None, None]
                delta = beta[t][:, None] * (v[t] - (s * k[t][:, None, :]).sum(-1))
                s = s + delta[:, :, None] * k[t][:, None, :]
                ys.append((s * q[t][:, None, :]).sum(-1))
                ss.append(s)
            o = _rms64(torch.stack(ys), l["norm"], 1e-6) * z * torch.sigmoid(z)
            outs.append(o.reshape(m, h * 128))
            last.append(s)
            states.append(torch.stack(ss))
        return outs + last + [torch.stack(states), torch.stack(window)]
    return None
