"""Attention steps of few query rows (one wave per chunk, fragments straight from memory) give each token
bitwise what a 16-token step over staged chunks gives it, and leave the same cache rows: chains and draft
trees, new tokens inside a chunk and across a chunk edge, contexts below one chunk to several merge blocks,
one, two and four chunks per workgroup."""

import pytest
import torch

from skinny_mlx import kernels as K
from skinny_mlx.tree import DraftTree

pytestmark = pytest.mark.gpu

# (kv heads, cache slots, cached tokens): the dense layout staged; chunks x heads <= 512, <= 1024, past it; long caches
# filled so far that a workgroup takes one chunk (general layouts: staged up to 256 chunks in all), two and four;
# workgroups dealt to the heads: the last chunk's edge, an odd count of heads, a full cache
CASES = [(2, 1024, 100), (2, 2048, 0), (2, 2048, 100), (2, 2048, 250), (8, 8192, 5000), (8, 12288, 12200), (8, 33024, 32765),
         (8, 33024, 60), (8, 33024, 2040), (8, 33024, 4090), (8, 33024, 8250), (8, 33024, 16700), (2, 33024, 8180),
         (3, 4096, 4070), (8, 4096, 3960), (1, 33024, 8300), (3, 33024, 32990)]


def _call(layout, rnd, dev, hkv, maxlen):
    if layout == "dense":
        hq, d = 4 * hkv, 128
        table, ws = K.rope_table(1e6, maxlen, dev), K.attn_workspace(hkv, maxlen, dev)
        qn, kn = rnd(d), rnd(d)

        def call(qkv, pos, k, vt, tree):
            return K.attention_fused(qkv, hq, hkv, d, qn, kn, 1e-6, table, pos, k, vt, d ** -0.5, ws, tree)
        return d, (hq + 2 * hkv) * d, call
    d = int(layout)
    hq, rd = 4 * hkv, d // 4
    table, ws = K.rope_table_dim(1e7, rd, maxlen, dev), K.attn_general_workspace(hq, hkv, d, maxlen, dev)
    qn, kn = rnd(d), rnd(d)

    def call(qkv, pos, k, vt, tree):
        return K.attention_general(qkv, hq, hkv, d, 2 * d, 2 * hq * d, 2 * hq * d + hkv * d, d, qn, kn, 1e-6, rd, table, pos,
                                   k, vt, d ** -0.5, ws, tree)
    return d, (2 * hq + 2 * hkv) * d, call


@pytest.mark.parametrize("hkv,maxlen,past", CASES)
@pytest.mark.parametrize("layout", ["dense", "64", "128", "256"])
def test_few_rows_equal_a_long_step(dev, layout, hkv, maxlen, past):
    g = torch.Generator(device=dev).manual_seed(past + hkv)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev).to(torch.bfloat16)
    d, cols, call = _call(layout, rnd, dev, hkv, maxlen)
    qkv, k0, v0 = rnd(16, cols), rnd(hkv, maxlen, d), rnd(hkv, d, maxlen)
    k, vt = k0.clone(), v0.clone()
    ref = call(qkv, torch.tensor([past], dtype=torch.int32, device=dev), k, vt, None)
    for m in (1, 3, 4):
        k2, v2, out = k0.clone(), v0.clone(), []
        for i in range(0, 16, m):
            out.append(call(qkv[i:i + m], torch.tensor([past + i], dtype=torch.int32, device=dev), k2, v2, None))
        assert torch.equal(torch.cat(out), ref), m
        assert torch.equal(k2, k) and torch.equal(v2, vt), m


@pytest.mark.parametrize("layout", ["dense", "256"])
@pytest.mark.parametrize("past", [5, 126, 1000])
def test_few_rows_of_a_tree(dev, layout, past):
    """The first four nodes of a five-node tree (20 rows: staged chunks) as a four-node tree (16 rows)."""
    hkv, maxlen = 2, 1280
    g = torch.Generator(device=dev).manual_seed(past)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev).to(torch.bfloat16)
    d, cols, call = _call(layout, rnd, dev, hkv, maxlen)
    qkv, k0, v0 = rnd(5, cols), rnd(hkv, maxlen, d), rnd(hkv, d, maxlen)
    parents = [-1, 0, 0, 1, 3]
    pos = torch.tensor([past], dtype=torch.int32, device=dev)
    a = call(qkv, pos, k0.clone(), v0.clone(), DraftTree(parents, dev).desc)
    b = call(qkv[:4], pos, k0.clone(), v0.clone(), DraftTree(parents[:4], dev).desc)
    assert torch.equal(a[:4], b)


def test_few_rows_past_the_cache_are_dropped(dev):
    """A step that begins at the cache's last two slots with four tokens (no caller of the package lets it):
    the tokens without a slot are dropped, as in a step over staged chunks. Nothing lands in the next head's
    rows (slot 2048 of a head is slot 0 of the next) or after the last head's, and the rows are the staged
    step's. The RoPE table covers the positions; caches and workspace have guards behind them."""
    hkv, maxlen, past, d = 2, 2048, 2046, 128
    hq, m, guard = 4 * hkv, 4, 1 << 16
    g = torch.Generator(device=dev).manual_seed(3)
    rnd = lambda *s: torch.randn(s, generator=g, device=dev).to(torch.bfloat16)
    qkv, table = rnd(16, (hq + 2 * hkv) * d), K.rope_table(1e6, maxlen + 128, dev)
    k0, v0 = rnd(hkv * maxlen * d + guard), rnd(hkv * maxlen * d + guard)
    pos = torch.tensor([past], dtype=torch.int32, device=dev)
    words = K.attn_workspace(hkv, maxlen, dev).numel()
    got = []
    for rows in (m, 16):  # few rows; staged chunks
        k, vt = k0.clone(), v0.clone()
        ws = torch.full((words + guard,), -7.0, device=dev)
        kc, vc = k[:-guard].view(hkv, maxlen, d), vt[:-guard].view(hkv, d, maxlen)
        out = K.attention_fused(qkv[:rows], hq, hkv, d, None, None, 1e-6, table, pos, kc, vc, d ** -0.5, ws[:words], None)
        assert (ws[words:] == -7).all() and torch.equal(k[-guard:], k0[-guard:]) and torch.equal(vt[-guard:], v0[-guard:])
        got.append((out[:m], k, vt))
    (a, k, vt), (b, k2, vt2) = got
    assert torch.equal(a, b) and torch.equal(k, k2) and torch.equal(vt, vt2)
    want_k, want_v = k0[:-guard].view(hkv, maxlen, d).clone(), v0[:-guard].view(hkv, d, maxlen).clone()
    want_v[:, :, past:] = qkv[:2, (hq + hkv) * d:].view(2, hkv, d).permute(1, 2, 0)
    assert torch.equal(vt[:-guard].view(hkv, d, maxlen), want_v)
    assert torch.equal(k[:-guard].view(hkv, maxlen, d)[:, :past], want_k[:, :past])
