"""The many-row matmul (skinny_qmm_w4g64_rows_bf16) is bitwise the 16-row pieces it replaces: every form
of the kernel (one part, 3 and 4 parts of K, both block widths, one to three kept sums) at the edges of
its blocks, rows and weight tiles that do not fill them, strided rows and the three epilogues. The
pieces themselves are held to the oracle in test_qmm_gpu.py."""

import pytest
import torch

from skinny_mlx import kernels as K
from skinny_mlx import qmm as Q

pytestmark = pytest.mark.gpu


def _weights(n, k, seed, dev, glu=False):
    g = torch.Generator(device=dev).manual_seed(seed)
    w, s, b = Q.random_w4g64(n, k, generator=g, device=dev, scale_std=0.01)
    b = b + (torch.randn(b.shape, generator=g, device=dev) * 0.01).to(b.dtype)
    return (Q.repack_gate_up if glu else Q.repack_for_skinny)(w, s, b), g


def _same(a, b):
    return torch.equal(a.contiguous().view(torch.int16), b.contiguous().view(torch.int16))


# (rows, K, N): the least K and N; weight tiles that do not fill a block; the decoders' shapes at each
# form's row counts (o_proj: 4 parts narrow, 4 parts wide, 2 parts of 48 rows, one part; down: 3 parts narrow, wide, 3
# parts of 48 rows, one part with three sums; q|k|v; gate|up-wide and the head: the 64-wide wave)
SHAPES = [(17, 128, 16), (33, 256, 48), (47, 384, 80), (64, 256, 512), (65, 640, 272), (33, 4096, 2560), (200, 4096, 2560),
          (450, 4096, 2560), (700, 4096, 2560), (65, 9728, 2560), (250, 9728, 2560), (401, 9728, 2560), (700, 9728, 2560), (77, 2560, 6144), (450, 2560, 19456),
          (33, 2560, 151936)]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_rows_equal_pieces(dev, m, k, n):
    w, g = _weights(n, k, m + n, dev)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    splits, tile = Q._plain_config(k, n)
    y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
    Q._rows(x, w, y, splits, tile, Q.EPI_PLAIN, "test")
    ref = torch.cat([Q.skinny_qmm(x[i:i + 16], w) for i in range(0, m, 16)])
    assert _same(y, ref)
    assert _same(Q.skinny_qmm(x, w), ref)  # whichever way the public call goes


@pytest.mark.parametrize("m,k,f", [(17, 128, 16), (33, 256, 80), (20, 2560, 9728), (129, 2560, 9728), (450, 2560, 9216)])
def test_rows_gate_up_equal_pieces(dev, m, k, f):
    w, g = _weights(2 * f, k, m + f, dev, glu=True)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    for swiglu, epi in ((True, Q.EPI_SWIGLU), (False, Q.EPI_GLU_SPLIT)):
        ref = torch.cat([Q.skinny_glu(x[i:i + 16], w, swiglu) for i in range(0, m, 16)])
        y = torch.full_like(ref, float("nan"))
        Q._rows(x, w, y, 1, Q.glu_tile(k, f), epi, "test")
        assert _same(y, ref), swiglu


@pytest.mark.parametrize("splits,waves", [(1, 1), (1, 2), (1, 16), (2, 4), (3, 4), (4, 4)])
@pytest.mark.parametrize("m,n", [(40, 1040), (600, 1040), (600, 2064), (600, 6416)])  # parts, of 48 rows, the wide wave
def test_rows_follow_the_cut(dev, splits, waves, m, n, monkeypatch):
    """Any cut of K, also one that no table holds (19 pairs: uneven groups and splits)."""
    k = 19 * 128
    w, g = _weights(n, k, splits * 100 + waves, dev)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    monkeypatch.setattr(Q, "SPLITK_OVERRIDE", (splits, 1, 1, waves, 2))
    ref = torch.cat([Q.skinny_qmm(x[i:i + 16], w) for i in range(0, m, 16)])
    y = torch.empty_like(ref)
    Q._rows(x, w, y, *Q._plain_config(k, n), Q.EPI_PLAIN, "test")
    assert _same(y, ref)


def test_rows_strided_and_unaligned_output(dev):
    m, k, n = 70, 512, 528
    w, g = _weights(n, k, 9, dev)
    wide = torch.randn((m, k + 64), generator=g, device=dev).to(torch.bfloat16)
    x = wide[:, 32:32 + k]
    ref = torch.cat([Q.skinny_qmm(x[i:i + 16].contiguous(), w) for i in range(0, m, 16)])
    for pad, off in ((0, 0), (8, 8), (3, 1)):  # 16-byte rows, then rows that take scalar stores
        buf = torch.full((m, n + pad), 7.0, dtype=torch.bfloat16, device=dev)
        out = buf[:, off:off + n]
        assert Q.skinny_qmm(x, w, out=out).data_ptr() == out.data_ptr()
        assert _same(out, ref)
        assert (buf[:, :off] == 7).all() and (buf[:, off + n:] == 7).all()


@pytest.mark.parametrize("m,k,n", [(17, 256, 48), (100, 4096, 2560), (77, 9728, 2560), (65, 9216, 2560), (40, 2048, 2560)])
def test_rows_of_a_residual_equal_the_summed_slices(dev, m, k, n):
    w, g = _weights(n, k, m + k, dev)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    ref = []
    for i in range(0, m, 16):
        parts = Q.skinny_qmm_partial(x[i:i + 16], w).parts
        total = parts[0]
        for p in parts[1:]:
            total = total + p
        ref.append(total.to(torch.bfloat16))
    assert _same(Q.skinny_qmm_rows(x, w, "partial"), torch.cat(ref))


@pytest.mark.parametrize("m,k,n,c", [(17, 256, 48, 16), (33, 512, 256, 64), (50, 2560, 8224, 6144), (33, 2560, 12352, 8192)])
def test_rows_before_the_conv_equal_its_product(dev, m, k, n, c):
    """The columns past the conv's are skinny_qmm_conv's own; its first c are the conv of ours."""
    w, g = _weights(n, k, m + n, dev)
    x = torch.randn((m, k), generator=g, device=dev).to(torch.bfloat16)
    cw = torch.randn((c, 4), generator=g, device=dev).to(torch.bfloat16)
    s1, s2 = (torch.zeros((3, c), dtype=torch.bfloat16, device=dev) for _ in range(2))
    ref = torch.cat([Q.skinny_qmm_conv(x[i:i + 16], w, c, s1, cw) for i in range(0, m, 16)])
    y = Q.skinny_qmm_rows(x, w, "conv")
    assert _same(y[:, c:], ref[:, c:])
    assert _same(K.gdn_conv_silu(y[:, :c], s2, cw, None), ref[:, :c]) and _same(s1, s2)


def test_rows_take_no_other_form(dev):
    w, _ = _weights(48, 256, 1, dev)
    with pytest.raises(ValueError, match="form"):
        Q.skinny_qmm_rows(torch.zeros((20, 256), dtype=torch.bfloat16, device=dev), w, "plain")
