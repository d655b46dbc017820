"""The draft block's launches that take their elementwise neighbours along, bit for bit against the separate operators."""
import pytest
import torch

from conftest import assert_bits_equal, bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,Hk,D,S,L", [(32, 8, 128, 1, 0), (32, 8, 128, 1, 300), (16, 4, 256, 1, 5000), (8, 8, 64, 3, 77),
                                        (16, 4, 256, 16, 40), (32, 8, 128, 7, 2048)])
def test_gated_attention(C, dev, H, Hk, D, S, L):
    g = torch.Generator().manual_seed(H + S + L)
    cap = L + 40
    r = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)  # noqa: E731
    q, k, v, xk, xv = r(1, H, S, D), r(1, Hk, cap, D), r(1, Hk, cap, D), r(1, Hk, S, D), r(1, Hk, S, D)
    qkv = r(S, 2 * H * D + 2 * Hk * D) * 3
    qg = qkv[:, :2 * H * D]
    sl = torch.tensor([L], dtype=torch.int32, device=dev)
    mask = torch.tensor([(1 << (i + 1)) - 1 for i in range(S)] if S > 1 else [], dtype=torch.int32, device=dev)
    if S == 1 and L == 0:
        mask = torch.ones(1, dtype=torch.int32, device=dev)
    y = C.attn_dpas(q, k, v, sl, xk, xv, mask)
    want = torch.empty(S, H * D, dtype=torch.bfloat16, device=dev)
    C.draft_sigmoid_mul(y.view(S, H * D), qg if S > 1 else qg.reshape(-1), D, want)
    assert_bits_equal(bits(C.attn_gated(q, k, v, sl, xk, xv, mask, qg).view(S, H * D)), bits(want), "gated")


@pytest.mark.parametrize("I,K", [(12288, 4096), (6160, 256), (12304, 2048), (24576, 96)])
@pytest.mark.parametrize("rows", [1, 3, 16])
def test_gate_up(C, dev, I, K, rows):
    from mdx import _lib, layout
    g = torch.Generator(device=dev).manual_seed(I + rows)
    w = layout.tile_major_bf16((torch.randn(2 * I, K, generator=g, device=dev) * 0.05).bfloat16())
    x = torch.randn(rows, K, generator=g, device=dev).bfloat16()
    assert _lib.lib().mdx_bf16_gate_up_fits(I, K)
    gu = C.bf16_linear(x, w)
    want, got = (torch.empty(rows, I, dtype=torch.bfloat16, device=dev) for _ in range(2))
    C.draft_silu_mul(gu, want)
    C.bf16_gate_up(x, w, got)
    assert_bits_equal(bits(got), bits(want), "gate/up")


def test_gate_up_refuses_many_slices(C, dev):
    from mdx import _lib
    assert not _lib.lib().mdx_bf16_gate_up_fits(64, 4096)
    with pytest.raises(RuntimeError):
        C.bf16_gate_up(torch.zeros(1, 4096, dtype=torch.bfloat16, device=dev),
                       torch.zeros(128, 4096, dtype=torch.bfloat16, device=dev),
                       torch.zeros(1, 64, dtype=torch.bfloat16, device=dev))


@pytest.mark.parametrize("H,rows", [(256, 1), (4096, 1), (4096, 5), (5120, 2)])
def test_norm_quant(C, dev, H, rows):
    g = torch.Generator().manual_seed(H + rows)
    x, h = ((torch.randn(rows, H, generator=g) * s).bfloat16().to(dev) for s in (3, 1))
    x[0, :4] *= 200
    w = (1 + 0.1 * torch.randn(H, generator=g)).bfloat16().to(dev)
    x2, n1, n2 = x.clone(), torch.empty_like(x), torch.empty_like(x)
    C.draft_norm_rot_quant(x, h, w, 1e-6, None, n1, None, None)
    q, s = C.quant_rows(n1)
    q2, s2 = torch.empty_like(q), torch.empty(rows, device=dev)
    C.draft_norm_quant(x2, h, w, 1e-6, n2, q2, s2)
    for a, b, n in ((x2, x, "x"), (n2, n1, "norm"), (q2, q, "codes"), (s2, s.view(-1), "scales")):
        assert_bits_equal(bits(a), bits(b), n)


@pytest.mark.parametrize("depth,pos", [(0, 0), (3, 17), (6, 60)])
def test_embed_prep(C, dev, depth, pos):
    g = torch.Generator().manual_seed(pos)
    H, V, cap, np_ = 4096, 99, 64, 16
    r = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)  # noqa: E731
    emb, hid, we, wh = r(V, H), r(1, H), r(H), r(H)
    tok = torch.tensor([V - 1 if depth else 5], device=dev)
    ftab = torch.randn(1, 1, cap, 32, 2, 2, generator=g).to(dev)
    st = torch.tensor([pos, pos // 2, 0, 0], dtype=torch.int64, device=dev)
    outs = []
    for fused in (False, True):
        cat, fr = torch.zeros(1, 2 * H, dtype=torch.bfloat16, device=dev), torch.zeros(1, 1, 1, 32, 2, 2, device=dev)
        mpos, mseq = torch.zeros(np_, dtype=torch.int64, device=dev), torch.zeros(1, dtype=torch.int32, device=dev)
        if fused:
            C.draft_embed_prep(tok, emb, hid, we, wh, 1e-6, 1e-6, cat, st, depth, ftab, fr, mpos, mseq)
        else:
            C.mtp_prep_draft(st, depth, ftab, fr, mpos, mseq)
            C.draft_embed_norm_cat(tok, None, None, None, emb, hid, we, wh, 1e-6, 1e-6, cat)
        outs.append((cat, fr, mpos, mseq))
    for a, b in zip(*outs):
        assert_bits_equal(bits(a), bits(b), "embed / prep")
