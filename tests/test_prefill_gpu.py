"""The many-row forms behind the prompt prefill: the W4A8 GEMM bit for bit against the oracle, the bf16 GEMM and the
causal attention against float64, and a whole prefill against the same prompt fed in chains through the verify path."""
import numpy as np
import pytest
import torch

from conftest import assert_bits_equal, bits
from oracle import ref

pytestmark = pytest.mark.gpu


def _w4(N, K, G, form, cb, g, dev):
    from mdx import _lib, layout
    q = torch.randint(-128, 128, (N, K // 2), generator=g, dtype=torch.int8)
    sc = torch.rand(N, generator=g) * 1e-3 + 1e-4
    if form == "fp8":
        s = torch.randint(0, 256, (N, K // G), generator=g, dtype=torch.uint8)
        sf, st = ref.fp8e4m3_to_f32(s.numpy()), s.view(torch.float8_e4m3fn)
    else:  # fp16 ratios, some past the packed-half table build (|s| > 15.875) and negative
        st = ((torch.rand(N, K // G, generator=g) - 0.3) * (40 if form == "fp16w" else 15)).half()
        sf = st.float().numpy()
    w = layout.W4(layout.tile_major_codes(q).to(dev), st.to(dev), sc.to(dev), cb, _lib.LAYOUT_TILE)
    return w, (q.numpy(), sf, sc.numpy(), None if cb is None else cb.cpu().numpy(), G)


@pytest.mark.parametrize("form,K,G", [("fp16", 256, 128), ("fp16w", 1280, 128), ("fp16", 1024, 512), ("fp8", 256, 16),
                                      ("fp8", 768, 32), ("fp8", 1024, 128), ("fp16", 4096, 128), ("fp8", 12288, 16)])
def test_w4a8_gemm_matches_oracle(C, dev, form, K, G):
    g = torch.Generator().manual_seed(K + G)
    cb = (torch.randn(16, generator=g) * 4).to(dev) if (form, K) in (("fp16", 1024), ("fp8", 768)) else None
    ws = [_w4(N, K, G, form, cb, g, dev) for N in (48, 272, 16)]
    for M in (1, 16, 63, 65, 129, 200):
        print(f"case {form} K={K} G={G} M={M}", flush=True)
        x = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
        xs = torch.rand(M, generator=g) * 0.05 + 1e-3
        res = [torch.randn(M, w.n, generator=g).to(torch.bfloat16) for w, _ in ws]
        outs = [torch.empty(M, w.n, dtype=torch.bfloat16, device=dev) for w, _ in ws]
        C.w4a8_gemm(x.to(dev), xs.to(dev), [w for w, _ in ws], outs, residuals=[res[0].to(dev), None, res[2].to(dev)])
        for i, (w, o) in enumerate(ws):
            want = ref.w4a8_linear(x.numpy(), xs.numpy(), *o, None if i == 1 else bits(res[i]))
            assert_bits_equal(bits(outs[i]), np.asarray(want), f"matrix {i} M={M}")


@pytest.mark.parametrize("form,G", [("fp16", 128), ("fp8", 16)])
def test_w4a8_gemm_gate_up_equals_the_gemv(C, dev, form, G):
    from mdx import layout
    g = torch.Generator().manual_seed(G)
    K, N = 512, 144
    (wg, _), (wu, _) = _w4(N, K, G, form, None, g, dev), _w4(N, K, G, form, None, g, dev)
    wg.sc *= 20
    lut = layout.silu_lut(dev)
    for M in (16, 100):
        x = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8).to(dev)
        xs = (torch.rand(M, generator=g) * 0.05 + 1e-3).to(dev)
        got, want = (torch.empty(M, N, dtype=torch.bfloat16, device=dev) for _ in range(2))
        C.w4a8_gemm(x, xs, [wg, wu], [got], gate_up=True, silu_lut=lut)
        for r in range(0, M, 16):
            C.stream_gemv(x[r:r + 16], xs[r:r + 16], [wg, wu], [want[r:r + 16]], gate_up=True, silu_lut=lut)
        assert_bits_equal(bits(got), bits(want), f"M={M}")


def test_w4a8_gemm_refuses_other_forms(C, dev):
    from mdx import _lib, layout
    g = torch.Generator().manual_seed(1)
    w, _ = _w4(16, 384, 128, "fp16", None, g, dev)  # an odd group count
    row = layout.W4(w.q, w.s, w.sc, None, _lib.LAYOUT_ROW)
    x, xs, o = torch.zeros(20, 384, dtype=torch.int8, device=dev), torch.ones(20, device=dev), torch.zeros(20, 16, dtype=torch.bfloat16, device=dev)
    for bad in (w, row):
        assert not _lib.lib().mdx_w4a8_gemm_fits(bad.struct())
        with pytest.raises(RuntimeError):
            C.w4a8_gemm(x, xs, [bad], [o])


@pytest.mark.parametrize("N,K", [(48, 64), (272, 192), (2048, 4096)])
def test_bf16_gemm_against_float64(C, dev, N, K):
    from mdx import layout
    g = torch.Generator().manual_seed(N)
    w = torch.randn(N, K, generator=g).to(torch.bfloat16)
    wt = layout.tile_major_bf16(w.to(dev))
    for M in (1, 64, 130):
        x = torch.randn(M, K, generator=g).to(torch.bfloat16)
        out = torch.empty(M, N - 16, dtype=torch.bfloat16, device=dev)
        C.bf16_gemm(x.to(dev), wt, out, n0=16)
        want = x.double() @ w.double().T[:, 16:]
        # one bf16 rounding (2^-8 relative), and fp32 sums: at most K 2^-23 of the sum of the products' magnitudes
        bound = want.abs() * 2.0 ** -8 + (x.double().abs() @ w.double().abs().T[:, 16:]) * K * 2.0 ** -23 + 1e-30
        assert ((out.cpu().double() - want).abs() <= bound).all(), f"N={N} K={K} M={M}"


@pytest.mark.parametrize("H,Hk,D,L,S", [(8, 2, 128, 0, 33), (4, 4, 64, 70, 17), (6, 2, 128, 31, 1), (8, 1, 64, 5, 100),
                                        (32, 8, 128, 129, 200)])
def test_attn_prefill_against_float64(C, dev, H, Hk, D, L, S):
    from mdx import _lib
    g = torch.Generator().manual_seed(H + S)
    cap = L + S + 3
    q = (torch.randn(H, S, D, generator=g) * 2).to(torch.bfloat16)
    k, v = (torch.randn(1, Hk, cap, D, generator=g).to(torch.bfloat16) for _ in range(2))
    qd, kd, vd = q.to(dev), k.to(dev), v.to(dev)
    out = torch.empty(S, H * D, dtype=torch.bfloat16, device=dev)
    seq = torch.tensor([L], dtype=torch.int32, device=dev)
    _lib.call("mdx_attn_prefill", _lib.ptr(qd), S * D, D, _lib.ptr(kd), _lib.ptr(vd), _lib.ptr(seq), _lib.ptr(out), H, Hk, S,
              D, cap, _lib.stream_of(qd))
    allow = torch.arange(cap)[None] <= L + torch.arange(S)[:, None]
    for h in range(H):
        sc = q[h].double() @ k[0, h // (H // Hk)].double().T / D ** 0.5
        p = torch.softmax(sc.masked_fill(~allow, -float("inf")), -1)
        vv = v[0, h // (H // Hk)].double()
        # P and the output are rounded to bf16 (2^-9 relative each way, over the weights and over the result)
        bound = 2.0 ** -7 * (p @ vv.abs()) + 1e-6
        got = out.view(S, H, D)[:, h].cpu().double()
        assert ((got - p @ vv).abs() <= bound).all(), f"head {h}"


def _pair(dev, layers, tokens, monkeypatch, twice=False, **kw):
    from mdx import hybrid
    ms = []
    for run in (True, False):
        cfg = hybrid.HybridConfig(layers=layers, inter=4096, vocab=32768, cap=512, **kw)
        m = hybrid.HybridModel(cfg, dev, seed=9)
        g = torch.Generator().manual_seed(tokens)
        with monkeypatch.context() as mp:
            if not run:
                mp.setattr(hybrid.HybridModel, "_run_fits", lambda self: False)
            else:
                assert m._run_fits()
            for n in ([tokens, tokens + 2] if twice else [tokens]):
                m.prefill(torch.randint(0, cfg.vocab, (n,), generator=g))
                m.pos_bound = int(m.st[0].item())
        ms.append(m)
    return ms


@pytest.mark.parametrize("tokens,slots,twice,kw", [(50, 16, False, {}), (97, 16, True, {}), (82, 8, False, dict(widths=(3,))),
                                                   (66, 16, False, dict(rotate=True)), (66, 16, False, dict(scales="integral"))])
def test_prefill_without_attention_is_bit_identical(dev, monkeypatch, tokens, slots, twice, kw):
    """Gated-DeltaNet layers only: every state tensor, the hidden row and the control words are the chains' bits (with
    twice: the second prompt starts with a chain pending from the first)."""
    a, b = _pair(dev, 3, tokens, monkeypatch, twice, slots=slots, **kw)
    assert torch.equal(a.st, b.st) and torch.equal(a.ctl, b.ctl) and torch.equal(a.nt, b.nt) and a.parity == b.parity
    assert_bits_equal(bits(a.hbuf), bits(b.hbuf), "hidden row")
    p = a.parity ^ 1  # the last chain's buffers, which the first decode step replays
    for i, (x, y) in enumerate(zip(a.gdn, b.gdn)):
        for n in ("rec", "conv"):
            assert_bits_equal(bits(x[n]), bits(y[n]), f"layer {i} {n}")
        for n in ("pb", "qb", "gates"):
            assert_bits_equal(bits(x[n][p]), bits(y[n][p]), f"layer {i} {n}")
    n = int(a.st[1].item())
    for x, y in zip(a.mkv, b.mkv):  # (the bf16 GEMM's sums are bf16_linear's)
        assert_bits_equal(bits(x[:, :, :n]), bits(y[:, :, :n]), "draft block cache")


def test_prefill_matches_the_chains(dev, monkeypatch):
    """With an attention layer: the attention's order of sums differs, so a rounding travels; the caches, the states and
    the decode that follows stay together."""
    a, b = _pair(dev, 4, 150, monkeypatch, greedy=True)
    n = int(a.st[0].item())
    assert torch.equal(a.st, b.st) and torch.equal(a.ctl, b.ctl)
    pairs = [(x[:, :, :n], y[:, :, :n]) for u, w in zip(a.kv + [a.mkv], b.kv + [b.mkv]) if u is not None for x, y in zip(u, w)]
    pairs += [(x["rec"], y["rec"]) for x, y in zip(a.gdn, b.gdn) if x is not None] + [(a.hbuf, b.hbuf)]
    for x, y in pairs:
        assert (x.double() - y.double()).norm() <= 5e-3 * y.double().norm()
    for m in (a, b):
        m.step(m.parity)
    assert (a.logits.double() - b.logits.double())[0].norm() <= 2e-2 * b.logits.double()[0].norm()
