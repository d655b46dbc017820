"""A traced decode step runs the draft block's elementwise operators as launches of their own (their inputs are in the
trace, which the oracle's step test checks stage by stage); an untraced one takes them inside the launches beside them
(attn_gated, bf16_gate_up, draft_norm_quant). Both leave the same bits, step after step."""
import pytest
import torch

from conftest import assert_bits_equal, bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(), dict(two_stage=True), dict(head="int8"), dict(head="int8", two_stage=True),
                                dict(two_stage=True, widths=(2, 1, 1), slots=8), dict(attn="exact"),
                                dict(head_dim=64, heads=64, rotary=32)],
                         ids=lambda kw: "-".join(f"{k}={v}" for k, v in kw.items()) or "one_stage")
def test_traced_step_equals_untraced(C, dev, monkeypatch, kw):
    from mdx import hybrid
    fused = []
    for name in ("attn_gated", "bf16_gate_up"):
        f = getattr(C, name)
        monkeypatch.setattr(C, name, lambda *a, _n=name, _f=f, **k: fused.append(_n) or _f(*a, **k))
    ms = []
    for traced in (False, True):
        cfg = hybrid.HybridConfig(layers=2, attn_every=2, vocab=32768, cap=256, greedy=True, **kw)
        m = hybrid.HybridModel(cfg, dev, seed=13)
        m.prefill(torch.randint(0, cfg.vocab, (21,), generator=torch.Generator().manual_seed(4)))
        ms.append(m)
    a, b = ms
    for step in range(4):
        print(f"case traced step {step} {kw}", flush=True)
        del fused[:]
        a.step(a.parity)
        want = {"bf16_gate_up"} | (set() if kw.get("attn") == "exact" else {"attn_gated"})
        assert set(fused) == want and len(fused) == len(want) * len(a.widths)
        del fused[:]
        b.trace = []
        b.step(b.parity)
        assert not fused and {"mtp.y", "mtp.gu"} <= {n for n, _ in b.trace}
        for n in ("dh", "dxf", "dgy", "dact", "dtok", "vtok", "toks", "result", "logits", "hbuf", "st", "ctl", "nt"):
            assert_bits_equal(bits(getattr(a, n)), bits(getattr(b, n)), f"step {step} {n}")
        if kw.get("head") == "int8" or kw.get("two_stage"):
            for n in ("dqx", "dsx"):
                assert_bits_equal(bits(getattr(a, n)), bits(getattr(b, n)), f"step {step} {n}")
        for x, y in zip(a.mkv + a.kv[1], b.mkv + b.kv[1]):
            assert_bits_equal(bits(x), bits(y), f"step {step} caches")
        for m in ms:
            m.parity ^= 1
