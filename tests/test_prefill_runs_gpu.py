"""The prompt prefill over several runs of rows (RUN_ROWS lowered so that short prompts take three and more) and on packed
W4A8 checkpoint weights (fp8 scales per 16, a codebook, H256 rotation), against the same prompt in chains of `slots`."""
import pytest
import torch

from conftest import assert_bits_equal, bits

pytestmark = pytest.mark.gpu

RUN = 32


def _fp8_weights(m, seed, default):
    """A checkpoint's linears for every layer of m: fp8 e4m3 scales per 16 and one codebook's values (default: code - 8), a
    tensor of its own per linear as a reader gives them."""
    from mdx import checkpoint
    g = torch.Generator().manual_seed(seed)
    cb = torch.linspace(-8, 7, 16) + (0 if default else 0.25) * torch.randn(16, generator=g)
    weights, plan = {}, {}
    for i, L in enumerate(m.layers):
        plan[i] = {}
        for r in ("qkv", "z", "q", "k", "v", "o", "g", "u", "d"):
            if r not in L:
                continue
            N, K = L[r].n, L[r].k
            q = torch.randint(-128, 128, (N, K // 2), generator=g, dtype=torch.int8)
            s = ((0.25 + 0.75 * torch.rand(N, K // 16, generator=g)) * 15).to(torch.float8_e4m3fn)
            sc = (0.8 + 0.4 * torch.rand(N, generator=g)) * (2e-4 if r in ("o", "d") else 8e-4)
            weights[f"{i}.{r}"] = checkpoint.w4_from_asym_w4a8(q, s, sc, cb.clone(), device=m.dev)
            plan[i][r] = f"{i}.{r}"
    return weights, plan


def _pair(dev, monkeypatch, bodies, layers, fp8=None, **kw):
    """The same prompts through the runs and through the chains; returns both models. fp8: checkpoint weights with their
    "default" codebook or an "own" one."""
    from mdx import hybrid
    ms = []
    for run in (True, False):
        cfg = hybrid.HybridConfig(layers=layers, inter=4096, vocab=32768, cap=512, greedy=True, rotate=fp8 is not None, **kw)
        m = hybrid.HybridModel(cfg, dev, seed=9)
        if fp8:
            m.load_w4(*_fp8_weights(m, 5, fp8 == "default"))
        calls = []
        f = m._prefill_run
        m._prefill_run = lambda tokens, *a, _f=f, _c=calls: _c.append(tokens.numel()) or _f(tokens, *a)
        g = torch.Generator().manual_seed(sum(bodies))
        with monkeypatch.context() as mp:
            mp.setattr(hybrid.HybridModel, "RUN_ROWS", RUN)
            if run:
                assert m._run_fits()
            else:
                mp.setattr(hybrid.HybridModel, "_run_fits", lambda self: False)
            for n in bodies:
                del calls[:]
                m.prefill(torch.randint(0, cfg.vocab, (n + 1,), generator=g))
                if run:
                    full = -(-max(n - RUN - cfg.slots, 0) // RUN)  # (runs of RUN rows while more than RUN + slots are left)
                    assert calls == [RUN] * full + [n - RUN * full], calls
                else:
                    assert not calls
        ms.append(m)
    return ms


def _same_state(a, b, what):
    assert torch.equal(a.st, b.st) and torch.equal(a.ctl, b.ctl) and torch.equal(a.nt, b.nt) and a.parity == b.parity, what
    assert_bits_equal(bits(a.hbuf), bits(b.hbuf), f"{what} hidden row")
    p = a.parity ^ 1  # the last chain's buffers, which the first decode step replays
    for i, (x, y) in enumerate(zip(a.gdn, b.gdn)):
        for n in ("rec", "conv") if x is not None else ():
            assert_bits_equal(bits(x[n]), bits(y[n]), f"{what} layer {i} {n}")
        for n in ("pb", "qb", "gates") if x is not None else ():
            assert_bits_equal(bits(x[n][p]), bits(y[n][p]), f"{what} layer {i} {n}")
    n = int(a.st[1].item())
    for x, y in zip(a.mkv, b.mkv):
        assert_bits_equal(bits(x[:, :, :n]), bits(y[:, :, :n]), f"{what} draft block cache")


# around the ends of a run: whole runs, one row more, a last run of RUN + slots rows and the first one past it
@pytest.mark.parametrize("slots,kw", [(16, {}), (8, dict(widths=(3,)))])
@pytest.mark.parametrize("k", [1, 3])
@pytest.mark.parametrize("more", ["0", "1", "slots", "slots+1"])
def test_runs_leave_the_chains_bits(dev, monkeypatch, slots, kw, k, more):
    """Gated-DeltaNet layers only: the state after several runs is the chains' bit for bit."""
    n = k * RUN + {"0": 0, "1": 1, "slots": slots, "slots+1": slots + 1}[more]
    print(f"case runs slots={slots} rows={n}", flush=True)
    a, b = _pair(dev, monkeypatch, [n], 3, slots=slots, **kw)
    _same_state(a, b, f"{n} rows")


@pytest.mark.parametrize("bodies", [[97, 70], [49, 113], [20, 96]])
def test_runs_of_a_second_prompt(dev, monkeypatch, bodies):
    """The second prompt's first run starts with rows pending from the first prompt, its others with none."""
    a, b = _pair(dev, monkeypatch, bodies, 3)
    _same_state(a, b, f"{bodies} rows")


@pytest.mark.parametrize("run", [True, False])
@pytest.mark.parametrize("first,second", [(10, 60), (20, 60), (40, 7), (97, 70)])
def test_two_prompts_equal_one(dev, monkeypatch, run, first, second):
    """A prompt fed in two pieces (the second starts with the first's last token) and the first decode step after it: the
    rows that the first piece leaves pending are replayed from its buffers, whichever parity they have."""
    from mdx import hybrid
    cfg = hybrid.HybridConfig(layers=3, inter=4096, vocab=32768, cap=512, greedy=True)
    if not run:
        monkeypatch.setattr(hybrid.HybridModel, "_run_fits", lambda self: False)
    tokens = torch.randint(0, cfg.vocab, (first + second + 1,), generator=torch.Generator().manual_seed(first))
    ms = []
    for pieces in ([tokens], [tokens[:first + 1], tokens[first:]]):
        m = hybrid.HybridModel(cfg, dev, seed=9)
        for t in pieces:
            m.prefill(t)
        ms.append(m)
    a, b = ms
    assert torch.equal(a.st, b.st) and torch.equal(a.nt, b.nt)
    assert_bits_equal(bits(a.hbuf), bits(b.hbuf), "hidden row")
    for m in ms:
        m.step(m.parity)
    assert_bits_equal(bits(a.logits), bits(b.logits), "logits")
    assert torch.equal(a.result, b.result) and torch.equal(a.st, b.st)
    for i, (x, y) in enumerate(zip(a.gdn, b.gdn)):
        for n in ("rec", "conv"):
            assert_bits_equal(bits(x[n]), bits(y[n]), f"layer {i} {n}")


@pytest.mark.parametrize("run", [True, False])
def test_a_second_prompt_counts_the_first(dev, monkeypatch, run):
    """The capacity that a prompt needs starts at the position before it, and so does the bound that decode steps are held
    to: past the cache neither a prompt nor a step is launched."""
    from mdx import hybrid
    if not run:
        monkeypatch.setattr(hybrid.HybridModel, "_run_fits", lambda self: False)
    cfg = hybrid.HybridConfig(layers=1, inter=4096, vocab=32768, cap=128, greedy=True)
    m = hybrid.HybridModel(cfg, dev, seed=9)
    tokens = torch.randint(0, cfg.vocab, (cfg.cap,), generator=torch.Generator().manual_seed(1))
    m.prefill(tokens[:70])
    st = m.st.clone()
    with pytest.raises(RuntimeError, match="position 69"):
        m.prefill(tokens[:cfg.cap - 69 - m.R + 1])
    assert torch.equal(m.st, st)
    m.prefill(tokens[:cfg.cap - 69 - m.R])
    assert m.pos_bound == int(m.st[0].item()) == cfg.cap - m.R - 1
    with pytest.raises(RuntimeError, match="cache capacity"):
        m.step(m.parity)


@pytest.mark.parametrize("codebook,n", [("own", 20), ("own", 113), ("default", 113)])
def test_checkpoint_weights_leave_the_chains_bits(dev, monkeypatch, codebook, n):
    """fp8 scales, codebook and rotation through the many-row GEMM, from the checkpoint reader's handles."""
    a, b = _pair(dev, monkeypatch, [n], 3, fp8=codebook)
    assert (a.layers[0]["g"].cb is None) == (codebook == "default")
    _same_state(a, b, f"fp8 {n} rows")


@pytest.mark.parametrize("n,fp8", [(96, None), (97, None), (112, None), (113, None), (200, None), (113, "own")])
def test_runs_with_attention(dev, monkeypatch, n, fp8):
    """With an attention layer the order of its fp32 sums differs from the chains', and a bf16 rounding that flips travels
    through the layers that follow: states, caches and the first decode step's logits within 2e-3 of the chains'. (8
    layers, 40 to 1000 rows: 0 to 4e-4 with the seed.)"""
    a, b = _pair(dev, monkeypatch, [n], 4, fp8=fp8)
    assert torch.equal(a.st, b.st) and torch.equal(a.ctl, b.ctl) and torch.equal(a.nt, b.nt) and a.parity == b.parity
    pairs = [(x[:, :, :n], y[:, :, :n]) for u, w in zip(a.kv + [a.mkv], b.kv + [b.mkv]) if u is not None for x, y in zip(u, w)]
    pairs += [(x["rec"], y["rec"]) for x, y in zip(a.gdn, b.gdn) if x is not None] + [(a.hbuf, b.hbuf)]
    rel = [float((x.double() - y.double()).norm() / y.double().norm()) for x, y in pairs]
    for m in (a, b):
        m.step(m.parity)
    lg = float((a.logits.double() - b.logits.double())[0].norm() / b.logits.double()[0].norm())
    print(f"case attention rows={n} fp8={fp8}: largest {max(rel):.2e}, logits {lg:.2e}", flush=True)
    assert max(rel) <= 2e-3 and lg <= 2e-3
