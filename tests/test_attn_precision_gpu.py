"""The attention's distance from float64 where its weights are rounded to bf16: no more than that of a softmax whose
weights are rounded against the maximum of their own 32 tokens, everything else float64 and the output one bf16 rounding."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _softmax(z, v, bf16_weights):
    """softmax(z) v of float64 scores z [rows, tokens] (-inf: not admitted), in float64; bf16_weights: each weight rounded
    to bf16 against the largest score of its 32 tokens."""
    M = z.amax(-1, keepdim=True)
    if not bf16_weights:
        p = torch.exp(z - M)
        return (p @ v) / p.sum(-1, keepdim=True)
    n = z.shape[1]
    zb = torch.nn.functional.pad(z, (0, -n % 32), value=-math.inf).view(z.shape[0], -1, 32)
    mb = zb.amax(-1, keepdim=True).clamp_min(-1e300)
    p = torch.exp(zb - mb).bfloat16().double() * torch.exp(mb - M[..., None])
    p = p.reshape(z.shape[0], -1)[:, :n]
    return (p @ v) / p.sum(-1, keepdim=True)


def _no_further_than_blocks(heads, what):
    """heads: (got [rows, D], z, v) of each kv head, one norm over all. The kernel's own fp32 sums and exp2 add errors of
    about 2^-22; the roundings those flip change the norm of the 2^-9 errors of thousands of outputs by well below 3e-3."""
    got = torch.cat([h[0] for h in heads])
    want = torch.cat([_softmax(z, v, False) for _, z, v in heads])
    blocks = torch.cat([_softmax(z, v, True) for _, z, v in heads]).bfloat16().double()
    e, eb = float((got - want).norm() / want.norm()), float((blocks - want).norm() / want.norm())
    print(f"{what}: {e:.4e}, blocks {eb:.4e}", flush=True)
    assert e <= 1.003 * eb, (what, e, eb)


@pytest.mark.parametrize("H,Hk,S,L", [(8, 1, 8, 16000), (16, 4, 8, 16384), (16, 4, 8, 8191), (4, 1, 16, 3000)])
def test_decode_attention_head_dim_256(C, dev, H, Hk, S, L):
    D, gr = 256, H // Hk
    g = torch.Generator(device=dev).manual_seed(L + S)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()  # noqa: E731
    q = (torch.randn(1, H, S, D, generator=g, device=dev) * 2).bfloat16()
    key, val, xk, xv = r(1, Hk, L + 64, D), r(1, Hk, L + 64, D), r(1, Hk, S, D), r(1, Hk, S, D)
    mask = torch.tensor([(1 << (i + 1)) - 1 for i in range(S)], dtype=torch.int32, device=dev)
    out = C.attn_dpas(q, key, val, torch.tensor([L], dtype=torch.int32, device=dev), xk, xv, mask).double().view(S, H, D)
    pad = -L % 32  # (the tree rows are blocks of their own)
    causal = torch.ones(S, S, dtype=torch.bool, device=dev).tril().repeat(gr, 1)
    heads = []
    for kh in range(Hk):
        qh = q[0, kh * gr:(kh + 1) * gr].double().reshape(-1, D)
        z = torch.full((gr * S, L + pad + S), -math.inf, dtype=torch.float64, device=dev)
        z[:, :L] = qh @ key[0, kh, :L].double().t().contiguous() / math.sqrt(D)
        z[:, L + pad:] = (qh @ xk[0, kh].double().t().contiguous() / math.sqrt(D)).masked_fill(~causal, -math.inf)
        v = torch.zeros(L + pad + S, D, dtype=torch.float64, device=dev)
        v[:L], v[L + pad:] = val[0, kh, :L].double(), xv[0, kh].double()
        heads.append((out[:, kh * gr:(kh + 1) * gr].transpose(0, 1).reshape(-1, D), z, v))
    _no_further_than_blocks(heads, f"H={H} Hk={Hk} S={S} L={L}")


@pytest.mark.parametrize("H,Hk,D,L,S", [(32, 8, 128, 0, 1000), (32, 8, 128, 500, 500), (16, 8, 64, 0, 200), (8, 2, 64, 1000, 300)])
def test_prefill_attention(C, dev, H, Hk, D, L, S):
    """Also no further than the same rows in chains of 16 through the decode attention."""
    from mdx import _lib
    gr, cap = H // Hk, L + S + 16
    g = torch.Generator(device=dev).manual_seed(L + S)
    r = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()  # noqa: E731
    q = (torch.randn(1, H, S, D, generator=g, device=dev) * 2).bfloat16()
    k, v = r(1, Hk, cap, D), r(1, Hk, cap, D)
    out = torch.empty(S, H * D, dtype=torch.bfloat16, device=dev)
    seq = torch.tensor([L], dtype=torch.int32, device=dev)
    _lib.call("mdx_attn_prefill", _lib.ptr(q), S * D, D, _lib.ptr(k), _lib.ptr(v), _lib.ptr(seq), _lib.ptr(out), H, Hk, S,
              D, cap, _lib.stream_of(q))
    chains = torch.empty_like(out)
    for s0 in range(0, S, 16):
        n = min(16, S - s0)
        new = slice(L + s0, L + s0 + n)
        mask = torch.tensor([(1 << (i + 1)) - 1 for i in range(n)], dtype=torch.int32, device=dev)
        chains[s0:s0 + n] = C.attn_dpas(q[:, :, s0:s0 + n], k, v, torch.tensor([L + s0], dtype=torch.int32, device=dev),
                                        k[:, :, new], v[:, :, new], mask).view(n, -1)
    allow = (torch.arange(L + S, device=dev)[None] <= L + torch.arange(S, device=dev)[:, None]).repeat(gr, 1)
    heads, errs = [], [0.0, 0.0]
    out, chains = (t.double().view(S, H, D) for t in (out, chains))
    for kh in range(Hk):
        own = slice(kh * gr, (kh + 1) * gr)
        z = q[0, own].double().reshape(-1, D) @ k[0, kh, :L + S].double().t().contiguous() / math.sqrt(D)
        z = z.masked_fill(~allow, -math.inf)
        vv = v[0, kh, :L + S].double()
        want = _softmax(z, vv, False)
        rows = [t[:, own].transpose(0, 1).reshape(-1, D) for t in (out, chains)]
        errs = [e + float((t - want).norm()) ** 2 for e, t in zip(errs, rows)]
        heads.append((rows[0], z, vv))
    _no_further_than_blocks(heads, f"H={H} Hk={Hk} D={D} L={L} S={S}")
    assert errs[0] <= errs[1] * 1.003 ** 2, (errs[0] ** 0.5, errs[1] ** 0.5)
