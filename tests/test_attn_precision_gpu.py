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
