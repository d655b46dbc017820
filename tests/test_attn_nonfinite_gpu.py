"""Non-finite inputs through the split-context attention: a chunk whose partial has weight 0 still takes part in the merge,
so a NaN or an infinity among its tokens is never dropped in silence."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(32, 8, 128, 8), (16, 4, 256, 8), (8, 8, 64, 1), (16, 4, 256, 1)]


def _inputs(dev, H, Hk, D, S, L):
    g = torch.Generator().manual_seed(D + S)
    r = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)  # noqa: E731
    mask = torch.tensor([(1 << (i + 1)) - 1 for i in range(S)], dtype=torch.int32, device=dev)
    return r(1, H, S, D), r(1, Hk, L + 64, D), r(1, Hk, L + 64, D), torch.tensor([L], dtype=torch.int32, device=dev), \
        r(1, Hk, S, D), r(1, Hk, S, D), mask


@pytest.mark.parametrize("H,Hk,D,S", SHAPES)
def test_a_chunk_of_nan_scores_is_not_dropped(C, dev, H, Hk, D, S):
    """Every key of the first 1024 tokens NaN: the chunks there have no maximum, and the rows' weight sums are NaN, for
    which the merge writes 0 (never the softmax of the other tokens)."""
    q, k, v, sl, xk, xv, mask = _inputs(dev, H, Hk, D, S, 4096)
    k[:, :, :1024] = float("nan")
    assert (C.attn_dpas(q, k, v, sl, xk, xv, mask) == 0).all()


@pytest.mark.parametrize("H,Hk,D,S", SHAPES)
def test_infinite_values_of_an_underflowed_chunk_are_not_dropped(C, dev, H, Hk, D, S):
    """Scores of the first 1024 tokens so low that their chunks' weights underflow to 0, their values infinite: 0 x inf."""
    q, k, v, sl, xk, xv, mask = _inputs(dev, H, Hk, D, S, 4096)
    q.fill_(1.0)
    k.fill_(1.0)
    xk.fill_(1.0)
    k[:, :, :1024] = -300.0  # scores sqrt(D) and -300 sqrt(D)
    v[:, :, :1024] = float("inf")
    assert C.attn_dpas(q, k, v, sl, xk, xv, mask).isnan().all()
