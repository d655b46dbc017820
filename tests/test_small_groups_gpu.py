"""The per-weight decode of groups below a chunk with f32 / fp16 scales and the default codebook, bit for bit against the
oracle: all scales within the magnitude table's fast range (|s| <= 15.875), exact ties of rint, and waves that also hold
scales past it, infinities, NaN, negatives, zeros and subnormals."""
import numpy as np
import pytest
import torch

from conftest import assert_bits_equal, bits
from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("G", [16, 32, 64])
@pytest.mark.parametrize("kind", ["fast", "edge", "special"])
def test_small_group_scales_match_oracle(C, dev, dtype, G, kind):
    from mdx import _lib, layout
    g = torch.Generator().manual_seed(G)
    N, K = 96, 1152
    q = torch.randint(-128, 128, (N, K // 2), generator=g, dtype=torch.int8)
    s = (torch.rand(N, K // G, generator=g) - 0.4) * 26
    if kind == "fast":
        s[::3] = torch.round(s[::3] * 4) / 4  # (k s lands on ties)
        s = s.clamp(-15.875, 15.875)
    elif kind == "edge":
        s[::2] = torch.tensor([15.875, -15.875, 15.8751, 16.0, 0.5, -1.5, 127.0, 1e-7])[torch.randint(0, 8, s[::2].shape, generator=g)]
    else:
        s[::2] = torch.tensor([float("nan"), float("inf"), -float("inf"), 0.0, -0.0, 6e4, 1e-40, 20.0])[
            torch.randint(0, 8, s[::2].shape, generator=g)]
    s = s.to(dtype)
    sc = torch.rand(N, generator=g) * 1e-3 + 1e-4
    for M in (1, 3, 16):
        print(f"case {dtype} G={G} {kind} M={M}", flush=True)
        x = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
        xs = torch.rand(M, generator=g) * 0.05 + 1e-3
        w = layout.W4(layout.tile_major_codes(q).to(dev), s.to(dev), sc.to(dev), None, _lib.LAYOUT_TILE)
        out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        C.stream_gemv(x.to(dev), xs.to(dev), [w], [out])
        want = ref.w4a8_linear(x.numpy(), xs.numpy(), q.numpy(), s.float().numpy(), sc.numpy(), None, G)
        assert_bits_equal(bits(out), np.asarray(want), f"M={M}")
