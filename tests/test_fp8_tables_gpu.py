"""The W4A8 GEMV's fp8-scale variant (one table per scale byte in LDS) at the edges of its range, bit for bit
against the CPU oracle: groups of 16 / 32 / 64, K from one chunk up (scale rows below 16 bytes are staged as they
lie, longer ones in transposed pieces), K that no slice count divides evenly, one tile and partial work-groups,
both layouts, every scale byte (zeros, subnormals, negatives, NaN, the largest), both codebook forms."""
import numpy as np
import pytest
import torch

from conftest import assert_bits_equal, bits
from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,G", [(16, 128, 16), (48, 384, 64), (16, 256, 16), (80, 1664, 32), (272, 4096, 16),
                                   (1024, 8192, 64), (4096, 2176, 16)])
@pytest.mark.parametrize("default_cb", [True, False])
def test_fp8_group_tables_match_oracle(C, dev, N, K, G, default_cb):
    from mdx import _lib, layout
    g = torch.Generator().manual_seed(N + K + G)
    q = torch.randint(-128, 128, (N, K // 2), generator=g, dtype=torch.int8)
    s = torch.randint(0, 256, (N, K // G), generator=g, dtype=torch.uint8)
    sc = torch.rand(N, generator=g) * 1e-3 + 1e-4
    cb = None if default_cb else torch.randn(16, generator=g) * 4
    sf = ref.fp8e4m3_to_f32(s.numpy())
    for M in (1, 2, 7, 16):
        print(f"case N={N} K={K} G={G} cb={not default_cb} M={M}", flush=True)
        x = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
        xs = torch.rand(M, generator=g) * 0.05 + 1e-3
        want = ref.w4a8_linear(x.numpy(), xs.numpy(), q.numpy(), sf, sc.numpy(), None if cb is None else cb.numpy(), G)
        for tiled in (False, True):
            w = layout.W4((layout.tile_major_codes(q) if tiled else q).to(dev), s.view(torch.float8_e4m3fn).to(dev),
                          sc.to(dev), None if cb is None else cb.to(dev),
                          _lib.LAYOUT_TILE if tiled else _lib.LAYOUT_ROW)
            out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
            _lib.gemv_trace()
            C.stream_gemv(x.to(dev), xs.to(dev), [w], [out])
            assert {r["decode"] for r in _lib.gemv_trace()} == {"bytes"}
            assert_bits_equal(bits(out), np.asarray(want), f"tiled={tiled}")
