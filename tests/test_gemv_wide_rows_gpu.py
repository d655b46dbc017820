"""The W4A8 GEMV with more row bytes than LDS holds (rows x K above 128 KiB): the rows come from L2 in one launch. Bit for
bit against the oracle at the first shapes past the line, odd chunk counts, partial work-groups, both table forms and
layouts, with and without residual; the shape just below the line stays on the LDS form."""
import numpy as np
import pytest
import torch

from conftest import assert_bits_equal, bits
from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,N,K,G,M", [("fp16", 48, 12288, 128, 11), ("fp16", 272, 8320, 128, 16), ("fp16", 4096, 12288, 256, 13),
                                          ("fp8", 48, 12288, 16, 11), ("fp8", 16, 14848, 64, 9), ("f32", 32, 8320, 128, 16),
                                          ("fp16", 64, 12288, 128, 10)])
@pytest.mark.parametrize("tiled", [True, False])
def test_rows_past_lds_match_oracle(C, dev, form, N, K, G, M, tiled):
    from mdx import _lib, layout
    g = torch.Generator().manual_seed(N + K + M)
    q = torch.randint(-128, 128, (N, K // 2), generator=g, dtype=torch.int8)
    sc = torch.rand(N, generator=g) * 1e-3 + 1e-4
    if form == "fp8":
        s = torch.randint(0, 256, (N, K // G), generator=g, dtype=torch.uint8)
        sf, st = ref.fp8e4m3_to_f32(s.numpy()), s.view(torch.float8_e4m3fn)
    else:
        st = (torch.rand(N, K // G, generator=g) * 30).to(torch.float16 if form == "fp16" else torch.float32)
        sf = st.float().numpy()
    cb = torch.randn(16, generator=g) * 4 if G == 256 else None
    x = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    xs = torch.rand(M, generator=g) * 0.05 + 1e-3
    res = torch.randn(M, N, generator=g).to(torch.bfloat16)
    w = layout.W4((layout.tile_major_codes(q) if tiled else q).to(dev), st.to(dev), sc.to(dev), None if cb is None else cb.to(dev),
                  _lib.LAYOUT_TILE if tiled else _lib.LAYOUT_ROW)
    out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    _lib.gemv_trace()
    C.stream_gemv(x.to(dev), xs.to(dev), [w], [out], residuals=[res.to(dev)])
    tr = _lib.gemv_trace()
    assert len(tr) == 1 and tr[0]["rows"] == M and tr[0]["decode"] in ("table16", "bytes"), tr
    want = ref.w4a8_linear(x.numpy(), xs.numpy(), q.numpy(), sf, sc.numpy(), None if cb is None else cb.numpy(), G, bits(res))
    assert_bits_equal(bits(out), np.asarray(want), "rows past LDS")


@pytest.mark.parametrize("custom,decode", [(False, ["table8"]), (True, None)])
def test_wide_work_groups_fall_back(C, dev, monkeypatch, custom, decode):
    """Six tiles per work-group (a tuning variable): the 16-byte tables of 13 rows x 12288 pass LDS. The default codebook
    takes 8-byte ones, another codebook the two halves, and neither is refused."""
    from mdx import _lib, layout
    monkeypatch.setenv("MDX_GEMV_TPW", "6")
    N, K, G, M = 192, 12288, 128, 13
    g = torch.Generator().manual_seed(6)
    q = torch.randint(-128, 128, (N, K // 2), generator=g, dtype=torch.int8)
    s = (torch.rand(N, K // G, generator=g) * 30).half()
    sc = torch.rand(N, generator=g) * 1e-3 + 1e-4
    cb = torch.randn(16, generator=g) * 4 if custom else None
    x = torch.randint(-127, 128, (M, K), generator=g, dtype=torch.int8)
    xs = torch.rand(M, generator=g) * 0.05 + 1e-3
    w = layout.W4(layout.tile_major_codes(q).to(dev), s.to(dev), sc.to(dev), None if cb is None else cb.to(dev), _lib.LAYOUT_TILE)
    out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    _lib.gemv_trace()
    C.stream_gemv(x.to(dev), xs.to(dev), [w], [out])
    tr = _lib.gemv_trace()
    assert [r["rows"] for r in tr] == ([8, 5] if custom else [13]), tr
    assert decode is None or [r["decode"] for r in tr] == decode, tr
    want = ref.w4a8_linear(x.numpy(), xs.numpy(), q.numpy(), s.float().numpy(), sc.numpy(), None if cb is None else cb.numpy(), G)
    assert_bits_equal(bits(out), np.asarray(want), "six tiles")
