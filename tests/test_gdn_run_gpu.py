"""The Gated-DeltaNet core over a run of rows (mdx_gdn_run): control words that are not valid write nothing at all."""
import pytest
import torch

pytestmark = pytest.mark.gpu

HK, HV, K, SLOTS = 2, 4, 512, 8
CH = (2 * HK + HV) * 128


@pytest.mark.parametrize("tail", [0, 5])
def test_invalid_control_words_write_nothing(C, dev, tail):
    from mdx import _lib
    g = torch.Generator(device=dev).manual_seed(tail)
    bf = lambda *s: torch.randn(*s, generator=g, device=dev).bfloat16()  # noqa: E731
    f32 = lambda *s: torch.rand(*s, generator=g, device=dev)  # noqa: E731
    M = 37
    proj, xn, wa, wb, cw = bf(M, CH), bf(M, K), bf(HV, K), bf(HV, K), bf(CH, 4)
    dt, gd = f32(HV), -f32(HV)
    out = dict(conv=bf(CH, 3), pb=bf(2, SLOTS, CH), qb=bf(2, SLOTS, CH), old=f32(2, SLOTS, HV, 2), rec=f32(HV, 128, 128),
               qkv=bf(M, CH), gates=f32(M, HV, 2), core=bf(M, HV * 128))
    p = _lib.ptr

    def run(words):
        o = {k: t.clone() for k, t in out.items()}
        ctl = torch.tensor(words + [0] * (2 + 3 * SLOTS - len(words)), dtype=torch.int32, device=dev)
        _lib.call("mdx_gdn_run", p(proj), p(xn), p(wa), p(wb), K, p(cw), p(o["conv"]), p(o["pb"]), p(o["qb"]), p(o["old"]),
                  p(ctl), p(dt), p(gd), p(o["rec"]), 128 ** -0.5, p(o["qkv"]), p(o["gates"]), p(o["core"]), M, tail, 0, HK, HV,
                  SLOTS, _lib.stream_of(proj))
        return {k for k in o if not torch.equal(o[k], out[k])}

    every = {"conv", "rec", "qkv", "gates", "core"} | ({"pb", "qb", "old"} if tail else set())
    assert run([2, 0, 3, 1]) == every  # (valid words: everything is written)
    for words in ([SLOTS + 1, 0], [-1, 0], [0, 2], [0, -1], [2, 0, 0, SLOTS], [2, 0, -1, 0], [SLOTS, 1] + [0] * (SLOTS - 1) + [99]):
        print(f"case {words} tail={tail}", flush=True)
        assert run(words) == set(), words
