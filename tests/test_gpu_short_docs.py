"""Many short docs of one query (stream_docs_kernel): a wave scores whole docs, so
the scores of a large call must equal, bit for bit, those of the same docs in
calls small enough for the general kernel, which the other tests pin."""

from __future__ import annotations

import pytest
import torch

import flash_maxsim_amd as fm

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize(
    "Lq, B, Ld, d",
    [(32, 8192, 77, 128), (17, 8193, 1, 128), (32, 8199, 16, 96), (31, 8200, 96, 100), (32, 8207, 33, 72),
     (32, 32768, 17, 128), (24, 32771, 50, 65), (32, 8192, 48, 128), (32, 8201, 80, 100), (32, 16390, 96, 128)],
)
def test_short_docs_equal_general_kernel(Lq, B, Ld, d, dtype):
    gen = torch.Generator(device=DEV).manual_seed(3000 + B + d)
    dp = (d + 7) // 8 * 8
    Q = torch.randn(Lq, d, generator=gen, device=DEV).to(dtype)
    store = torch.full((B, Ld, dp), float("nan"), dtype=dtype, device=DEV)  # NaN past d: never used
    store[..., :d] = torch.randn(B, Ld, d, generator=gen, device=DEV).to(dtype)
    D = store[..., :d]
    lengths = torch.randint(-1, Ld + 2, (B,), generator=gen, device=DEV, dtype=torch.int32)
    lengths[:3] = torch.tensor([0, Ld, 0], dtype=torch.int32)
    D[5, Ld // 2, 0] = float("nan")
    D[6, 0, d - 1] = float("inf")

    def parts(ln):
        return torch.cat([fm.flash_maxsim(Q, D[i : i + 4096], None if ln is None else ln[i : i + 4096])
                          for i in range(0, B, 4096)])

    for ln in (None, lengths):
        want = parts(ln)
        got = fm.flash_maxsim(Q, D, ln)
        assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    for srt in (False, True):
        docs = fm.pack_docs(D, lengths, srt)
        assert torch.equal(fm.flash_maxsim_packed(Q, docs).view(torch.int32), want.view(torch.int32))
    cut = fm.pack_docs(D, lengths)
    cut = cut._replace(tokens=cut.tokens[: cut.tokens.shape[0] // 2])  # docs past the rows read zeros
    assert torch.equal(fm.flash_maxsim_packed(Q, cut)[: B // 8].view(torch.int32), want[: B // 8].view(torch.int32))
    values, idx = fm.flash_maxsim_topk(Q, D, 50, lengths)
    assert torch.equal(values.view(torch.int32), want[idx].view(torch.int32))


@pytest.mark.parametrize("B, Ld", [(40000, 96), (40000, 77)])
def test_long_docs_take_less_than_their_parts(B, Ld):
    """Docs without lengths in one call against the same docs in calls of 8000, too
    few for the kernel of short docs, which takes 1.1 times as long on docs of five
    or six full tiles: one call is the faster (0.91 and 0.86 of the parts' time, by
    that kernel 1.00 and 0.96)."""
    gen = torch.Generator(device=DEV).manual_seed(3400 + Ld)
    Q = torch.randn(32, 128, generator=gen, device=DEV).half()
    D = torch.randn(B, Ld, 128, generator=gen, device=DEV).half()
    calls = {"whole": lambda: fm.flash_maxsim(Q, D),
             "parts": lambda: [fm.flash_maxsim(Q, D[i : i + 8000]) for i in range(0, B, 8000)]}
    best = dict.fromkeys(calls, float("inf"))
    for _ in range(8):
        for name, call in calls.items():
            call()
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(10):
                call()
            end.record()
            torch.cuda.synchronize()
            best[name] = min(best[name], start.elapsed_time(end))
    assert best["whole"] < 0.945 * best["parts"], best
