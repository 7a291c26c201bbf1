"""Many short docs of one query (stream_docs_kernel): a wave scores whole docs, so
the scores of a large call must equal, bit for bit, those of the same docs in
calls small enough for the general kernel, which the other tests pin."""

from __future__ import annotations

import pytest
import torch

import flash_maxsim_amd as fm
from launches import launches

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


@pytest.mark.parametrize(
    "B, Ld, ragged, whole",
    [(8192, 48, False, True), (8192, 49, False, False), (40000, 96, False, False), (8191, 40, True, False),
     (8192, 80, True, True), (8192, 81, True, False), (16383, 96, True, False), (16384, 96, True, True),
     (16384, 97, True, False)],
)
def test_short_docs_kernel_takes_what_it_is_faster_for(B, Ld, ragged, whole, tmp_path):
    """The kernel whose waves score whole docs takes a tenth longer for docs of four
    tiles or more that are all long: without lengths it takes up to 48 tokens."""
    Q, D = (torch.randn(*n, 128, device=DEV).half() for n in ((32,), (B, Ld)))
    lengths = torch.randint(1, Ld + 1, (B,), dtype=torch.int32, device=DEV) if ragged else None
    (name, _), = launches(lambda: fm.flash_maxsim(Q, D, lengths), tmp_path)
    assert ("stream_docs_kernel" in name) == whole, name
