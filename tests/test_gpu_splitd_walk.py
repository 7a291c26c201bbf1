"""The split-d kernel's walk (256 < d): units of several whole queries or of one
pass of a long query over shared docs, against integer arithmetic, exact in every
sum, so scores and the saved argmax must be equal."""

from __future__ import annotations

import pytest
import torch

import flash_maxsim_amd as fm
from flash_maxsim_amd.flash_maxsim import _launch_fwd
from launches import launches

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize(
    "Nq, Lq, B, Ld, d",
    [
        (5, 32, 300, 20, 384),    # four queries a unit, the second unit with one
        (2, 128, 300, 33, 1024),  # a query a unit, 128 rows
        (7, 20, 130, 17, 512),    # six a unit, rows past the unit's queries
        (3, 43, 260, 50, 300),    # three units: 32 workgroups an XCD do not divide
        (17, 120, 40, 16, 384),   # seventeen units, no XCD mapping
        (9, 8, 600, 31, 260),     # sixteen tokens' room left over
        (6, 32, 140, 48, 768),    # masked width past 512: two queries a unit
        (4, 32, 5, 40, 1024),     # too few docs for units
        (3, 33, 100, 1, 640),     # one-token docs
        (300, 128, 3, 16, 320),   # more units than workgroups that fit
        (130, 128, 7, 20, 264),   # units queued behind those that fit
        (2, 128, 13, 33, 1024),   # fewer docs than groups: not a multiple of eight
        (3, 100, 41, 20, 512),    # the same, three units
        (2, 128, 203, 33, 512),   # up to two docs a group: a workgroup for each
        (20, 64, 30, 20, 384),    # two 64-row queries apart
        (7, 41, 300, 20, 272),    # three 41-row queries a unit, the last with one
        (5, 20, 301, 24, 264),    # three 20-row queries a 64-row unit, the last with two
        (3, 100, 163, 300, 264),  # a workgroup a doc, queued: docs of one length and of several
        (2, 128, 290, 200, 264),  # one round of 128 groups, or a workgroup a doc
        (8, 64, 150, 260, 300),   # 64-row units, two workgroups a CU
        (33, 100, 19, 200, 264),  # no XCD mapping, queued
        (1, 200, 270, 70, 1024),  # passes of one query
        (1, 64, 9, 90, 512),
        (1, 128, 600, 31, 1024),  # one unit of 128 VGPRs
        (1, 1000, 20, 35, 384),
        (2, 200, 70, 30, 384),    # several passes of several queries
        (2, 20, 70, 30, 2048),    # past the walk
    ],
)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_walk_exact_on_integer_grid(Nq, Lq, B, Ld, d, dtype):
    gen = torch.Generator().manual_seed(2700 + d + Lq)
    Q = torch.randint(-2, 3, (Nq, Lq, d), generator=gen)
    D = torch.randint(-2, 3, (B, Ld, d), generator=gen)
    lengths = torch.randint(0, Ld + 1, (B,), generator=gen, dtype=torch.int32)
    lengths[:2] = torch.tensor([Ld, 0], dtype=torch.int32)
    S = torch.mm(D.reshape(-1, d).double().to(DEV), Q.reshape(-1, d).double().t().contiguous().to(DEV))
    S = S.view(B, Ld, Nq * Lq)
    past = torch.arange(Ld)[None, :, None] >= lengths[:, None, None]
    S.masked_fill_(past.to(DEV), float("-inf"))
    best = S.max(dim=1).values  # [B, Nq * Lq]
    first = (S == best[:, None]).to(torch.int32).argmax(dim=1)  # the first place that reaches it
    want = best.view(B, Nq, Lq).sum(dim=2).t()
    want_at = first.view(B, Nq, Lq).transpose(0, 1).reshape(Nq * B, Lq)

    dp = (d + 7) // 8 * 8
    wide = torch.full((Nq, Lq + 1, dp), float("nan"), dtype=dtype, device=DEV)  # queries apart, rows past Lq unread
    wide[:, :Lq, :d] = Q.to(dtype).to(DEV)
    Qd, Dd = wide[:, :Lq, :d], D.to(dtype).to(DEV)
    if d % 8:
        Dd = torch.nn.functional.pad(Dd, (0, dp - d))
    for save in (False, True):
        scores, at = _launch_fwd(Qd, Dd, lengths.to(DEV), Nq, B, Lq, Ld, d, True, save)
        assert torch.equal(scores.double(), want)
        if save:
            live = (lengths > 0).repeat(Nq).to(DEV)
            assert torch.equal(at[live].long(), want_at[live].long())
            assert (at[~live] == 0).all()


def _us(call):
    call()
    best = float("inf")
    for _ in range(6):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(20):
            call()
        end.record()
        torch.cuda.synchronize()
        best = min(best, start.elapsed_time(end) * 50)
    return best


def _batch(Nq, Lq, B, Ld, d):
    gen = torch.Generator(device=DEV).manual_seed(Nq + B)
    Q, D = (torch.randn(n, L, d, generator=gen, device=DEV).half() for n, L in ((Nq, Lq), (B, Ld)))
    return lambda: _launch_fwd(Q, D, None, Nq, B, Lq, Ld, d, True, False)


def test_walk_fills_the_gpu_for_any_number_of_units():
    """130 units do not divide 256 workgroups as 128 do, and take about as long
    (one group of workgroups a unit leaves half the GPU out: 1.8 times)."""
    assert _us(_batch(130, 128, 100, 300, 1024)) < 1.4 * _us(_batch(128, 128, 100, 300, 1024))


def test_walk_of_few_docs_takes_one_doc_a_workgroup():
    """Four units over 15 docs fit the GPU at once, as over 16 (groups rounded down
    to a multiple of eight put two docs on a workgroup: 1.6 times)."""
    assert _us(_batch(4, 128, 15, 600, 1024)) < 1.25 * _us(_batch(4, 128, 16, 600, 1024))


def test_two_long_docs_among_short_ones_do_not_wait_for_each_other():
    """Two units over 200 docs, 128 groups: docs 3 and 131 would fall to one workgroup,
    docs 3 and 4 do not; both pairs take about as long (one workgroup for two long
    docs: 1.8 times)."""
    Q, D = (torch.randn(n, L, 512, device=DEV).half() for n, L in ((2, 128), (200, 2000)))
    times = []
    for other in (131, 4):
        ln = torch.full((200,), 16, dtype=torch.int32, device=DEV)
        ln[[3, other]] = 2000
        times.append(_us(lambda: _launch_fwd(Q, D, ln, 2, 200, 128, 2000, 512, True, False)))
    assert times[0] < 1.3 * times[1], times


@pytest.mark.parametrize(
    "Nq, Lq, B, Ld, d, ragged, blocks, groups",
    [
        (2, 64, 300, 300, 384, False, 4, None),   # 64-row tiles, two a CU
        (16, 32, 140, 300, 264, False, 4, None),
        (60, 40, 102, 300, 320, False, 8, None),  # but three queries in 128 rows
        (2, 64, 358, 100, 512, True, 4, None),    # d = 512: with lengths,
        (2, 64, 358, 100, 512, False, 4, None),   # or few docs
        (2, 64, 665, 100, 512, False, 8, None),
        (2, 128, 15, 300, 1024, False, 8, 16),    # few docs: one a workgroup
        (3, 100, 162, 300, 384, False, 8, 168),   # one length: the fewest rounds of docs,
        (2, 128, 448, 300, 512, False, 8, 128),   # here one
        (2, 128, 332, 1000, 384, True, 8, 336),   # long docs of several lengths: one a workgroup
        (2, 128, 448, 300, 512, True, 8, 128),    # shorter ones: one round
        (2, 128, 192, 72, 512, True, 8, 128),
    ],
)
def test_walk_units_and_groups(Nq, Lq, B, Ld, d, ragged, blocks, groups, tmp_path):
    """How queries are gathered into units and docs into groups on 256 CUs: 16-row
    blocks of the query tile, and doc groups of the launch (None: not looked at)."""
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("256 CUs")
    Q, D = (torch.randn(n, L, d, device=DEV).half() for n, L in ((Nq, Lq), (B, Ld)))
    lengths = torch.randint(1, Ld + 1, (B,), dtype=torch.int32, device=DEV) if ragged else None
    (name, grid), = launches(lambda: fm.flash_maxsim_batched(Q, D, lengths), tmp_path)
    assert f"splitd_fwd_kernel<0, {blocks}," in name
    assert groups is None or grid == groups * Nq, grid


def test_uint8_docs_are_not_loaded_ahead(tmp_path):
    """The walk loads the next fp16 doc's tiles ahead of the current one's end. For
    uint8 docs that took up to a sixth longer: their walk does not (the kernel's last
    template argument)."""
    Q = torch.randn(100, 512, device=DEV).half()
    D = torch.randn(600, 16, 512, device=DEV).half()
    codes = fm.quantize_int8(D)
    (half, _), = launches(lambda: fm.flash_maxsim(Q[:64], D), tmp_path)
    (byte, _), = launches(lambda: fm.flash_maxsim_int8(Q[:64], *codes), tmp_path)
    (long, _), = launches(lambda: fm.flash_maxsim_int8(Q, *codes), tmp_path)
    assert "splitd_fwd_kernel<0, 4, 2, false, false, true, true, true, true>" in half
    assert "splitd_fwd_kernel<2, 4, 2, false, false, true, true, true, false>" in byte
    assert "splitd_fwd_kernel<2, 8, 2, false, false, true, true, true, false>" in long
