"""The native host path (csrc/native.cpp) against the Python path it stands in
front of: every form of operand that either takes gives the same bits, and what
one refuses the other refuses in the same words."""

from __future__ import annotations

import pytest
import torch

import flash_maxsim_amd as fm
from launches import launches
from conftest import sim
from flash_maxsim_amd import _lib

pytestmark = pytest.mark.gpu

DEV = "cuda"


class _Absent:
    """A native module that takes no call."""

    def __getattr__(self, name):
        return lambda *args: None


def both(monkeypatch, call):
    """(result or error of the call as it is, the same by the Python path alone)."""
    out = []
    for absent in (False, True):
        with monkeypatch.context() as m:
            if absent:
                m.setattr(_lib, "native", lambda: _Absent())
            try:
                out.append(call())
            except Exception as e:  # noqa: BLE001
                out.append((type(e), str(e)))
    return out


def same(a, b):
    if torch.is_tensor(a):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
        return torch.equal(a, b)
    if isinstance(a, tuple) and a and torch.is_tensor(a[0]):
        return len(a) == len(b) and all(same(x, y) for x, y in zip(a, b))
    return a == b


def forms(t):
    """t and other layouts of the same values: rows of a wider buffer (in place and
    off alignment), transposed storage, a copy at an odd address."""
    wide = torch.zeros(*t.shape[:-1], t.shape[-1] + 8, dtype=t.dtype, device=t.device)
    wide[..., : t.shape[-1]] = t
    odd = torch.zeros(*t.shape[:-1], t.shape[-1] + 1, dtype=t.dtype, device=t.device)
    odd[..., 1:] = t
    turned = t.transpose(0, 1).contiguous().transpose(0, 1)
    flat = torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)
    flat[1:] = t.reshape(-1)
    return [t, wide[..., : t.shape[-1]], odd[..., 1:], turned, flat[1:].view(t.shape)]


@pytest.mark.parametrize("dtypes", [("f16", "f16"), ("bf16", "bf16"), ("f16", "bf16"), ("f32", "f32")])
@pytest.mark.parametrize("d", [64, 100, 128, 300])
def test_scoring_forms(monkeypatch, dtypes, d):
    kinds = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
    Q = sim((3, 20, d), 1, torch.float32).to(kinds[dtypes[0]]).to(DEV)
    D = sim((3, 6, 37, d), 2, torch.float32).to(kinds[dtypes[1]]).to(DEV)
    ln = torch.tensor([37, 0, 5, 40, -1, 16], device=DEV)
    idx = torch.randint(-1, 22, (6, 7), generator=torch.Generator().manual_seed(3)).to(DEV)
    lengths = [None, ln, ln.to(torch.int32), ln.to(torch.int32).cpu(), torch.stack([ln, ln], 1).to(torch.int32)[:, 0]]
    for q in forms(Q[0]):
        for x in forms(D[0]):
            for le in lengths:
                assert same(*both(monkeypatch, lambda: fm.flash_maxsim(q, x, le)))
                assert same(*both(monkeypatch, lambda: fm.flash_maxsim_topk(q, x, 4, le)))
            for ix in (idx, idx.to(torch.int32), idx.to(torch.int32).t().contiguous().t()):
                assert same(*both(monkeypatch, lambda: fm.flash_maxsim_sparse(q, x, ix, lengths[2])))
            assert same(*both(monkeypatch, lambda: fm.flash_maxsim_packed(q, fm.pack_docs(x, ln, True))))
    for q in forms(Q):
        for x in forms(D[0]):
            assert same(*both(monkeypatch, lambda: fm.flash_maxsim_batched(q, x, lengths[2])))
        for x in forms(D):
            for le in (None, torch.stack([ln, ln, ln]).to(torch.int32)):
                assert same(*both(monkeypatch, lambda: fm.flash_maxsim_batched(q, x, le, False)))


def test_int8_forms(monkeypatch):
    Q = sim((20, 128), 4, torch.float16).to(DEV)
    codes, sc, mn = (t.to(DEV) for t in fm.quantize_int8(sim((6, 36, 128), 5, torch.float32)))
    ln = torch.tensor([36, 0, 5, 40, -1, 16], dtype=torch.int32, device=DEV)
    wide = torch.zeros(6, 40, 1, dtype=torch.float16, device=DEV)
    wide[:, :36] = sc
    for q in forms(Q) + [Q.float()]:
        for x in forms(codes):
            for s, m in ((sc, mn), (sc[..., 0], mn[..., 0]), (wide[:, :36], mn), (sc.float(), mn)):
                assert same(*both(monkeypatch, lambda: fm.flash_maxsim_int8(q, x, s, m, ln)))
        p = fm.quantize_int8_packed(sim((6, 36, 128), 5, torch.float32).to(DEV), ln, True)
        for docs in (p, p._replace(scales=p.scales.float()), p._replace(tok_group=p.tok_group.clone())):
            assert same(*both(monkeypatch, lambda: fm.flash_maxsim_int8_packed(q, docs)))


@pytest.mark.parametrize("nq", [1, 3])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_training_forms(monkeypatch, nq, dtype):
    Q = sim((nq, 20, 100), 6, torch.float32).to(dtype).to(DEV)
    D = sim((6, 37, 100), 7, torch.float32).to(dtype).to(DEV)
    ln = torch.tensor([37, 1, 5, 37, 9, 16], dtype=torch.int32, device=DEV)
    g = torch.randn(nq, 6, generator=torch.Generator().manual_seed(8)).to(DEV)

    def step(need_q, need_d, grad):
        q = (Q if nq > 1 else Q[0]).clone().requires_grad_(need_q)
        x = D.clone().requires_grad_(need_d)
        s = (fm.flash_maxsim_train_batched if nq > 1 else fm.flash_maxsim_train)(q, x, ln)
        if grad is None:
            s.sum().backward()
        else:
            s.backward(grad)
        return tuple(t for t in (s.detach(), q.grad, x.grad) if t is not None)

    g1 = g if nq > 1 else g[0]
    turned = g.t().contiguous().t() if nq > 1 else torch.stack([g[0], g[0]], 1)[:, 0]
    for need_q, need_d in ((True, True), (True, False), (False, True)):
        for grad in (None, g1, turned, torch.zeros_like(g1)):
            assert same(*both(monkeypatch, lambda: step(need_q, need_d, grad)))


def test_refusals(monkeypatch):
    Q, D = sim((20, 128), 9, torch.float16).to(DEV), sim((6, 36, 128), 10, torch.float16).to(DEV)
    calls = [
        lambda: fm.flash_maxsim(Q, D[0]),
        lambda: fm.flash_maxsim(Q[:, :64], D),
        lambda: fm.flash_maxsim(Q.cpu(), D),
        lambda: fm.flash_maxsim(Q, D, torch.ones(5, dtype=torch.int32, device=DEV)),
        lambda: fm.flash_maxsim_batched(Q, D),
        lambda: fm.flash_maxsim_topk(Q, D, 7),
        lambda: fm.flash_maxsim_topk(Q, D, -1),
        lambda: fm.flash_maxsim_topk(Q, D, 0),
        lambda: fm.flash_maxsim_sparse(Q, D, torch.zeros(5, 2, dtype=torch.int32, device=DEV)),
        lambda: fm.flash_maxsim(Q[:0], D),
        lambda: fm.flash_maxsim(Q, D[:0]),
        lambda: fm.flash_maxsim(Q, D[:, :0]),
    ]
    for call in calls:
        assert same(*both(monkeypatch, call))


def test_native_takes_the_ordinary_calls():
    Q, D = sim((2, 20, 128), 11, torch.float16).to(DEV), sim((6, 36, 128), 12, torch.float16).to(DEV)
    n = _lib.native()
    assert n.score(Q[0], D, None) is not None and n.batched(Q, D, None, True) is not None
    assert n.topk(Q[0], D, 3, None) is not None and n.forward(Q, D, None) is not None
    assert n.score(Q[0].float(), D[..., :100], None) is None  # shapes are the Python path's to refuse
    assert n.score(Q[0].float(), D, None) is not None and n.score(Q[0][:, 1:], D[..., 1:], None) is not None
    assert n.score(Q[0].cpu(), D, None) is None and n.score(Q[0].double(), D, None) is None
    assert n.score(Q[0], [1], None) is None
    with pytest.raises(TypeError):
        n.score(Q[0], D)


@pytest.mark.parametrize("d", [1, 4, 7, 8, 30, 100, 128, 130])
@pytest.mark.parametrize("kinds", [("f32", "f16"), ("bf16", "f16"), ("f16", "f16"), ("bf16", "bf16")])
def test_convert_rows_bitwise_torch(d, kinds):
    """fmx_convert_rows against torch's cast and pad: halfway cases, overflow to
    infinity, fp16 subnormals, NaN, strided rows, sources off alignment."""
    types = {"f16": (torch.float16, 0), "bf16": (torch.bfloat16, 1), "f32": (torch.float32, 2)}
    (src_t, src_c), (dst_t, dst_c) = types[kinds[0]], types[kinds[1]]
    gen = torch.Generator().manual_seed(2800 + d)
    x = torch.randn(3, 21, d + 3, generator=gen)
    x[0] *= 2.0 ** torch.randint(-30, 20, (21, d + 3), generator=gen)
    x[1, :4, 0] = torch.tensor([float("inf"), float("nan"), 65520.0, -65519.0])
    x[2, :5] = torch.tensor([1 + 2.0**-11, 1 + 3 * 2.0**-11, 2.0**-25, 3 * 2.0**-25, 0.0])[:, None]
    x = x.to(src_t).to(DEV)
    dp = (d + 7) // 8 * 8
    for lead in (0, 1, 3):
        for v in (x[..., lead : lead + d], x[..., lead : lead + d].contiguous(), x[:1, :, lead : lead + d].expand(3, 21, d)):
            out = torch.full((3, 21, dp), 7.0, dtype=dst_t, device=DEV)
            _lib.check(_lib.load().fmx_convert_rows(src_c, v.data_ptr(), v.stride(0), v.stride(1), 3, 21, d, None, dst_c,
                                                    out.data_ptr(), dp, torch.cuda.current_stream().cuda_stream))
            want = torch.nn.functional.pad(v.to(dst_t), (0, dp - d))
            nan = torch.isnan(want)
            assert torch.equal(torch.isnan(out), nan)
            assert torch.equal(out.masked_fill(nan, 0).view(torch.int16), want.masked_fill(nan, 0).view(torch.int16))
            ln = torch.tensor([4, -1, 30], dtype=torch.int32, device=DEV)
            part = torch.full_like(out, 7.0)
            _lib.check(_lib.load().fmx_convert_rows(src_c, v.data_ptr(), v.stride(0), v.stride(1), 3, 21, d, ln.data_ptr(),
                                                    dst_c, part.data_ptr(), dp, torch.cuda.current_stream().cuda_stream))
            out[0, 4:], out[1] = 7.0, 7.0
            assert torch.equal(part.view(torch.int16), out.view(torch.int16))


@pytest.mark.parametrize("Nq, B, Lq, Ld, d", [(1, 40, 20, 33, 128), (3, 12, 50, 30, 100), (1, 6, 300, 9, 30), (9, 5, 40, 17, 520),
                                              (2, 4, 30, 40, 1100), (1, 3, 5, 2, 7)])
def test_float32_gradients_are_the_sums(Nq, B, Lq, Ld, d):
    """float32 leaves: gradients against float64 sums over the same argmax, to the
    rounding of an fp32 sum of that many terms, in both writers and past one
    wave's width; the same by a 2-byte store of the same sums for fp16 leaves."""
    gen = torch.Generator().manual_seed(2900 + d)
    Q = (torch.randint(-8, 9, (Nq, Lq, d), generator=gen) / 8).to(DEV)
    D = (torch.randint(-8, 9, (B, Ld, d), generator=gen) / 8).to(DEV)
    g = torch.randn(Nq, B, generator=gen).to(DEV)
    ln = torch.randint(1, Ld + 1, (B,), generator=gen, dtype=torch.int32).to(DEV)
    grads = {}
    for dtype in (torch.float32, torch.float16):
        q, x = Q.to(dtype).requires_grad_(True), D.to(dtype).requires_grad_(True)
        s = fm.flash_maxsim_train_batched(q, x, ln)
        grads[dtype] = torch.autograd.grad(s, (q, x), g)
    _, am = _argmax(Q, D, ln, Nq, B, Lq, Ld, d)
    am = am.view(Nq, B, Lq).long()
    dQ, dD = torch.zeros(Nq, Lq, d, dtype=torch.float64), torch.zeros(B, Ld, d, dtype=torch.float64)
    aQ, aD = dQ.clone(), dD.clone()  # sums of absolute values
    Qc, Dc, gc, amc = Q.double().cpu(), D.double().cpu(), g.double().cpu(), am.cpu()
    for i in range(Nq):
        for b in range(B):
            rows = Dc[b][amc[i, b]]
            dQ[i] += gc[i, b] * rows
            aQ[i] += (gc[i, b] * rows).abs()
            dD[b].index_add_(0, amc[i, b], gc[i, b] * Qc[i])
            aD[b].index_add_(0, amc[i, b], (gc[i, b] * Qc[i]).abs())
    for got, half, want, total, terms in zip(grads[torch.float32], grads[torch.float16], (dQ, dD), (aQ, aD), (B, Nq * Lq)):
        assert got.dtype == torch.float32
        assert ((got.double().cpu() - want).abs() <= terms * 2.0**-24 * total).all()
        assert torch.equal(got.half(), half)


def _argmax(Q, D, ln, Nq, B, Lq, Ld, d):
    from flash_maxsim_amd.flash_maxsim import _launch_fwd, _prep

    return _launch_fwd(_prep(Q, torch.float16), _prep(D, torch.float16), ln, Nq, B, Lq, Ld, d, True, True)


def test_native_launches_on_the_current_stream():
    """A captured call replays on new inputs: it was recorded, so it ran on the
    capturing stream; replays with eager work between them equal the eager result."""
    Q, D = sim((20, 128), 13, torch.float16).to(DEV), sim((60, 36, 128), 14, torch.float16).to(DEV)
    fm.flash_maxsim(Q, D)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fm.flash_maxsim(Q, D)
    for i in range(4):
        D.copy_(sim((60, 36, 128), 20 + i, torch.float16))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, fm.flash_maxsim(Q, D))


@pytest.mark.parametrize("Lq, B, Ld, d", [(1, 1, 1, 4), (16, 7, 128, 128), (17, 8, 129, 128), (32, 301, 300, 128), (32, 5, 77, 100),
                                          (9, 30, 16, 32), (32, 11, 17, 36), (30, 6, 131, 64), (32, 4, 200, 68), (5, 9, 40, 124)])
def test_float32_operands_read_in_place(Lq, B, Ld, d):
    """fp32 docs and query rounded as they are read: the bits of the same call on
    operands cast to fp16, for overflow, subnormals, NaN in and past d, views of
    wider rows, ragged and empty docs, packed and sparse."""
    gen = torch.Generator(device=DEV).manual_seed(3100 + d + Ld)
    store = torch.full((B, Ld, d + 4), float("nan"), device=DEV)
    store[..., :d] = torch.randn(B, Ld, d, generator=gen, device=DEV)
    D = store[..., :d]
    D[0, 0, : d // 2] *= 2.0**-16
    D[B // 2, Ld // 2, 0] = 70000.0
    D[B - 1, Ld - 1, d - 1] = float("nan")
    Q = torch.randn(Lq, d, generator=gen, device=DEV)
    ln = torch.randint(0, Ld + 1, (B,), generator=gen, device=DEV, dtype=torch.int32)
    idx = torch.randint(-1, Lq + 1, (B, min(Lq, 13)), generator=gen, device=DEV, dtype=torch.int32)

    def bits(t):
        return t.nan_to_num(7e30).view(torch.int32)  # NaN's payload may differ

    for x in (D, D.contiguous()):
        assert _lib.load().fmx_fwd_reads_f32(Lq, d)
        for le in (None, ln):
            assert torch.equal(bits(fm.flash_maxsim(Q, x, le)), bits(fm.flash_maxsim(Q.half(), x.half(), le)))
            assert torch.equal(bits(fm.flash_maxsim_sparse(Q, x, idx, le)), bits(fm.flash_maxsim_sparse(Q.half(), x.half(), idx, le)))
        docs = fm.pack_docs(x, ln, True)
        half = docs._replace(tokens=docs.tokens.half())
        assert torch.equal(bits(fm.flash_maxsim_packed(Q, docs)), bits(fm.flash_maxsim_packed(Q.half(), half)))
        v, i = fm.flash_maxsim_topk(Q, x, B, ln)
        w, j = fm.flash_maxsim_topk(Q.half(), x.half(), B, ln)
        assert torch.equal(bits(v), bits(w)) and torch.equal(i, j)
    lib = _lib.load()
    assert not lib.fmx_fwd_reads_f32(33, d) and not lib.fmx_fwd_reads_f32(Lq, 129)


def test_float32_rows_too_far_apart_are_cast():
    """float32 operands whose rows span 2 GiB as they lie (documents and queries in
    token-major storage): not for the kernels to read in place, so they are cast to
    a contiguous copy, and score as the same values do from contiguous rows."""
    B, d = 9, 64
    gen = torch.Generator(device=DEV).manual_seed(3200)
    Q, D = torch.randn(5, d, generator=gen, device=DEV), torch.randn(B, 2, d, generator=gen, device=DEV)
    store = torch.empty(2, (1 << 29) // (18 * d) + 1, d, device=DEV)  # (2 + 16) rows of it are 2 GiB
    far = store[:, :B].transpose(0, 1)
    far.copy_(D)
    assert 18 * far.stride(1) * 4 >= 1 << 31
    apart = torch.empty(5, (1 << 29) // 133 // 4 * 4 + 4, device=DEV)[:, :d]  # 5 + 128 rows
    apart.copy_(Q)
    assert 133 * apart.stride(0) * 4 >= 1 << 31
    ln = torch.tensor([2, 0, 1, 2, 2, 1, 2, 2, 2], dtype=torch.int32, device=DEV)
    idx = torch.randint(-1, 6, (B, 3), generator=gen, device=DEV, dtype=torch.int32)
    docs = fm.pack_docs(D[:2], ln[:2])
    tokens = torch.empty(len(docs.tokens), (1 << 29) // 18 // 4 * 4 + 4, device=DEV)[:, :d]
    tokens.copy_(docs.tokens)
    for q, x in ((Q, far), (apart, D), (apart, far)):
        for le in (None, ln):
            assert torch.equal(fm.flash_maxsim(q, x, le), fm.flash_maxsim(Q, D, le))
            assert same(fm.flash_maxsim_topk(q, x, 4, le), fm.flash_maxsim_topk(Q, D, 4, le))
            assert torch.equal(fm.flash_maxsim_sparse(q, x, idx, le), fm.flash_maxsim_sparse(Q, D, idx, le))
    assert torch.equal(fm.flash_maxsim_packed(Q, docs._replace(tokens=tokens)), fm.flash_maxsim_packed(Q, docs))


def test_calls_from_two_host_threads():
    """Two host threads, each on its own stream, score and train at the same time,
    several times over: operands that are read in place and operands that each call
    converts. Every result, read on its own stream, equals the serial one."""
    import threading

    def work(i):
        gen = torch.Generator().manual_seed(3300 + i)
        Q = torch.randn(3, 40, 100, generator=gen).to(DEV)
        D = torch.randn(150, 60, 100, generator=gen).to(DEV)
        ln = torch.randint(1, 61, (150,), generator=gen, dtype=torch.int32).to(DEV)
        g = torch.randn(3, 150, generator=gen).to(DEV)
        half = torch.randn(150, 60, 128, generator=gen).to(torch.float16).to(DEV)

        def call():
            q, x = Q.detach().requires_grad_(True), D.detach().requires_grad_(True)
            s = fm.flash_maxsim_train_batched(q, x, ln)
            return (fm.flash_maxsim(half[0, :32], half, ln), fm.flash_maxsim(Q[0], D, ln), fm.flash_maxsim(Q[1, :20], D),
                    *fm.flash_maxsim_topk(Q[2], D, 70, ln), s.detach(), *torch.autograd.grad(s, (q, x), g))

        return call

    calls = [work(i) for i in range(2)]
    want = [c() for c in calls]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got, errors = [[], []], []

    def worker(i):
        try:
            with torch.cuda.stream(streams[i]):
                for _ in range(8):
                    got[i].append(calls[i]())
                streams[i].synchronize()
        except Exception as e:  # reported on the main thread
            errors.append(e)

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for i in range(2):
        assert len(got[i]) == 8
        for out in got[i]:
            assert len(out) == len(want[i]) and all(torch.equal(a, b) for a, b in zip(out, want[i]))


@pytest.mark.parametrize("Ld, d, whole", [(13, 24, True), (1, 1, True), (7, 140, True), (8, 128, False), (40, 100, False)])
def test_small_float32_docs_are_converted_whole(Ld, d, whole, tmp_path):
    """Documents of fewer than 1024 elements are not converted by their lengths, a
    workgroup each, but all rows as one; rows past a length (NaN here) reach no score."""
    gen = torch.Generator(device=DEV).manual_seed(3600 + Ld)
    Q, D = (torch.randn(*n, d, generator=gen, device=DEV) for n in ((40,), (3000, Ld)))
    ln = torch.randint(0, Ld + 1, (3000,), generator=gen, device=DEV, dtype=torch.int32)
    D[torch.arange(Ld, device=DEV) >= ln[:, None]] = float("nan")
    assert torch.equal(fm.flash_maxsim(Q, D, ln), fm.flash_maxsim(Q.half(), D.half(), ln))
    grids = [grid for name, grid in launches(lambda: fm.flash_maxsim(Q, D, ln), tmp_path) if "convert_kernel" in name]
    groups = Ld * ((d + 7) // 8 * 2)
    assert len(grids) == 2 and grids[1] == -(-(3000 * groups if whole else groups) // 1024), grids
