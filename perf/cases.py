"""Measured cases of MaxSim scoring, training and storage on one GPU.

Each case is one call (or one forward and backward) of a public function of
flash_maxsim_amd on data that is already on the GPU, the way retrieval programs
call it: rerank a few candidates, scan a collection, score a batch of queries,
train an encoder, encode and decode stored documents. `listed` holds the sizes
that stand for each use, `draw` more of the same uses over their whole range.

Rows are N(0, 1) vectors normalised to unit length, as multi-vector encoders
emit them. "ragged" cases have one length per document, spread evenly over
[Ld / 32, Ld] in an order of the seed's.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import flash_maxsim_amd as fm

DEV = "cuda"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
CHUNK = 1 << 26  # elements made, or scored in 64 bits, at a time


def listed():
    return [
        # one query against a first stage's hundred candidates, ragged: the smallest call, where latency counts
        {"name": "rerank_100", "call": "score", "dtype": "f16", "Lq": 32, "B": 100, "Ld": 300, "d": 128, "ragged": True},
        # one query against a shard of a collection: the benchmark's metric
        {"name": "scan_5000", "call": "score", "dtype": "f16", "Lq": 32, "B": 5000, "Ld": 300, "d": 128,
         "ragged": False},
        # one query against passages of sentence length, the best hundred returned
        {"name": "passages_top100", "call": "topk", "dtype": "f16", "Lq": 32, "B": 20000, "Ld": 77, "d": 128, "k": 100,
         "ragged": True},
        # page images: a thousand patch vectors on both sides, in the encoder's bf16
        {"name": "pages_bf16", "call": "score", "dtype": "bf16", "Lq": 1024, "B": 1000, "Ld": 1024, "d": 128,
         "ragged": False},
        # a batch of queries against one shard: evaluation runs, distillation
        {"name": "batch_100", "call": "batched", "dtype": "f16", "Nq": 100, "Lq": 32, "B": 5000, "Ld": 300, "d": 128,
         "ragged": False},
        # one query against a compressed shard of ragged documents
        {"name": "int8_ragged", "call": "int8", "Lq": 32, "B": 5000, "Ld": 1024, "d": 128, "ragged": True},
        # the same documents under a long query
        {"name": "int8_long_query", "call": "int8", "Lq": 128, "B": 5000, "Ld": 1024, "d": 128, "ragged": True},
        # candidates scored with the sixteen query tokens that a filter kept for each
        {"name": "sparse_1000", "call": "sparse", "dtype": "f16", "Lq": 32, "K": 16, "B": 1000, "Ld": 300, "d": 128,
         "ragged": True},
        # training step on one query and its candidates, wide embeddings
        {"name": "train_wide", "call": "train", "dtype": "f16", "Nq": 1, "Lq": 128, "B": 1000, "Ld": 512, "d": 1024,
         "ragged": False},
        # training step with in-batch negatives, float32 embeddings as a normalising layer emits them
        {"name": "train_batch", "call": "train", "dtype": "f32", "Nq": 32, "Lq": 32, "B": 256, "Ld": 180, "d": 128,
         "ragged": True},
        # an index built: ragged float32 documents into packed 8-bit storage
        {"name": "encode_packed", "call": "encode", "dtype": "f32", "B": 5000, "Ld": 300, "d": 128, "ragged": True,
         "packed": True},
        # stored documents read back as float32
        {"name": "decode", "call": "decode", "B": 2000, "Ld": 512, "d": 128},
    ]


def _spread(rng, lo, hi):
    """A whole number in [lo, hi], uniform in its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["score", "score", "batched", "topk", "int8", "int8", "sparse", "train", "train", "encode",
                       "decode", "pack"])
    while True:
        # mostly query-sized inputs, some longer, page images at the end of the range
        Lq = rng.choice([32, 32, rng.randint(8, 64), rng.randint(65, 256), _spread(rng, 256, 1024)])
        d = rng.choice([128, 128, 128, 128, 96, 64, 100, 256, 384, 1024])
        B, Ld, ragged = _spread(rng, 20, 20000), _spread(rng, 40, 1100), rng.random() < 0.6
        dtype = rng.choice(["f16", "f16", "bf16", "f32"])
        case = {"call": call, "dtype": dtype, "Lq": Lq, "B": B, "Ld": Ld, "d": d, "ragged": ragged}
        if call == "batched":
            case.update(Nq=_spread(rng, 2, 128), Lq=min(Lq, 128))
        elif call == "topk":
            case["k"] = min(B, rng.choice([10, 100, 1000]))
        elif call == "int8":
            del case["dtype"]
            case["packed"] = rng.random() < 0.4
        elif call == "sparse":
            case["K"] = max(1, min(Lq, 128) * rng.choice([25, 50, 75]) // 100)
        elif call == "train":
            # one query and its candidates, or a batch of short queries with in-batch negatives
            case["Nq"] = rng.choice([1, _spread(rng, 2, 64)])
            case["Lq"] = min(Lq, 256 if case["Nq"] == 1 else 64)
            case["B"] = B = min(B, 2000)
        elif call in ("encode", "pack"):
            del case["Lq"]
            if call == "encode":
                case["packed"] = ragged
        elif call == "decode":
            case = {"call": call, "B": B, "Ld": Ld, "d": d}
        w = work(case)
        if w["bytes"] < 2.1e9 and w["flops"] < 6e11:
            return case


# ---- inputs ----

def _rows(gen, shape, dtype):
    """Unit-length rows of N(0, 1) values, made a part at a time."""
    out = torch.empty(shape, dtype=dtype, device=DEV)
    flat = out.view(-1, shape[-1])
    step = max(1, CHUNK // shape[-1])
    for i in range(0, flat.shape[0], step):
        part = flat[i:i + step]
        part.copy_(F.normalize(torch.randn(part.shape, generator=gen, device=DEV), dim=-1))
    return out


def _lengths(gen, case):
    if not case.get("ragged"):
        return None
    low, high = max(1, case["Ld"] // 32), case["Ld"]
    even = torch.linspace(low, high, case["B"], device=DEV).round().to(torch.int32)
    return even[torch.randperm(case["B"], generator=gen, device=DEV)]


def _codes(gen, shape):
    """8-bit codes and the fp16 step and minimum of each token, as the stored format defines them."""
    codes = torch.empty(shape, dtype=torch.uint8, device=DEV)
    scales = torch.empty(*shape[:2], 1, dtype=torch.float16, device=DEV)
    mins = torch.empty_like(scales)
    step = max(1, CHUNK // (shape[1] * shape[2]))
    for i in range(0, shape[0], step):
        x = _rows(gen, (min(step, shape[0] - i),) + tuple(shape[1:]), torch.float32)
        lo, hi = torch.aminmax(x, dim=-1, keepdim=True)
        s = torch.clamp_min((hi - lo) / 255.0, 1e-8)
        codes[i:i + step] = torch.clamp(torch.round((x - lo) / s), 0, 255).to(torch.uint8)
        scales[i:i + step], mins[i:i + step] = s.half(), lo.half()
    return codes, scales, mins


def _inputs(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    call, d = case["call"], case["d"]
    x = {"lengths": _lengths(gen, case)}
    shape = (case["B"], case["Ld"], d)
    if call in ("int8", "decode"):
        x["codes"], x["scales"], x["mins"] = _codes(gen, shape)
    else:
        x["D"] = _rows(gen, shape, DTYPES[case["dtype"]])
    if "Lq" in case:
        nq = (case["Nq"],) if case.get("Nq", 1) > 1 else ()
        dtype = DTYPES[case["dtype"]] if "dtype" in case else torch.float16
        x["Q"] = _rows(gen, nq + (case["Lq"], d), dtype)
    if call == "sparse":
        # the K query tokens of each document, in the query's order
        pick = torch.rand(case["B"], case["Lq"], generator=gen, device=DEV).topk(case["K"], dim=1).indices
        x["indices"] = pick.sort(dim=1).values.to(torch.int32)
    if call == "train":
        # the loss's gradient: what a softmax over the documents sends back
        nq = case["Nq"]
        g = torch.softmax(torch.randn(nq, case["B"], generator=gen, device=DEV), dim=1)
        g[:, 0] -= 1.0
        x["grad"] = g if nq > 1 else g[0]
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    if case["call"] == "train":
        x["Q"].requires_grad_(True)
        x["D"].requires_grad_(True)
    elif case["call"] == "int8" and case.get("packed"):
        x["packed"] = _pack_codes(x)
    return {"case": case, **x}


def _pack_codes(x):
    """The codes of the documents back to back on 4-token groups: a collection stored without padding."""
    codes, lengths = x.pop("codes"), x["lengths"]
    scales, mins = x.pop("scales")[..., 0], x.pop("mins")[..., 0]
    B, Ld, d = codes.shape
    if lengths is None:
        lengths = torch.full((B,), Ld, dtype=torch.int32, device=DEV)
    pad = (lengths.long() + 3) // 4 * 4
    start = torch.cumsum(pad, 0) - pad
    T = int(pad.sum())
    j = torch.arange(Ld, device=DEV)
    keep = j[None, :] < lengths[:, None]
    at = (start[:, None] + j[None, :])[keep]
    out = [torch.zeros(T, d, dtype=torch.uint8, device=DEV), *(torch.zeros(T, dtype=torch.float16, device=DEV)
                                                               for _ in range(2))]
    for to, of in zip(out, (codes, scales, mins)):
        to[at] = of[keep]
    return fm.PackedInt8Docs(*out, start // 4, lengths, int(lengths.max()))


# ---- the calls ----

def run(s):
    case = s["case"]
    call = case["call"]
    if call == "score":
        return fm.flash_maxsim(s["Q"], s["D"], s["lengths"])
    if call == "batched":
        return fm.flash_maxsim_batched(s["Q"], s["D"], s["lengths"])
    if call == "topk":
        return fm.flash_maxsim_topk(s["Q"], s["D"], case["k"], s["lengths"])
    if call == "int8":
        if case.get("packed"):
            return fm.flash_maxsim_int8_packed(s["Q"], s["packed"])
        return fm.flash_maxsim_int8(s["Q"], s["codes"], s["scales"], s["mins"], s["lengths"])
    if call == "sparse":
        return fm.flash_maxsim_sparse(s["Q"], s["D"], s["indices"], s["lengths"])
    if call == "train":
        step = fm.flash_maxsim_train if case["Nq"] == 1 else fm.flash_maxsim_train_batched
        scores = step(s["Q"], s["D"], s["lengths"])
        dQ, dD = torch.autograd.grad(scores, (s["Q"], s["D"]), s["grad"])
        return scores.detach(), dQ, dD
    if call == "encode":
        if case["packed"]:
            return fm.quantize_int8_packed(s["D"], s["lengths"])
        return fm.quantize_int8(s["D"])
    if call == "decode":
        return fm.dequantize_int8(s["codes"], s["scales"], s["mins"])
    if call == "pack":
        return fm.pack_docs(s["D"], s["lengths"])
    raise ValueError(call)


def work(case):
    """Every input read once, every output written once; ragged documents count their mean length."""
    call, B, Ld, d = case["call"], case["B"], case["Ld"], case["d"]
    tokens = B * Ld
    if case.get("ragged"):
        tokens = B * (max(1, Ld // 32) + Ld) / 2
    esz = {"f16": 2, "bf16": 2, "f32": 4}.get(case.get("dtype"), 1)
    nq = case.get("Nq", 1)
    rows = nq * case.get("Lq", 0)  # query tokens
    per_doc = case["K"] if call == "sparse" else rows
    if call in ("int8", "decode"):
        docs = tokens * (d + 4)
    else:
        docs = tokens * d * esz
    query = rows * d * (esz if "dtype" in case else 2)
    flops = 2.0 * per_doc * tokens * d
    if call == "train":
        # documents read, their gradient (padding included) written, and the same for the queries; the
        # gradients' sums are small beside the forward's products
        return {"bytes": docs + B * Ld * d * esz + 2 * query + 8 * nq * B, "flops": flops + 4.0 * rows * B * d}
    if call == "encode":
        return {"bytes": docs + tokens * (d + 4), "flops": 0}
    if call == "pack":
        return {"bytes": 2 * docs, "flops": 0}
    if call == "decode":
        return {"bytes": docs + tokens * d * 4, "flops": 0}
    out = 4 * nq * B + 12 * case.get("k", 0) + (4 * B * case["K"] if call == "sparse" else 0)
    return {"bytes": docs + query + out, "flops": flops}


def tolerance(case):
    call = case["call"]
    if call in ("encode", "pack", "decode"):
        return "exact"  # bytes, moved values, and one rounded multiply and add per value
    if call == "train":
        # gradients are fp16 or bf16 numbers (bf16: eight bits), whatever the leaves hold
        return {"rel": 1e-2, "max": 3e-2} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 4e-3}
    if call == "int8":
        # decoded values may be rounded to fp16 before the products or not
        return {"rel": 3e-5, "max": 3e-4}
    # float32 sums of float32 maxima
    tol = {"rel": 1e-6, "max": 1e-5}
    if call == "topk":
        tol["differ"] = 0.01  # neighbours in rank whose scores agree to the last bits
    return tol


# ---- the same in 64 bits ----

def _operand(t):
    """What the functions score: fp16 values, unless the input is bf16 (float32 is cast to fp16)."""
    return (t.detach() if t.dtype == torch.bfloat16 else t.detach().half()).double()


def _best(Q, docs, lengths, first):
    """Per document of `docs` (float64 [b, Ld, d]) and query token: the best similarity and its place."""
    b, Ld, d = docs.shape
    S = torch.mm(docs.reshape(b * Ld, d), Q.reshape(-1, d).t().contiguous()).view(b, Ld, -1)
    if lengths is not None:
        past = torch.arange(Ld, device=DEV)[None, :] >= lengths[first:first + b, None]
        S.masked_fill_(past[:, :, None], float("-inf"))
    return S.max(dim=1)


def exact(case, seed):
    x = _inputs(case, seed)
    call, B, Ld, d = case["call"], case["B"], case["Ld"], case["d"]
    if call == "pack":
        return None  # values are moved, none is computed
    if call == "decode":
        return x["codes"].double() * x["scales"].double() + x["mins"].double()
    if call == "encode":
        lo, hi = (v.double() for v in torch.aminmax(x["D"], dim=-1, keepdim=True))
        step = ((hi - lo) / 255.0).clamp_min(1e-8)
        if not case["packed"]:
            return None, step, lo
        lengths = x["lengths"].long()
        pad = (lengths + 3) // 4 * 4
        start = torch.cumsum(pad, 0) - pad
        j = torch.arange(Ld, device=DEV)
        keep = j[None, :] < lengths[:, None]
        at = (start[:, None] + j[None, :])[keep]
        out = []
        for v in (step, lo):
            t = torch.zeros(int(pad.sum()), dtype=torch.float64, device=DEV)
            t[at] = v[..., 0][keep]
            out.append(t)
        return (None, *out, None, None, None)

    Q = _operand(x["Q"])
    nq, Lq = case.get("Nq", 1), case["Lq"]
    Qr = Q.reshape(nq * Lq, d)
    scores = torch.empty(nq, B, dtype=torch.float64, device=DEV)
    train = call == "train"
    if train:
        grad = x["grad"].double().view(nq, B)
        dQ = torch.zeros_like(Qr)
        dD = torch.zeros(B, Ld, d, dtype=torch.float64, device=DEV)
    step = max(1, CHUNK // (Ld * max(d, nq * Lq)))
    for i in range(0, B, step):
        n = min(step, B - i)
        if call == "int8":
            docs = x["codes"][i:i + n].double() * x["scales"][i:i + n].double() + x["mins"][i:i + n].double()
        else:
            docs = _operand(x["D"][i:i + n])
        best, at = _best(Qr, docs, x["lengths"], i)  # [n, nq * Lq]
        if call == "sparse":
            best = best.gather(1, x["indices"][i:i + n].long())
        scores[:, i:i + n] = best.view(n, nq, -1).sum(dim=2).t()
        if train:
            g = grad[:, i:i + n].t().repeat_interleave(Lq, dim=1)  # [n, nq * Lq]
            for k in range(n):
                rows = docs[k][at[k]]  # [nq * Lq, d]
                dQ += g[k][:, None] * rows
                dD[i + k].index_add_(0, at[k], g[k][:, None] * Qr)
    if train:
        return (scores if nq > 1 else scores[0]), dQ.view_as(x["Q"]), dD
    if call == "topk":
        return torch.topk(scores[0], case["k"]).values, None
    return scores if call == "batched" else scores[0]
