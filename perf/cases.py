"""The measured cases of the MaxSim operators: what a program that uses this
package has it do, through the package's public functions.

Three surfaces (padded candidates, packed pairs, all-pairs contrastive), each
in inference and in training, in fp32 / fp16 / bf16, from the smallest calls
(a handful of queries, where latency counts) to the largest configurations of
the benchmark, with ragged lengths, odd sizes, long queries and embedding
widths from 64 to 768.

``listed`` names the cases, ``draw`` gives others of the same ranges,
``prepare`` makes a case's inputs on the GPU from a seed, ``run`` is one pass,
``work`` its unavoidable bytes and operations, ``exact`` its results in 64
bits by plain torch, and ``tolerance`` how far two correct implementations
may be apart.
"""

import math

import torch
import torch.nn.functional as F

import maxsim_amd

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def _padded(name, mode, dtype, b, c, lq, ld, dim, q_lo=None, d_lo=32):
    return dict(name=name, kind="padded", mode=mode, dtype=dtype, b=b, c=c, lq=lq,
                q_lo=lq if q_lo is None else q_lo, ld=ld, d_lo=d_lo, dim=dim)


def _packed(name, mode, dtype, nq, nd, pairs, q_lo, q_hi, d_lo, d_hi, dim, median=0):
    """``median`` > 0: log-normal document lengths around it, else uniform.
    ``pairs`` = 0: every query against its own ``nd / nq`` documents."""
    return dict(name=name, kind="packed", mode=mode, dtype=dtype, nq=nq, nd=nd, pairs=pairs,
                q_lo=q_lo, q_hi=q_hi, d_lo=d_lo, d_hi=d_hi, dim=dim, median=median)


def _contrastive(name, mode, dtype, nq, nb, lq, d_lo, d_hi, dim, dup=0.0, temperature=1.0):
    return dict(name=name, kind="contrastive", mode=mode, dtype=dtype, nq=nq, nb=nb, lq=lq,
                d_lo=d_lo, d_hi=d_hi, dim=dim, dup=dup, temperature=temperature)


def listed():
    return [
        # -- reranking: each query against its own padded candidates
        # the smallest call: 8 queries x 16 candidates in fp32 with the
        # argmax (explaining a match); latency and launches count
        _padded("rerank_tiny_f32_argmax", "argmax", "f32", 8, 16, 32, 300, 128, d_lo=64),
        # an ordinary server batch: 32 queries x 100 candidates
        _padded("rerank_f16", "score", "f16", 32, 100, 32, 256, 128),
        # the largest: a whole evaluation set, 256 x 1000 candidates
        _padded("rerank_large_f16", "score", "f16", 256, 1000, 32, 300, 128),
        # training against 16 mined negatives per query
        _padded("rerank_train_bf16", "train", "bf16", 256, 16, 32, 300, 128, q_lo=8),
        # -- packed pairs
        # an ordinary rerank of ragged rows without padding, every query
        # against its own 100 documents
        _packed("packed_f16", "score", "f16", 32, 3200, 0, 8, 32, 16, 256, 128),
        # distillation over a pool: 20,000 random pairs, long-tailed lengths
        _packed("packed_train_bf16", "train", "bf16", 512, 8192, 20000, 8, 64, 16, 2048, 128,
                median=180),
        # a small odd batch of a narrower model, queries of up to 77 tokens
        _packed("packed_train_odd_bf16", "train", "bf16", 61, 389, 777, 5, 77, 9, 413, 96),
        # -- in-batch contrastive training and evaluation
        # a small batch, loss and gradients in one call
        _contrastive("contrastive_small_bf16", "value_and_grad", "bf16", 64, 64, 32, 64, 512, 128),
        # the largest batch, through autograd, with repeated tokens (exact ties)
        _contrastive("contrastive_large_bf16", "train", "bf16", 512, 512, 32, 128, 1024, 128,
                     dup=0.01),
        # full-precision training
        _contrastive("contrastive_f32", "train", "f32", 72, 72, 32, 64, 512, 128,
                     temperature=0.5),
        # evaluation of long queries: an encoder's padded documents are
        # packed and scored against every query
        _contrastive("contrastive_long_f16", "pack_score", "f16", 150, 501, 96, 40, 512, 128),
        # a wide encoder's embeddings used without a projection
        _contrastive("contrastive_wide_bf16", "train", "bf16", 64, 64, 32, 64, 512, 768),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case.  Sizes are spread over their logarithm; the widths are
    mostly the common 128, with narrower, wider and unaligned ones among them.
    A case larger than the listed ones of its kind is drawn again."""
    while True:
        kind = rng.choice(["padded", "packed", "contrastive", "contrastive"])
        dtype = rng.choice(["bf16", "bf16", "f16", "f16", "f32"])
        dim = rng.choice([64, 96, 128, 128, 128, 128, 256, 300, 384, 768])
        if kind == "padded":
            mode = rng.choice(["score", "score", "argmax", "train"])
            lq = _log_int(rng, 8, 100)
            ld = _log_int(rng, 40, 600)
            case = _padded("", mode, dtype, _log_int(rng, 1, 256), _log_int(rng, 4, 1000), lq, ld,
                           dim, q_lo=rng.randint(max(1, lq // 4), lq),
                           d_lo=rng.randint(1, max(1, ld // 2)))
        elif kind == "packed":
            mode = rng.choice(["score", "argmax", "train"])
            nq, nd = _log_int(rng, 4, 512), _log_int(rng, 16, 8192)
            d_hi = _log_int(rng, 60, 1000)
            case = _packed("", mode, dtype, nq, nd, _log_int(rng, 64, 20000), rng.randint(1, 16),
                           _log_int(rng, 16, 100), rng.randint(1, d_hi // 2), d_hi, dim,
                           median=rng.choice([0, 0, max(1, d_hi // 3)]))
        else:
            mode = rng.choice(["score", "pack_score", "train", "train", "value_and_grad"])
            nq = _log_int(rng, 4, 512)
            nb = max(nq, _log_int(rng, 4, 1024))
            d_hi = _log_int(rng, 40, 1024)
            case = _contrastive("", mode, dtype, nq, nb, _log_int(rng, 8, 128),
                                rng.randint(1, d_hi // 2), d_hi, dim,
                                dup=rng.choice([0.0, 0.0, 0.01]),
                                temperature=rng.choice([1.0, 0.5]))
        del case["name"]
        w = work(case)
        plain = dtype != "f32" and dim in (64, 128)
        if w["bytes"] <= (4e9 if kind == "padded" else 1.2e9) and \
                w["flops"] <= (1.0e12 if plain else 6e10):
            return case


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _rows(shape, dim, dtype, gen):
    """L2-normalised Gaussian rows: what an encoder's head gives."""
    x = torch.randn(*shape, dim, generator=gen, device="cuda")
    return F.normalize(x, dim=-1).to(DTYPES[dtype])


def _lengths(n, lo, hi, gen, median=0):
    """The distribution's own quantiles in an order of the seed's: every seed
    has the same rows in all, so its outputs have the same shapes."""
    at = (torch.arange(n, dtype=torch.float64) + 0.5) / n
    if median:
        x = torch.exp(torch.special.ndtri(at) * 0.6 + math.log(median))
        x = x.round().clamp(lo, hi)
    else:
        x = torch.floor(lo + at * (hi + 1 - lo))
    return x.to(torch.int64)[torch.randperm(n, generator=gen)]


def _offsets(lens):
    off = torch.zeros(lens.numel() + 1, dtype=torch.int64)
    off[1:] = lens.cumsum(0)
    return off


def prepare(case, seed):
    kind, dtype, dim, mode = case["kind"], case["dtype"], case["dim"], case["mode"]
    host = torch.Generator().manual_seed(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed + 1)
    grad = mode == "train"
    state = {"case": case}
    if kind == "padded":
        b, c = case["b"], case["c"]
        q = _rows((b, case["lq"]), dim, dtype, gen)
        d = torch.empty(b, c, case["ld"], dim, dtype=DTYPES[dtype], device="cuda")
        for i in range(b):  # a query's candidates at a time: the largest set is 20 GB
            d[i] = _rows((c, case["ld"]), dim, dtype, gen)
        qlen = _lengths(b, case["q_lo"], case["lq"], host).to(torch.int32)
        dlen = _lengths(b * c, case["d_lo"], case["ld"], host).to(torch.int32).view(b, c)
        state.update(q=q.requires_grad_(grad), d=d.requires_grad_(grad), qlen=qlen.cuda(),
                     dlen=dlen.cuda())
        if grad:  # the positive is the first candidate
            state["targets"] = torch.zeros(b, dtype=torch.int64, device="cuda")
    elif kind == "packed":
        nq, nd, pairs = case["nq"], case["nd"], case["pairs"]
        ql = _lengths(nq, case["q_lo"], case["q_hi"], host)
        dl = _lengths(nd, case["d_lo"], case["d_hi"], host, case["median"])
        if pairs:
            qids = torch.randint(0, nq, (pairs,), generator=host, dtype=torch.int32)
            dids = torch.randint(0, nd, (pairs,), generator=host, dtype=torch.int32)
        else:
            dids = torch.arange(nd, dtype=torch.int32)
            qids = (dids // (nd // nq)).to(torch.int32)
        q = _rows((int(ql.sum()),), dim, dtype, gen)
        d = _rows((int(dl.sum()),), dim, dtype, gen)
        state.update(q=q.requires_grad_(grad), d=d.requires_grad_(grad),
                     qoff=_offsets(ql).to(torch.int32).cuda(),
                     doff=_offsets(dl).to(torch.int32).cuda(), qids=qids.cuda(),
                     dids=dids.cuda(), max_q=int(ql.max()))
        if grad:  # the gradient that a loss over the pairs hands down
            state["dscore"] = torch.randn(qids.numel(), generator=gen, device="cuda")
    else:
        nq, nb = case["nq"], case["nb"]
        q = _rows((nq, case["lq"]), dim, dtype, gen)
        lens = _lengths(nb, case["d_lo"], case["d_hi"], host)
        if mode == "pack_score":
            state.update(q=q, padded=_rows((nb, case["d_hi"]), dim, dtype, gen),
                         lens=lens.to(torch.int32).cuda())
            return state
        off = _offsets(lens)
        d = _rows((int(lens.sum()),), dim, dtype, gen)
        n = int(int(lens.sum()) * case["dup"])
        if n:  # tokens that repeat an earlier one of their document
            doc = torch.randint(0, nb, (n,), generator=host)
            pos = (torch.rand(n, generator=host) * (lens[doc] - 1)).long() + 1
            pos = torch.minimum(pos, lens[doc] - 1)
            src = (torch.rand(n, generator=host) * pos).long()
            to, first = (off[doc] + pos).cuda().unique(return_inverse=True)
            # one source for a token that is picked twice
            pick = torch.zeros_like(to).scatter_reduce_(0, first, (off[doc] + src).cuda(), "amax")
            d[to] = d[pick]
        state.update(q=q.requires_grad_(grad), d=d.requires_grad_(grad),
                     off=off.to(torch.int32).cuda(),
                     targets=torch.arange(nq, device="cuda"))
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind, mode = case["kind"], case["mode"]
    q = state["q"]
    if kind == "padded":
        args = (q, state["d"], state["qlen"], state["dlen"])
        if mode == "score":
            return maxsim_amd.score_candidates_padded(*args)
        if mode == "argmax":
            return maxsim_amd.score_candidates_padded_with_argmax(*args)
        scores = maxsim_amd.score_candidates_padded_train(*args)
        loss = F.cross_entropy(scores, state["targets"])
        return (scores, *torch.autograd.grad(loss, args[:2]))
    if kind == "packed":
        args = (q, state["qoff"], state["d"], state["doff"], state["qids"], state["dids"])
        if mode == "score":
            return maxsim_amd.score_pairs_packed(*args, max_q_len=state["max_q"])
        if mode == "argmax":
            return maxsim_amd.score_pairs_packed_with_argmax(*args, max_q_len=state["max_q"])
        scores = maxsim_amd.score_pairs_packed_train(*args, max_q_len=state["max_q"])
        return (scores, *torch.autograd.grad(scores, (q, state["d"]), state["dscore"]))
    if mode == "pack_score":
        packed, off = maxsim_amd.pack_documents(state["padded"], state["lens"])
        return packed, off, maxsim_amd.score_contrastive(q, packed, off)
    d, off = state["d"], state["off"]
    if mode == "score":
        return maxsim_amd.score_contrastive(q, d, off)
    if mode == "value_and_grad":
        return maxsim_amd.score_contrastive_cross_entropy_value_and_grad(
            q, d, off, temperature=case["temperature"])
    scores = maxsim_amd.score_contrastive_train(q, d, off)
    loss = F.cross_entropy(scores / case["temperature"], state["targets"])
    return (scores, *torch.autograd.grad(loss, (q, d)))


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _mean_length(case):
    if not case.get("median"):
        return (case["d_lo"] + (case["d_hi"] if "d_hi" in case else case["ld"])) / 2
    return min(max(case["median"] * math.exp(0.18), case["d_lo"]), case["d_hi"])


def work(case):
    """Valid rows read once, outputs written once; two operations per
    multiply-add, one product per (query token, document token) of a scored
    pair and, in training, one added row per (pair, query token) on either
    side."""
    s, dim, kind, mode = BYTES[case["dtype"]], case["dim"], case["kind"], case["mode"]
    mean_d = _mean_length(case)
    if kind == "padded":
        mean_q = (case["q_lo"] + case["lq"]) / 2
        pairs = case["b"] * case["c"]
        q_rows, d_rows = case["b"] * mean_q, pairs * mean_d
        q_out, d_out, slots = case["b"] * case["lq"], pairs * case["ld"], case["lq"]
        extra = 4 * (case["b"] + pairs)
    elif kind == "packed":
        mean_q = (case["q_lo"] + case["q_hi"]) / 2
        pairs = case["pairs"] or case["nd"]
        used = case["nd"]
        if case["pairs"]:  # documents that some pair names
            used *= 1 - (1 - 1 / case["nd"]) ** case["pairs"]
        q_rows = q_out = case["nq"] * mean_q
        d_rows, d_out, slots = used * mean_d, case["nd"] * mean_d, case["q_hi"]
        extra = 4 * (case["nq"] + case["nd"] + 2 * pairs)
    else:
        mean_q = case["lq"]
        pairs = case["nq"] * case["nb"]
        q_rows = q_out = case["nq"] * mean_q
        d_rows = d_out = case["nb"] * mean_d
        slots, extra = mean_q, 4 * case["nb"]
    flops = 2 * dim * pairs * mean_q * mean_d
    total = s * dim * (q_rows + d_rows) + 4 * pairs + extra
    if mode == "argmax":
        total += 4 * pairs * slots
    elif mode == "pack_score":
        total += s * dim * d_rows
    elif mode in ("train", "value_and_grad"):
        flops += 2 * 2 * dim * pairs * mean_q
        total += s * dim * (q_out + d_out)
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Scores are 32-bit sums (of exact products, for 16-bit inputs);
    gradients are 32-bit sums rounded to the inputs' type.  Where the two best
    document tokens of a query token are closer than the rounding of the
    32-bit sums, two correct implementations may pick different ones, which
    moves that token's whole gradient row and, with ``argmax``, an index.
    About one token in 10^5 is that close."""
    mode, dtype = case["mode"], case["dtype"]
    if mode in ("train", "value_and_grad"):
        rel = {"f32": 2e-3, "f16": 4e-3, "bf16": 1e-2}[dtype]
        return {"rel": rel, "max": 0.99}
    return {"rel": 2e-6, "max": 2e-5, "differ": 1e-3}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _best(sim):
    """Largest similarity over the last axis, the first index that has it
    (rows that are equal in the inputs may differ in the product's last bits),
    and whether another value is within the rounding of 32-bit sums."""
    top = sim.max(dim=-1, keepdim=True).values
    same = sim >= top - 1e-13
    near = ((sim >= top - 1e-7) & ~same).any()
    return top.squeeze(-1), same.to(torch.uint8).argmax(dim=-1), near


def _gradients(case, near, *grads):
    """In fp32, a token whose two best are that close has no gradient that
    every correct implementation agrees on (in 16 bits the gradients' own
    rounding hides it)."""
    return tuple(None if near and case["dtype"] == "f32" else g for g in grads)


def _exact_padded(case, st):
    q, d = st["q"].detach(), st["d"].detach()
    b, lq, c = case["b"], case["lq"], case["c"]
    scores = torch.zeros(b, c, dtype=torch.float64, device="cuda")
    argmax = torch.zeros(b, c, lq, dtype=torch.int32, device="cuda")
    cols = torch.arange(case["ld"], device="cuda")
    near = torch.zeros((), dtype=torch.bool, device="cuda")
    for i in range(b):
        n = int(st["qlen"][i])
        sim = d[i].double().reshape(-1, case["dim"]) @ q[i, :n].double().T
        sim = sim.view(c, case["ld"], n).transpose(1, 2)
        sim = sim.masked_fill((cols >= st["dlen"][i][:, None])[:, None, :], -math.inf)
        m, a, close = _best(sim)
        near |= close
        scores[i] = m.sum(1)
        argmax[i, :, :n] = a.to(torch.int32)
    if case["mode"] == "score":
        return scores
    if case["mode"] == "argmax":
        return scores, argmax
    w = torch.softmax(scores, dim=1)
    w[torch.arange(b), st["targets"]] -= 1
    w /= b
    dq = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    dd = torch.zeros(d.shape, dtype=torch.float64, device="cuda")
    for i in range(b):
        n = int(st["qlen"][i])
        a = argmax[i, :, :n].long()
        rows = torch.gather(d[i].double(), 1, a[:, :, None].expand(c, n, case["dim"]))
        dq[i, :n] = (rows * w[i][:, None, None]).sum(0)
        flat = (a + torch.arange(c, device="cuda")[:, None] * case["ld"]).reshape(-1)
        add = (q[i, :n].double()[None] * w[i][:, None, None]).reshape(-1, case["dim"])
        dd[i].view(-1, case["dim"]).index_add_(0, flat, add)
    return scores, *_gradients(case, near, dq, dd)


def _exact_packed(case, st):
    q, d = st["q"].detach().double(), st["d"].detach().double()
    qoff, doff = st["qoff"].tolist(), st["doff"].tolist()
    qids, dids = st["qids"].tolist(), st["dids"].tolist()
    of_doc = {}
    for p, j in enumerate(dids):
        of_doc.setdefault(j, []).append(p)
    train = case["mode"] == "train"
    scores = torch.zeros(len(qids), dtype=torch.float64, device="cuda")
    argmax = torch.zeros(len(qids), st["max_q"], dtype=torch.int32, device="cuda")
    dq = torch.zeros(q.shape if train else (0,), dtype=torch.float64, device="cuda")
    dd = torch.zeros(d.shape if train else (0,), dtype=torch.float64, device="cuda")
    slot = torch.arange(st["max_q"], device="cuda")
    near = torch.zeros((), dtype=torch.bool, device="cuda")
    starts, ends = st["qoff"][:-1].long(), st["qoff"][1:].long()
    for j, ps in of_doc.items():
        ps = torch.tensor(ps, device="cuda")
        qi = st["qids"][ps].long()
        rows = starts[qi][:, None] + slot                       # [pairs of j, max_q]
        valid = rows < ends[qi][:, None]
        rows = torch.where(valid, rows, starts[qi][:, None])
        doc = d[doff[j]:doff[j + 1]]
        m, a, close = _best(q[rows] @ doc.T)
        near |= close
        scores[ps] = (m * valid).sum(1)
        argmax[ps] = (a * valid).to(torch.int32)
        if train:
            w = (st["dscore"][ps].double()[:, None] * valid)[..., None]
            dq.index_add_(0, rows.reshape(-1), (doc[a] * w).reshape(-1, case["dim"]))
            dd.index_add_(0, (a + doff[j]).reshape(-1), (q[rows] * w).reshape(-1, case["dim"]))
    if train:
        return scores, *_gradients(case, near, dq, dd)
    return (scores, argmax) if case["mode"] == "argmax" else scores


def _exact_contrastive(case, st):
    q = st["q"].detach().double().reshape(-1, case["dim"])
    nq, nb, lq = case["nq"], case["nb"], case["lq"]
    if case["mode"] == "pack_score":
        off = _offsets(st["lens"].cpu().long())
        keep = torch.arange(case["d_hi"], device="cuda") < st["lens"][:, None]
        packed = st["padded"][keep]
        d = packed.double()
    else:
        off = st["off"].cpu().long()
        d = st["d"].detach().double()
    off = off.tolist()
    scores = torch.empty(nq, nb, dtype=torch.float64, device="cuda")
    near = torch.zeros((), dtype=torch.bool, device="cuda")
    argmax = []
    for j in range(nb):
        m, a, close = _best(q @ d[off[j]:off[j + 1]].T)
        near |= close
        scores[:, j] = m.view(nq, lq).sum(1)
        argmax.append(a)
    if case["mode"] == "score":
        return scores
    if case["mode"] == "pack_score":
        return packed.double(), None, scores
    logits = scores / case["temperature"]
    loss = F.cross_entropy(logits, st["targets"])
    w = torch.softmax(logits, dim=1)
    w[torch.arange(nq), st["targets"]] -= 1
    w /= nq * case["temperature"]
    dq, dd = torch.zeros_like(q), torch.zeros_like(d)
    for j in range(nb):
        wj = w[:, j].repeat_interleave(lq)[:, None]
        dq += d[off[j]:off[j + 1]][argmax[j]] * wj
        dd[off[j]:off[j + 1]].index_add_(0, argmax[j], q * wj)
    first = loss if case["mode"] == "value_and_grad" else scores
    return first, *_gradients(case, near, dq.view(nq, lq, -1), dd)


def exact(case, seed):
    st = prepare(case, seed)
    with torch.no_grad():
        if case["kind"] == "padded":
            return _exact_padded(case, st)
        if case["kind"] == "packed":
            return _exact_packed(case, st)
        return _exact_contrastive(case, st)
