"""What a program that uses this sampling library has it do, as measurable cases.

Eight families, over the vocabulary of 129,280 tokens that the library is
built for and smaller ones, odd sizes among them:

  seed     one ``TerminalSampler.begin_seed`` call: the first token of a
           request, from one FP32 row and dense host counts
  topk     a decode batch whose rows cut to top-k (with top-p), with or
           without an allow mask, token histories or a logit bias
  whole    a decode batch whose rows keep the whole vocabulary (default
           policy, top-p, min-p), with or without an allow mask or histories
  stress   a large batch of penalised rows with long histories, half of them
           greedy, half of them nearly flat with tied maxima
  verify   exact speculative verification, default policy
  filtered exact speculative verification under top-k / top-p policies
  head     the vocabulary projection with its per-tile records
  history  token histories appended to device count tables

A program keeps its launch marshalled (``PreparedSample`` and its like) while
the buffers stay the same, so ``prepare`` holds one and ``run`` launches it.
All inputs are made on the GPU from the seed.
"""
import math

import numpy as np
import torch

from deepseekrpc_amd import batch
from deepseekrpc_amd.sampling import SamplingPolicy
from deepseekrpc_amd.terminal_sampling import TerminalSampler

VOCAB = 129280
DEV = "cuda"


# ---------------------------------------------------------------------------
# The cases.


def listed():
    return [
        # The first token of a request, as the reference's callers ask for
        # it: one row, latency is everything.
        dict(name="seed_call", op="seed", vocab=VOCAB, policy="topk", top_k=50),
        # One decode step of a full serving batch, per-row temperature /
        # top-k / top-p and a grammar mask; bf16 logits.
        dict(name="topk_bf16_256", op="topk", dtype="bf16", rows=256, vocab=VOCAB, top_k=0, mask=True, hist=0, bias=0,
             probs=False),
        # The same rows as the FP32 logits the terminal stage hands over.
        dict(name="topk_f32_256", op="topk", dtype="f32", rows=256, vocab=VOCAB, top_k=0, mask=True, hist=0, bias=0,
             probs=False),
        # A small batch with repetition penalties over the conversation and a
        # chat-style top-k 50: the most usual penalised request.
        dict(name="penalised_topk_bf16_64", op="topk", dtype="bf16", rows=64, vocab=VOCAB, top_k=50, mask=False,
             hist=4096, bias=0, probs=False),
        # A full batch with no top-k: default, top-p, min-p, both.
        dict(name="whole_bf16_256", op="whole", dtype="bf16", rows=256, vocab=VOCAB, policy="mixed", mask=True, hist=0,
             bias=0, probs=False),
        # The same policies on FP32 rows, with the distributions written out
        # (a speculative step's target and proposal rows need them).
        dict(name="whole_f32_32_probs", op="whole", dtype="f32", rows=32, vocab=VOCAB, policy="mixed", mask=False,
             hist=0, bias=0, probs=True),
        # Penalised rows with top-p only over 4,096-token histories.
        dict(name="penalised_bf16_64", op="whole", dtype="bf16", rows=64, vocab=VOCAB, policy="top_p", mask=False,
             hist=4096, bias=0, probs=False),
        # The largest batch: 1,024 penalised rows, 16,384-token histories,
        # greedy and sampled, half of them nearly tied.
        dict(name="stress_bf16_1024", op="stress", dtype="bf16", rows=1024, vocab=VOCAB, hist=16384),
        # Speculative verification of 32 requests x 4 drafts.
        dict(name="verify_f32_32x4", op="verify", dtype="f32", rows=32, drafts=4, vocab=VOCAB),
        # Verification of 8 requests whose policies cut to top-k and top-p.
        dict(name="filtered_f32_8x4", op="filtered", dtype="f32", rows=8, drafts=4, vocab=VOCAB, policy="topk"),
        # The terminal stage's projection of 32 requests x 5 target rows.
        dict(name="head_160x5120", op="head", rows=160, dim=5120, vocab=VOCAB),
        # Prompt ingestion of a large batch: device history tables from
        # 16,384-token prompts.
        dict(name="history_1024x16384", op="history", rows=1024, vocab=VOCAB, old=0, new=16384),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng):
    """Half the time the library's own vocabulary; else another size from
    16,384 up, a multiple of 8 as padded vocabularies are, or odd."""
    if rng.random() < 0.5:
        return VOCAB
    v = _log(rng, 16384, VOCAB)
    return v if rng.random() < 0.3 else v & ~7


def draw(rng):
    op = rng.choice(["seed", "topk", "topk", "topk", "whole", "whole", "whole", "stress", "verify", "filtered", "head",
                     "history"])
    vocab = _vocab(rng)
    dtype = rng.choice(["bf16", "f32"])
    if op == "seed":
        return dict(op=op, vocab=vocab, policy=rng.choice(["topk", "plain", "penalised"]), top_k=rng.choice([20, 40, 50, 100, 200]))
    if op in ("topk", "whole"):
        rows = _log(rng, 1, 256)
        extra = dict(mask=rng.random() < 0.3, hist=_log(rng, 16, 16384) if rng.random() < 0.4 else 0,
                     bias=_log(rng, 1, 300) if rng.random() < 0.15 else 0, probs=rows <= 16 and rng.random() < 0.5)
        if op == "topk":
            return dict(op=op, dtype=dtype, rows=rows, vocab=vocab, top_k=rng.choice([0, 20, 40, 50, 100, 1000]), **extra)
        return dict(op=op, dtype=dtype, rows=rows, vocab=vocab, policy=rng.choice(["mixed", "plain", "top_p"]), **extra)
    if op == "stress":
        return dict(op=op, dtype="bf16", rows=_log(rng, 256, 1000), vocab=vocab & ~7, hist=_log(rng, 1024, 16384))
    if op == "verify":
        return dict(op=op, dtype=dtype, rows=_log(rng, 1, 32), drafts=rng.randint(1, 4), vocab=vocab)
    if op == "filtered":
        return dict(op=op, dtype=dtype, rows=_log(rng, 1, 8), drafts=rng.randint(1, 4), vocab=vocab,
                    policy=rng.choice(["topk", "top_p"]))
    if op == "head":
        return dict(op=op, rows=_log(rng, 1, 160), dim=256 * rng.randint(4, 20), vocab=vocab & ~127)
    return dict(op=op, rows=_log(rng, 1, 1000), vocab=vocab, old=_log(rng, 1, 8192) if rng.random() < 0.5 else 0,
                new=_log(rng, 1, 16384))


# ---------------------------------------------------------------------------
# Inputs.


class _Inputs:
    """Plain tensors and policies of one sampling case, made from the seed."""


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _spiked(rows, vocab, g):
    """N(0, 1) with 32 tokens per row raised by U[8, 15]: the few likely
    tokens over a broad floor that a language model's rows show."""
    x = torch.randn(rows, vocab, generator=g, device=DEV)
    pos = torch.randint(0, vocab, (rows, 32), generator=g, device=DEV)
    return x.scatter_add_(1, pos, 8 + 7 * torch.rand(rows, 32, generator=g, device=DEV))


_PENALTIES = dict(repetition_penalty=1.1, presence_penalty=0.5, frequency_penalty=0.3)


def _sample_inputs(case, seed):
    g = _generator(seed)
    r = np.random.default_rng(int(seed))
    s = _Inputs()
    op, rows, vocab, hist = case["op"], case["rows"], case["vocab"], case["hist"]
    penalties = dict(_PENALTIES) if hist else {}
    if op == "stress":
        half = rows // 2
        x = torch.randn(rows, vocab, generator=g, device=DEV)
        flat = 2e-3 * torch.rand(rows - half, vocab, generator=g, device=DEV) - 1e-3
        tied = torch.randint(0, vocab, (rows - half, 8), generator=g, device=DEV)
        x[half:] = flat.scatter_(1, tied, flat.amax(1, keepdim=True).expand(-1, 8))
        s.policies = [dict(penalties, **(dict(temperature=0.0) if i % 2 == 0 else dict(temperature=1.0, top_p=0.9)))
                      for i in range(rows)]
    elif op == "topk":
        x = _spiked(rows, vocab, g)
        s.policies = [dict(penalties, temperature=0.7, top_k=case["top_k"], top_p=0.9) if case["top_k"] else
                      dict(penalties, temperature=float(r.uniform(0.2, 1.5)), top_k=int(r.integers(1, 1025)),
                           top_p=float(r.uniform(0.5, 1.0))) for _ in range(rows)]
    elif case["policy"] == "top_p":
        x = 3 * torch.randn(rows, vocab, generator=g, device=DEV)
        s.policies = [dict(penalties, temperature=1.0, top_p=0.95) for _ in range(rows)]
    else:
        x = _spiked(rows, vocab, g)
        kinds = [dict(), dict(temperature=float(r.uniform(0.5, 1.5)), top_p=float(r.uniform(0.8, 0.99))),
                 dict(min_p=0.05), dict(temperature=0.8, top_p=0.95, min_p=0.01)]
        s.policies = [dict(penalties, **(kinds[i % 4] if case["policy"] == "mixed" else {})) for i in range(rows)]
    s.logits = x.to(torch.bfloat16 if case["dtype"] == "bf16" else torch.float32)
    s.uniforms = torch.from_numpy(r.random(rows)).to(DEV)
    s.tokens = torch.randint(0, vocab, (rows, hist), generator=g, device=DEV, dtype=torch.int32) if hist else None
    s.allowed = torch.rand(rows, vocab, generator=g, device=DEV) < 0.9 if case.get("mask") else None
    s.bias = None
    if case.get("bias"):
        s.bias = [{int(t): float(v) for t, v in zip(r.choice(vocab, case["bias"], replace=False),
                                                    r.uniform(-5, 5, case["bias"]))} for _ in range(rows)]
    return s


def _pack(allowed):
    """bool [rows, V] -> int32 [rows, ceil(V / 32)], bit i & 31 of word i >> 5."""
    rows, vocab = allowed.shape
    words = (vocab + 31) // 32
    b = torch.zeros(rows, words * 32, dtype=torch.int64, device=allowed.device)
    b[:, :vocab] = allowed
    w = (b.view(rows, words, 32) << torch.arange(32, device=allowed.device)).sum(-1)
    return torch.where(w >= 2**31, w - 2**32, w).to(torch.int32).contiguous()


def _offsets(rows, length):
    return torch.arange(rows + 1, device=DEV, dtype=torch.int64) * length


def _table(tokens, vocab):
    rows, length = tokens.shape
    return batch.PreparedHistoryAppend(tokens.reshape(-1).contiguous(), _offsets(rows, length),
                                       vocab=vocab).launch().table()


def _verify_inputs(case, seed):
    g = _generator(seed)
    r = np.random.default_rng(int(seed))
    s = _Inputs()
    rows, K, vocab = case["rows"], case["drafts"], case["vocab"]
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    if case["op"] == "verify":
        target = 2 * torch.randn(rows, K + 1, vocab, generator=g, device=DEV)
        s.policies = [dict() for _ in range(rows)]
    else:
        target = _spiked(rows * (K + 1), vocab, g).view(rows, K + 1, vocab)
        s.policies = [dict(temperature=float(r.uniform(0.5, 1.2)), top_p=float(r.uniform(0.8, 0.99)),
                           **(dict(top_k=int(r.integers(20, 200))) if case["policy"] == "topk" else {}))
                      for _ in range(rows)]
    draft = target[:, :K] + 0.5 * torch.randn(rows, K, vocab, generator=g, device=DEV)
    s.target, s.draft = target.to(dt).contiguous(), draft.to(dt).contiguous()
    # The proposals, drawn from the draft rows under the request's policy.
    ids = torch.empty(rows, K, dtype=torch.int32, device=DEV)
    for i in range(rows):
        q = _probabilities(s.draft[i].double(), [s.policies[i]] * K)
        ids[i] = torch.multinomial(q, 1, generator=g)[:, 0].to(torch.int32)
    s.ids = ids
    s.u_accept = torch.from_numpy(r.random((rows, K))).to(DEV)
    s.u_target = torch.from_numpy(r.random(rows)).to(DEV)
    s.limit = torch.full((rows,), 10, dtype=torch.int32, device=DEV)
    return s


def _probabilities(z, policies):
    """Final probabilities of float64 rows ``z`` under the policies' temperature, top-k, min-p and top-p, in
    plain float64 (ties at a cut keep their lowest token ids)."""
    for_each = []
    for row, p in zip(z, policies):
        T = p.get("temperature", 1.0)
        if T == 0.0:
            out = torch.zeros_like(row)
            out[int((row == row.max()).nonzero()[0, 0])] = 1.0
            for_each.append(out)
            continue
        s = (row - row.max()) / T
        k = p.get("top_k", 0)
        if 0 < k < row.numel():
            s = s.clone()
            s[torch.sort(s, descending=True, stable=True).indices[k:]] = -math.inf
        e = torch.exp(s)
        q = e / e.sum()
        if p.get("min_p", 0.0):
            q = torch.where(q < p["min_p"] * q.max(), torch.zeros_like(q), q)
            q = q / q.sum()
        if p.get("top_p", 1.0) < 1.0:
            order = torch.sort(q, descending=True, stable=True)
            before = torch.cumsum(order.values, 0) - order.values
            drop = before >= p["top_p"]
            drop[0] = False
            q = q.clone()
            q[order.indices[drop]] = 0.0
        for_each.append(q / q.sum())
    return torch.stack(for_each)


def _head_inputs(case, seed):
    g = _generator(seed)
    s = _Inputs()
    s.hidden = torch.randn(case["rows"], case["dim"], generator=g, device=DEV).to(torch.bfloat16)
    # Uniform on 2^-10 * [-64, 63]: logits of about N(0, 2.6^2) at dim 5,120.
    s.weight = torch.randint(-64, 64, (case["vocab"], case["dim"]), generator=g, device=DEV, dtype=torch.int8)
    s.weight = s.weight.to(torch.bfloat16) * 2.0**-10
    return s


def _history_inputs(case, seed):
    g = _generator(seed)
    s = _Inputs()
    rows, vocab = case["rows"], case["vocab"]
    ids = lambda n: torch.randint(0, vocab, (rows, n), generator=g, device=DEV, dtype=torch.int32)
    s.old = ids(case["old"]) if case["old"] else None
    s.new = ids(case["new"])
    return s


def prepare(case, seed):
    op = case["op"]
    st = {"op": op}
    if op == "seed":
        g = _generator(seed)
        st["logits"] = 2 * torch.randn(1, case["vocab"], generator=g, device=DEV)
        r = np.random.default_rng(int(seed))
        st["counts"] = np.bincount(r.integers(0, case["vocab"], 64), minlength=case["vocab"]).astype(np.int32)
        st["policy"] = SamplingPolicy(**{"topk": dict(temperature=0.7, top_k=case["top_k"], top_p=0.9), "plain": dict(),
                                         "penalised": dict(temperature=0.7, top_k=case["top_k"], top_p=0.9,
                                                           repetition_penalty=1.1)}[case["policy"]])
        st["sampler"] = TerminalSampler(int(seed), vocabulary=case["vocab"])
    elif op in ("topk", "whole", "stress"):
        s = _sample_inputs(case, seed)
        kw = dict(uniforms=s.uniforms)
        if s.tokens is not None:
            kw["history"] = _table(s.tokens, case["vocab"])
        if s.allowed is not None:
            kw["allow_bits"] = _pack(s.allowed)
        if s.bias is not None:
            kw["bias"] = batch.BiasTable.from_dicts(s.bias, device=DEV)
        if case.get("probs"):
            kw["probs"] = "f32"
        st["call"] = batch.PreparedSample(s.logits, batch.policy_tensor(s.policies, DEV), **kw)
    elif op in ("verify", "filtered"):
        s = _verify_inputs(case, seed)
        st["call"] = batch.PreparedVerify(s.target, s.draft, s.ids, batch.policy_tensor(s.policies, DEV), s.u_accept,
                                          s.u_target, s.limit)
    elif op == "head":
        s = _head_inputs(case, seed)
        st["head"] = batch.vocab_head(s.hidden, s.weight, policies=batch.policy_tensor([dict()], DEV),
                                      rows_per_policy=case["rows"])
    else:
        s = _history_inputs(case, seed)
        table = None
        if s.old is not None:  # at its capacity, as a table that grows on the device is kept: the offsets say what is real
            t = batch.PreparedHistoryAppend(s.old.reshape(-1).contiguous(), _offsets(case["rows"], case["old"]),
                                            vocab=case["vocab"]).launch()
            table = batch.HistoryTable(t.off, *t.out)
        p = batch.PreparedHistoryAppend(s.new.reshape(-1).contiguous(), _offsets(case["rows"], case["new"]), table,
                                        vocab=case["vocab"])
        for t in p.out:  # entries past the total stay as they are
            t.zero_()
        st["call"] = p
    return st


def run(state):
    op = state["op"]
    if op == "seed":
        # abort() restores the random streams, so the same state can be drawn from again.
        work = state["sampler"].begin_seed(state["logits"], policy=state["policy"], counts=state["counts"], remaining=9)
        token = work.decision.pending_token
        work.abort()
        return {"token": token}
    if op in ("topk", "whole", "stress"):
        r = state["call"].launch()
        out = {"tokens": r.tokens, "consumed": r.consumed, "status": r.status}
        if r.probs is not None:
            out["probs"] = r.probs
        return out
    if op in ("verify", "filtered"):
        r = state["call"].launch()
        return {"accepted": r.accepted, "ids": r.ids, "count": r.count, "pending": r.pending, "stop": r.stop,
                "used_accept": r.used_accept, "used_target": r.used_target, "status": r.status}
    if op == "head":
        h = batch.vocab_head_launch(state["head"])
        # The records' fields (dsr_head_part_t) as views: a consumer on the device reads them where they are.
        return {"logits": h.logits, "part_sum": h.parts.view(torch.float64)[..., 0],
                "part_max": h.parts.view(torch.float32)[..., 2], "part_info": h.parts[..., 3]}
    p = state["call"].launch()
    ids, counts, generated = p.out
    return {"offsets": p.off, "ids": ids, "counts": counts, "generated": generated, "status": p.status}


# ---------------------------------------------------------------------------
# What one pass cannot do without, and how exact its results are.


def _distinct(tokens, vocab):
    """Expected distinct ids among ``tokens`` uniform ones."""
    return vocab * -math.expm1(tokens * math.log1p(-1.0 / vocab))


def work(case):
    """Bytes: every input read once, every output written once.  Operations:
    for sampling and verification about four per logit that is read (compare,
    subtract, scale, exp), for the projection its products and sums."""
    op, vocab = case["op"], case["vocab"]
    elt = 2 if case.get("dtype") == "bf16" else 4
    if op == "seed":
        return {"bytes": vocab * 4 + vocab * 4 + 100, "flops": 4 * vocab}
    rows = case["rows"]
    if op in ("topk", "whole", "stress"):
        per = vocab * elt + 68 + 12 * _distinct(case["hist"], vocab) + 12 * case.get("bias", 0)
        per += 4 * ((vocab + 31) // 32) if case.get("mask") else 0
        per += 4 * vocab if case.get("probs") else 0
        return {"bytes": rows * per, "flops": 4.0 * rows * vocab}
    if op in ("verify", "filtered"):
        n = rows * (2 * case["drafts"] + 1) * vocab
        return {"bytes": n * elt + 120 * rows, "flops": 4.0 * n}
    if op == "head":
        d = case["dim"]
        return {"bytes": vocab * d * 2 + rows * (d * 2 + vocab * 4 + vocab // 128 * 16), "flops": 2.0 * rows * d * vocab}
    old, both = _distinct(case["old"], vocab), _distinct(case["old"] + case["new"], vocab)
    return {"bytes": rows * (12 * old + 4 * case["new"] + 12 * both + 28), "flops": float(rows * case["new"])}


def tolerance(case):
    """Tokens, decisions, counts and statuses are whole numbers and exact.
    FP32 probabilities are rounded once from float64; the projection sums
    FP32 products in any order."""
    if case["op"] == "head":
        return {"rel": 4e-6, "max": 4e-5, "differ": 1e-4}
    if case.get("probs"):
        return {"rel": 2e-7, "max": 5e-7}
    return "exact"


def exact(case, seed):
    op = case["op"]
    if op == "head":
        s = _head_inputs(case, seed)
        # Products of these inputs are exact in float64; blocks of columns keep the converted weight small.
        h = s.hidden.double()
        logits = torch.cat([h @ w.double().t() for w in s.weight.split(16384)], 1)
        tiles = logits.view(case["rows"], -1, 128)
        m = tiles.amax(-1)
        return {"logits": logits, "part_sum": torch.exp(tiles - m[..., None]).sum(-1), "part_max": m, "part_info": None}
    if not case.get("probs"):
        return None
    s = _sample_inputs(case, seed)
    x = s.logits.double()
    for i, p in enumerate(s.policies):
        if s.tokens is not None:
            c = torch.bincount(s.tokens[i], minlength=case["vocab"]).double()
            rep = p["repetition_penalty"]
            x[i] = torch.where(c > 0, torch.where(x[i] >= 0, x[i] / rep, x[i] * rep), x[i])
            x[i] -= p["presence_penalty"] * (c > 0).double() + p["frequency_penalty"] * c
        if s.bias is not None:
            for t, v in s.bias[i].items():
                x[i, t] += v
    if s.allowed is not None:
        x = torch.where(s.allowed, x, torch.full_like(x, -math.inf))
    return {"tokens": None, "consumed": None, "status": None, "probs": _probabilities(x, s.policies)}
