"""The work a user of this package has it do, as timed cases.

Every case is one call (or one decode step's calls) through the public entry
points, with what a serving program holds before it: logits or hidden states of
the step, the vocabulary head's weight, the KV pool, the decision policy.

Kinds and their ranges (`draw` takes more cases of the same ranges):

  greedy   verify.greedy_verify: batch 1 .. 256, k 1 .. 8, vocabulary 8000 ..
           152064 (any, odd ones too), f32 / bf16 / f16, draft logits or ids
  spec     verify.speculative_verify (and, with `draft`, verify.sample_logits
           of the draft rows before it): batch 1 .. 128, k 1 .. 6, vocabulary a
           multiple of 8, temperature, top-p, top-k, repetition penalty
  filter   verify.filter_logits: 1 .. 256 rows to the dense filtered rows
  head     the vocabulary head: lm_head_greedy_verify, lm_head_argmax and
           lm_head_logits, 1 .. 2304 rows, hidden size 512 .. 4096
  kv       graph_ops.commit_kv: accepted branch tokens into the paged pool
  policy   SamplingDecisionPolicy.queue and .read over mixed endpoint rows
"""

from __future__ import annotations

from types import SimpleNamespace

import numpy as np
import torch

from loopspec_amd import verify
from loopspec_amd.loopspec import graph_ops
from loopspec_amd.loopspec.pipeline import PipelineLane
from loopspec_amd.loopspec.sampling.policy import SamplingDecisionPolicy
from loopspec_amd.loopspec.sampling.sampler import CategoricalSampler

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
# the most a drawn case may read and write, and the most it may multiply
MOST_BYTES = 1.3e9
MOST_FLOPS = 1.3e12


def _greedy(name, batch, k, vocab, dtype, ids=False):
    return {"name": name, "kind": "greedy", "batch": batch, "k": k, "vocab": vocab, "dtype": dtype, "ids": ids}


def _spec(name, batch, k, vocab, dtype, temperature, top_p, top_k=0, penalty=1.0, hist_max=0, draft=False, std=3.0):
    return {"name": name, "kind": "spec", "batch": batch, "k": k, "vocab": vocab, "dtype": dtype,
            "temperature": temperature, "top_p": top_p, "top_k": top_k, "penalty": penalty, "hist_max": hist_max,
            "draft": draft, "std": std}


def _filter(name, rows, vocab, dtype, temperature, top_p, top_k=0):
    return {"name": name, "kind": "filter", "rows": rows, "vocab": vocab, "dtype": dtype, "temperature": temperature,
            "top_p": top_p, "top_k": top_k, "std": 3.0}


def _head(name, op, batch, k, hidden, vocab):
    return {"name": name, "kind": "head", "op": op, "batch": batch, "k": k, "hidden": hidden, "vocab": vocab}


def _kv(name, batch, k, planes, token_bytes, page_size):
    return {"name": name, "kind": "kv", "batch": batch, "k": k, "planes": planes, "token_bytes": token_bytes,
            "page_size": page_size}


def _policy(name, vocab, q1, q2, direct, verified, second, temperature, top_p, dtype, std):
    return {"name": name, "kind": "policy", "vocab": vocab, "q1": q1, "q2": q2, "direct": direct,
            "verified": verified, "second": second, "temperature": temperature, "top_p": top_p, "dtype": dtype,
            "std": std}


def listed():
    return [
        # one interactive sequence, greedy: the smallest step, all latency
        _greedy("greedy_single", 1, 2, 49152, "f32"),
        # a serving batch, greedy: 320 endpoint rows of a step
        _greedy("greedy_batch", 64, 2, 49152, "bf16"),
        # a batch whose vocabulary is odd, so that rows lie at any alignment;
        # the proposals come as ids from a separate drafter
        _greedy("greedy_ragged", 96, 3, 50257, "f16", ids=True),
        # one interactive sequence, sampled: the draft tokens are drawn, then verified
        _spec("spec_single", 1, 4, 32000, "bf16", 0.8, 0.95, top_k=50, draft=True),
        # a serving batch, sampled with top-p
        _spec("spec_batch", 64, 2, 49152, "f32", 1.0, 0.7),
        # a serving batch at a large vocabulary with a repetition penalty over the token history
        _spec("spec_penalty", 32, 4, 128256, "bf16", 0.7, 0.9, penalty=1.1, hist_max=4096, std=4.0),
        # dense filtered distributions of a batch's rows, for a program that draws by itself
        _filter("filter_rows", 64, 49152, "f32", 1.0, 0.7),
        # one sequence from hidden states: the head's weight is streamed for three rows
        _head("head_single", "verify", 1, 2, 2048, 49152),
        # a serving batch from hidden states (k = 2, target and draft rows)
        _head("head_batch", "argmax", 64, 2, 2048, 49152),
        # the largest: a full batch's logits for sampling, wide hidden states, large vocabulary
        _head("head_logits", "logits", 256, 4, 4096, 128256),
        # the accepted tokens of a step move from their branch slots into the paged KV pool
        _kv("kv_commit", 64, 2, 192, 4096, 16),
        # one cycle of the decision policy a pipeline drives, host readback included
        _policy("policy_cycle", 49152, 16, 16, 8, 24, 12, 1.0, 0.7, "f32", 3.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _draw_once(rng):
    kind = rng.choice(["greedy", "spec", "filter", "head", "head", "kv", "policy"])
    if kind == "greedy":
        vocab = rng.choice([_log_int(rng, 8000, 152064), 8 * _log_int(rng, 1000, 19008)])
        c = _greedy("", _log_int(rng, 1, 256), rng.randint(1, 8), vocab, rng.choice(["f32", "bf16", "f16"]),
                    rng.random() < 0.4)
    elif kind == "spec":
        pen = rng.random() < 0.35
        c = _spec("", _log_int(rng, 1, 128), rng.randint(1, 6), 8 * _log_int(rng, 1000, 19008),
                  rng.choice(["f32", "bf16", "f16"]), rng.choice([0.6, 0.7, 0.9, 1.0]),
                  rng.choice([0.7, 0.9, 0.95, 1.0]), rng.choice([0, 0, 0, 20, 50]), 1.1 if pen else 1.0,
                  _log_int(rng, 64, 8192) if pen else 0, rng.random() < 0.3, rng.choice([3.0, 4.0]))
    elif kind == "filter":
        c = _filter("", _log_int(rng, 1, 256), 8 * _log_int(rng, 1000, 19008), rng.choice(["f32", "bf16", "f16"]),
                    rng.choice([0.6, 0.7, 0.9, 1.0]), rng.choice([0.7, 0.9, 0.95]), rng.choice([0, 0, 50]))
    elif kind == "head":
        op = rng.choice(["verify", "argmax", "logits"])
        c = _head("", op, _log_int(rng, 1, 256), rng.randint(1, 4), 64 * _log_int(rng, 8, 64),
                  _log_int(rng, 8000, 128256))
    elif kind == "kv":
        c = _kv("", _log_int(rng, 1, 128), rng.randint(1, 8), 2 * _log_int(rng, 8, 96),
                rng.choice([1024, 2048, 4096]), rng.choice([1, 16, 64]))
    else:
        second = rng.randint(0, 8)
        c = _policy("", 8 * _log_int(rng, 1000, 16032), rng.randint(0, 24), rng.randint(0, 24), rng.randint(1, 12),
                    second + rng.randint(0, 24), second, rng.choice([0.7, 1.0]), rng.choice([0.7, 0.9]),
                    rng.choice(["f32", "bf16"]), 3.0)
    del c["name"]
    return c


def draw(rng):
    while True:
        c = _draw_once(rng)
        w = work(c)
        if w["bytes"] <= MOST_BYTES and w["flops"] <= MOST_FLOPS and not (c["kind"] == "kv" and _pool_bytes(c) > 4e9):
            return c


# ----------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _chain_logits(case, g, std):
    """Final logits [B, k+1, V] and the draft's, one readout earlier: the same
    plus noise at the first k positions."""
    b, k, v = case["batch"], case["k"], case["vocab"]
    target = torch.randn((b, k + 1, v), generator=g, device=DEVICE) * std
    draft = target[:, :k] + torch.randn((b, k, v), generator=g, device=DEVICE)
    dt = DTYPES[case["dtype"]]
    return target.to(dt), draft.to(dt)


def _nucleus(logits, temperature, top_p, top_k):
    """Filtered, renormalised probabilities in the logits' own precision: ties
    at the cutoff kept, top-p and top-k cutoffs joined, one renormalisation."""
    p = torch.softmax(logits / temperature, dim=-1)
    cut = torch.zeros(p.shape[:-1] + (1,), dtype=p.dtype, device=p.device)
    if top_p < 1.0:
        s = p.sort(dim=-1, descending=True).values
        n = (s.cumsum(-1) < top_p).sum(-1, keepdim=True).clamp_(max=p.shape[-1] - 1)
        cut = torch.maximum(cut, s.gather(-1, n))
    if 0 < top_k < p.shape[-1]:
        cut = torch.maximum(cut, p.topk(top_k, dim=-1).values[..., -1:])
    p = torch.where(p >= cut, p, torch.zeros_like(p))
    return p / p.sum(-1, keepdim=True)


def _inputs(case, seed):
    """The tensors of a case, from its seed."""
    g = _gen(seed)
    kind = case["kind"]
    s = {}
    if kind == "greedy":
        s["target"], s["draft"] = _chain_logits(case, g, 3.0)
        s["ids"] = None
        if case["ids"]:
            s["ids"] = s["draft"].float().argmax(-1)
            s["draft"] = None
    elif kind == "spec":
        b, k, v = case["batch"], case["k"], case["vocab"]
        s["target"], s["draft"] = _chain_logits(case, g, case["std"])
        s["uniforms"] = torch.rand((b, 2 * k + 1), generator=g, device=DEVICE)
        s["draft_uniforms"] = torch.rand(b * k, generator=g, device=DEVICE)
        s["history"] = s["history_len"] = None
        if case["penalty"] != 1.0:
            h = case["hist_max"]
            zipf = torch.arange(1, v + 1, device=DEVICE, dtype=torch.float32) ** -1.1
            s["history"] = torch.multinomial(zipf.expand(b, v), h, replacement=True, generator=g).to(torch.int32)
            s["history_len"] = torch.randint(h // 16, h + 1, (b,), generator=g, device=DEVICE, dtype=torch.int32)
        if not case["draft"]:
            q = _nucleus(s["draft"].float(), case["temperature"], case["top_p"], case["top_k"]).reshape(b * k, v)
            s["ids"] = torch.multinomial(q, 1, generator=g).reshape(b, k)
    elif kind == "filter":
        rows, v = case["rows"], case["vocab"]
        s["logits"] = (torch.randn((rows, v), generator=g, device=DEVICE) * case["std"]).to(DTYPES[case["dtype"]])
    elif kind == "head":
        rows, h, v = _head_rows(case), case["hidden"], case["vocab"]
        s["hidden"] = torch.randn((rows, h), generator=g, device=DEVICE).to(torch.bfloat16)
        s["weight"] = (torch.randn((v, h), generator=g, device=DEVICE) * h ** -0.5).to(torch.bfloat16)
        s["ids"] = torch.randint(0, v, (case["batch"], case["k"]), generator=g, device=DEVICE)
    elif kind == "kv":
        b, k, ps = case["batch"], case["k"], case["page_size"]
        ring, branch = _ring_pages(case), -(-b * k // ps)
        pages = b + ring + branch
        kv = torch.empty((case["planes"], pages * ps, case["token_bytes"] // 2), dtype=torch.bfloat16, device=DEVICE)
        s["kv"] = kv.normal_(generator=g)
        s["accept_len"] = torch.randint(0, k + 1, (b,), generator=g, device=DEVICE, dtype=torch.int32)
        ctx = torch.randint(512, 8193, (b,), generator=g, device=DEVICE)
        # room for the timed passes in every row's page table
        s["page_table"] = torch.zeros((b, (8192 + 40000 * k) // ps + 2), dtype=torch.int32, device=DEVICE)
        row = torch.arange(b, device=DEVICE)
        s["page_table"][row, -(-ctx // ps) - 1] = row.to(torch.int32)  # each row's last page
        s["ctx_len"] = ctx
        s["free_pages"] = b + torch.randperm(ring, generator=g, device=DEVICE)
        s["page_state"] = torch.tensor([0, 1 << 62], dtype=torch.int64, device=DEVICE)
        s["branch_slots"] = ((b + ring) * ps + torch.arange(b * k, device=DEVICE)).reshape(b, k)
    else:
        m, v = _policy_rows(case), case["vocab"]
        logits = torch.randn((m, v), generator=g, device=DEVICE) * case["std"]
        s["logits"] = logits.to(DTYPES[case["dtype"]])
        for name, noise in (("first", 1.0), ("second", 1.5)):
            noisy = logits + torch.randn((m, v), generator=g, device=DEVICE) * noise
            s[name] = _nucleus(noisy, case["temperature"], case["top_p"], 0)
            s[name + "_token"] = torch.multinomial(s[name], 1, generator=g).flatten()
    return s


def _head_rows(case):
    """Endpoint rows: the k + 1 target positions of each sequence, and for the
    argmax over a whole step the k draft positions too."""
    return case["batch"] * (2 * case["k"] + 1 if case["op"] == "argmax" else case["k"] + 1)


def _ring_pages(case):
    # enough that a page comes round again only after its row has left it
    return case["batch"] * (case["k"] + 1) + 64


def _pool_bytes(case):
    b, k, ps = case["batch"], case["k"], case["page_size"]
    return (b + _ring_pages(case) + -(-b * k // ps)) * ps * case["planes"] * case["token_bytes"]


def _policy_rows(case):
    return case["q1"] + case["q2"] + case["direct"] + case["verified"]


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "policy":
        m, v = _policy_rows(case), case["vocab"]
        n1, n2, nd = case["q1"], case["q2"], case["direct"]
        kinds = ["q1"] * n1 + ["q2"] * n2 + ["final"] * (nd + case["verified"])
        first, second = s["first_token"].tolist(), s["second_token"].tolist()
        lanes = []
        for r in range(m):
            lane = PipelineLane(stage=0, index=r, token=0)
            verified = r - (n1 + n2 + nd)
            if n1 <= r < n1 + n2 or verified >= 0:
                lane.first_token, lane.first_state = first[r], s["first"][r]
            if 0 <= verified < case["second"]:
                lane.second_token, lane.second_state = second[r], s["second"][r]
            lanes.append(lane)
        sampler = CategoricalSampler(m, v, DEVICE)
        options = {"temperature": case["temperature"], "top_k": 1 << 30, "top_p": case["top_p"]}
        s["policy"] = SamplingDecisionPolicy(m, DEVICE, options, sampler, generator=_gen(seed + 1))
        s["lanes"], s["endpoints"] = lanes, dict(enumerate(kinds))
        s["post"] = SimpleNamespace(next_token_logits=s["logits"])
    return s


# ----------------------------------------------------------------------------
# one pass
# ----------------------------------------------------------------------------


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "greedy":
        return verify.greedy_verify(s["target"], s["draft"], s["ids"])
    if kind == "spec":
        b, k, v = case["batch"], case["k"], case["vocab"]
        t, p, tk = case["temperature"], case["top_p"], case["top_k"]
        ids = (verify.sample_logits(s["draft"].view(b * k, v), s["draft_uniforms"], t, p, top_k=tk).view(b, k)
               if case["draft"] else s["ids"])
        accept_len, tokens = verify.speculative_verify(
            s["target"], s["draft"], ids, s["uniforms"], t, p, top_k=tk, penalty=case["penalty"],
            history=s["history"], history_len=s["history_len"])
        return accept_len, tokens, ids
    if kind == "filter":
        return verify.filter_logits(s["logits"], case["temperature"], case["top_p"], top_k=case["top_k"])
    if kind == "head":
        if case["op"] == "verify":
            return verify.lm_head_greedy_verify(s["hidden"], s["weight"], case["k"], s["ids"])
        if case["op"] == "argmax":
            return verify.lm_head_argmax(s["hidden"], s["weight"])
        return verify.lm_head_logits(s["hidden"], s["weight"], dtype=torch.bfloat16)
    if kind == "kv":
        dst = graph_ops.commit_kv(s["kv"], s["accept_len"], s["branch_slots"], s["page_table"], s["ctx_len"],
                                  s["free_pages"], s["page_state"], case["page_size"])
        return dst, s["kv"], s["page_table"], s["ctx_len"], s["page_state"]
    policy = s["policy"]
    batch = policy.queue(s["post"], s["endpoints"], s["lanes"])
    decisions = policy.read(s["lanes"], s["endpoints"], batch)
    return np.array(list(decisions.values())), list(batch.proposal_states.values())


# ----------------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind in ("greedy", "spec"):
        b, k, v = case["batch"], case["k"], case["vocab"]
        elem = 4 if case["dtype"] == "f32" else 2
        rows = b * (2 * k + 1) if not case.get("ids") else b * (k + 1)
        n = rows * v * elem + b * (4 + 8 * (k + 1) + 8 * k)
        if kind == "spec":
            n += b * (2 * k + 1) * 4 + b * int(case["hist_max"] * 0.53) * 4
        return {"bytes": n, "flops": 0}
    if kind == "filter":
        elem = 4 if case["dtype"] == "f32" else 2
        return {"bytes": case["rows"] * (case["vocab"] * (elem + 4) + 8), "flops": 0}
    if kind == "head":
        rows, h, v = _head_rows(case), case["hidden"], case["vocab"]
        out = rows * v * 2 if case["op"] == "logits" else rows * 8
        return {"bytes": (rows + v) * h * 2 + out, "flops": 2 * rows * h * v}
    if kind == "kv":
        tokens = case["batch"] * case["k"] / 2
        return {"bytes": int(2 * tokens * case["planes"] * case["token_bytes"]) + case["batch"] * (20 + 16 * case["k"]),
                "flops": 0}
    m, v = _policy_rows(case), case["vocab"]
    elem = 4 if case["dtype"] == "f32" else 2
    # logits in, the filtered rows and the residual rows out, the proposal rows in
    n = m * v * (elem + 4) + case["q2"] * v * 8 + (case["verified"] + case["second"]) * v * 4 + m * 40
    return {"bytes": n, "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind == "head":
        # float32 sums in another order move some bf16 logits by one step of
        # 2^-7 of their value: 1.1e-5 to 4.1e-5 measured against a GEMM library
        # and against the rounded 64-bit product, times four. Ids change only
        # where two float32 logits lie that close (none measured).
        return {"rel": 1.6e-4, "max": 1e-2} if case["op"] == "logits" else {"rel": 0.0, "differ": 0.004}
    # ids, lengths, slots and copies are whole values; the probabilities are
    # defined operation by operation, so they do not depend on the order either
    return "exact"


def exact(case, seed):
    """run()'s answer in 64 bits by plain torch, None where it has no such value."""
    kind = case["kind"]
    if kind == "greedy":
        s = _inputs(case, seed)
        return _accepted(s["target"].double().argmax(-1),
                         s["ids"] if s["ids"] is not None else s["draft"].double().argmax(-1))
    if kind == "filter":
        s = _inputs(case, seed)
        filtered = _nucleus(s["logits"].double(), case["temperature"], case["top_p"], case["top_k"])
        p = torch.softmax(s["logits"].double() / case["temperature"], dim=-1)
        kept = filtered > 0
        return {"cutoff": torch.where(kept, p, 1.0).amin(-1), "mass": (p * kept).sum(-1), "filtered": filtered}
    if kind == "head":
        s = _inputs(case, seed)
        h, w = s["hidden"].double(), s["weight"]
        logits = torch.empty((h.shape[0], w.shape[0]), dtype=torch.float64, device=DEVICE)
        for i in range(0, w.shape[0], 16384):
            logits[:, i:i + 16384] = h @ w[i:i + 16384].double().T
        if case["op"] == "logits":
            return logits
        ids = logits.argmax(-1)
        return ids if case["op"] == "argmax" else _accepted(ids.view(case["batch"], case["k"] + 1), s["ids"])
    # draws, copies and decisions
    return None


def _accepted(target, draft):
    k = draft.shape[1]
    accept_len = (target[:, :k] == draft).long().cumprod(1).sum(1)
    pos = torch.arange(k + 1, device=target.device)
    return accept_len.to(torch.int32), torch.where(pos <= accept_len[:, None], target, -1)
