"""Workloads of the decode-attention library, as a program that uses it runs
them, with their inputs, their least work and the outputs expected of them.

A case is one attention call of a decode step: `layout` (packed, bhsd or
paged), `batch` sequences, `hq` query and `hkv` KV heads of `head_dim` dims,
lengths up to `max_len` spread as `lengths` says, and for paged caches the
rows of a `page`.  `numerics` picks one of the tensor interface's options.

Lengths are the same set for every seed (in another order), so that a case
always moves the same bytes:
  full      every sequence has max_len rows: a static batch
  poisson   quantiles of Poisson(4) in [1, 16]: the lengths of the
            repository's variable-length benchmark table
  spread    quantiles of a log-uniform spread over [max_len / 32, max_len]:
            sequences of a continuous batch, at all stages of their lives
"""
import math

import torch

import fmha_amd

# (query heads, KV heads) of the repository's benchmarks and tests: multi-head
# attention, grouped queries, and the heads one GPU keeps of a model sharded
# by KV head.
HEADS = ((16, 16), (32, 32), (8, 8), (32, 16), (32, 8), (64, 8), (40, 8), (28, 4), (16, 2), (8, 1), (4, 1), (32, 1))


def _case(layout, batch, hq, hkv, head_dim, max_len, lengths, page=0, numerics="default"):
    return {"layout": layout, "batch": batch, "hq": hq, "hkv": hkv, "head_dim": head_dim, "max_len": max_len,
            "lengths": lengths, "page": page, "numerics": numerics}


def listed():
    cases = {
        # The smallest row of the variable-length table: launch latency.
        "small_varlen": _case("packed", 10, 16, 16, 128, 16, "poisson"),
        # The headline batch: 30720 sequences of 16 rows, 4.3 GB.
        "short_uniform": _case("packed", 30720, 16, 16, 128, 16, "full"),
        # Two query heads per KV head on an odd length.
        "short_gqa": _case("packed", 20000, 32, 16, 128, 11, "full"),
        # The largest row of the variable-length table, 5.6 GB.
        "short_varlen_d256": _case("packed", 30720, 32, 32, 256, 16, "poisson"),
        # Many short conversations just past the short kernels' 16 rows.
        "many_short_rows": _case("packed", 3000, 32, 8, 128, 100, "spread"),
        # A full static batch of medium contexts.
        "batch_1k": _case("packed", 256, 64, 8, 128, 1024, "full"),
        # Continuous batching on 16-row pages: every stage of a 4k window.
        "serving_paged": _case("paged", 64, 32, 8, 128, 4096, "spread", page=16),
        # The same on one GPU of a model sharded over its 8 KV heads.
        "serving_paged_sharded": _case("paged", 48, 8, 1, 128, 8000, "spread", page=16),
        # A single user: one sequence, nothing to batch.
        "single_user": _case("paged", 1, 32, 8, 128, 3001, "full", page=16),
        # A small static multi-head batch in a padded [B, H, S, D] cache.
        "static_bhsd": _case("bhsd", 8, 16, 16, 64, 1500, "spread"),
        # One very long document.
        "long_document": _case("packed", 1, 32, 8, 128, 131072, "full"),
        # A few long contexts with wide groups on pages.
        "long_batch_paged": _case("paged", 6, 64, 8, 128, 32768, "spread", page=16),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    hq, hkv = rng.choice(HEADS)
    head_dim = rng.choice((64, 128, 128, 256))
    if rng.random() < 0.35:
        max_len = rng.randint(1, 16)
        lengths = "full" if rng.random() < 0.5 else "poisson"
        layout, page, numerics = "packed", 0, "default"
        if lengths == "poisson":
            max_len = 16
            layout = rng.choice(("packed", "packed", "paged"))
            page = rng.choice((16, 64)) if layout == "paged" else 0
            if layout == "packed" and hq <= 8 * hkv:
                numerics = rng.choice(("default", "default", "fast", "fp32_weights"))
        elif rng.random() < 0.3:
            layout = "bhsd"
        batch = _log_int(rng, 1, 30720)
    else:
        max_len = _log_int(rng, 17, 131072)
        lengths = rng.choice(("full", "spread", "spread"))
        layout = rng.choice(("packed", "bhsd", "paged", "paged"))
        page = rng.choice((16, 16, 64, 1)) if layout == "paged" else 0
        numerics = "default"
        batch = _log_int(rng, 1, 4096)
    row = 4 * hkv * head_dim
    # at most 1 GB of K and V
    batch = max(1, min(batch, int(1e9 / (max_len * row))))
    max_len = min(max_len, int(1e9 / row))
    return _case(layout, batch, hq, hkv, head_dim, max_len, lengths, page, numerics)


def _lengths(case):
    n, m = case["batch"], case["max_len"]
    if case["lengths"] == "full":
        return [m] * n
    if case["lengths"] == "poisson":
        out, k, term = [], 0, math.exp(-4.0)
        below = term
        for i in range(n):
            while (i + 0.5) / n > below and k < m:
                k += 1
                term *= 4.0 / k
                below += term
            out.append(min(max(k, 1), m))
        return out
    # The longest sequence has all max_len rows.
    return [max(1, int(round(m * 32.0 ** (i / max(n - 1, 1) - 1.0)))) for i in range(n - 1)] + [m]


def _workspace(case, device):
    n = fmha_amd.splitkv_workspace_size(case["batch"], case["hq"], case["hkv"], case["max_len"], case["head_dim"])
    return torch.empty(max(n, 1), dtype=torch.uint8, device=device)


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    cpu = torch.Generator().manual_seed(seed)
    n, hkv, d, m = case["batch"], case["hkv"], case["head_dim"], case["max_len"]

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=torch.bfloat16)

    lens = torch.tensor(_lengths(case), dtype=torch.int32)[torch.randperm(n, generator=cpu)]
    state = {"case": case, "q": normal(n, case["hq"], d), "lens": lens.to(dev)}
    if m > 16:
        state["workspace"] = _workspace(case, dev)
    if case["layout"] == "packed":
        rows = int(lens.sum())
        shape = (n, m, hkv, d) if case["lengths"] == "full" and m <= 16 else (rows, hkv, d)
        state["k"], state["v"] = normal(*shape), normal(*shape)
        state["cu"] = torch.cat((torch.zeros(1, dtype=torch.int64), lens.cumsum(0))).to(torch.int32).to(dev)
    elif case["layout"] == "bhsd":
        # [B, H, S, D] in memory, handed over as the [B, S, H, D] view of it
        state["k"], state["v"] = (normal(n, hkv, m, d).transpose(1, 2) for _ in range(2))
    else:
        page = case["page"]
        used = (lens.long() + page - 1) // page
        order = torch.randperm(int(used.sum()), generator=cpu).to(torch.int32)
        table = torch.zeros(n, (m + page - 1) // page, dtype=torch.int32)
        table[torch.arange(table.shape[1])[None, :] < used[:, None]] = order
        state["table"] = table.to(dev)
        state["k"], state["v"] = (normal(order.numel(), page, hkv, d) for _ in range(2))
    return state


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    if case["layout"] == "paged":
        if case["max_len"] <= 16:
            return fmha_amd.fmha_decode_paged(q, k, v, state["table"], state["lens"])
        return fmha_amd.fmha_decode_paged(q, k, v, state["table"], state["lens"], max_seqlen_kv=case["max_len"],
                                          workspace=state["workspace"])
    if case["layout"] == "bhsd":
        return fmha_amd.fmha_decode_strided(q, k, v, state["lens"], workspace=state.get("workspace"))
    if case["max_len"] > 16:
        return fmha_amd.fmha_decode_splitkv(q, k, v, state["cu"], case["max_len"], workspace=state["workspace"])
    if k.dim() == 4:
        return fmha_amd.fmha_decode(q, k, v)
    return fmha_amd.fmha_decode(q, k, v, cu_seqlens_kv=state["cu"], fast=case["numerics"] == "fast",
                                fp32_weights=case["numerics"] == "fp32_weights")


def work(case):
    """Q, K and V read once, O written once; two products per row and head."""
    rows = sum(_lengths(case))
    return {"bytes": 4 * case["head_dim"] * (case["batch"] * case["hq"] + rows * case["hkv"]),
            "flops": 4 * case["head_dim"] * rows * case["hq"]}


def tolerance(case):
    # Weights are rounded to 8 significant bits and outputs to fp16: against
    # 64 bits the listed cases are 1.4e-3 to 1.7e-3 off (fp16 outputs alone:
    # 2e-4).  A weight next to a rounding midpoint may go either way,
    # which moves an output by 2^-8 of a weight times a value.
    return {"rel": 6e-3, "max": 6e-2}


def exact(case, seed):
    s = prepare(case, seed)
    n, hq, hkv, d = case["batch"], case["hq"], case["hkv"], case["head_dim"]
    q = s["q"].view(n, hkv, hq // hkv, d)
    lens = s["lens"].long()
    order = torch.argsort(lens)  # batches of like lengths together: little padding
    sizes = lens[order].tolist()
    out = torch.empty(n, hkv, hq // hkv, d, dtype=torch.float64, device=q.device)
    first = 0
    while first < n:
        last = first + 1
        while last < n and (last + 1 - first) * sizes[last] * hkv * d <= 1 << 26:
            last += 1
        b = order[first:last]
        j = torch.arange(sizes[last - 1], device=q.device)
        there = j[None, :] < lens[b][:, None]

        def rows(x):
            if case["layout"] == "paged":
                at = s["table"].long()[b][:, j // case["page"]] * case["page"] + j % case["page"]
                x = x.view(-1, hkv, d)[torch.where(there, at, 0)]
            elif x.dim() == 4:
                x = x[b][:, :j.numel()]
            else:
                x = x[torch.where(there, s["cu"].long()[b][:, None] + j, 0)]
            return x.double().transpose(1, 2).contiguous()

        t = torch.matmul(q[b].double(), rows(s["k"]).transpose(2, 3).contiguous()) / math.sqrt(d)
        t.masked_fill_(~there[:, None, None, :], -math.inf)
        out[b] = torch.matmul(torch.softmax(t, -1), rows(s["v"]))
        first = last
    return out.view(n, hq, d)
