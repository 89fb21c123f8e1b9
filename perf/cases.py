"""Performance cases of the fused-operator compute core.

Each case is one pass of work that a program using this package has it do,
through the package's public entry points: plain GEMMs, the flag-gated
AllGather+GEMM, GEMM+ReduceScatter, GEMM+AllReduce (both forms), the routed
MoE layer from device top-k, and the token dispatch + grouped GEMM of the
reference-named module.  Sizes are the workloads this repository's benchmark
and baseline tables name (and their smaller and larger neighbours), at one
GPU's share of the work.

Inputs are drawn on the GPU from the seed alone.  ``exact`` gives what ``run``
returns in 64 bits from plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from mkernel_amd import load_module, ops

DEV = "cuda"
BLOCK = 128                 # rows per ready flag and per expert padding block
BF16 = torch.bfloat16
# the MoE layer of the baseline tables: hidden, expert width, experts, top-k
H, INTER, EXPERTS, TOPK, ZIPF = 7168, 2048, 256, 8, 1.1


# ------------------------------------------------------------------- cases
def listed():
    return [
        # a projection of a small decode batch: one launch, latency-bound
        _gemm("gemm_small", 128, 2048, 2048),
        # the square GEMM of the baseline tables
        _gemm("gemm_4096", 4096, 4096, 4096),
        # a mid-sized projection whose tiles fill neither the row grid nor the K stages evenly
        _gemm("gemm_ragged", 1920, 2816, 5600),
        # AllGather+GEMM: one TP=8 rank, every shard staged inside the launch (the headline workload)
        _ag("ag_large", 8, 16384, 3584, 8192, own=False),
        # the smallest point of the AllGather+GEMM size sweep (K = M, N = M/16), own shard already in place
        _ag("ag_small", 16, 4096, 256, 4096, own=True),
        # GEMM+ReduceScatter: one TP=8 rank, partials arriving in random block order
        _rs("rs_large", 8, 0, 16384, 8192, 3584, "random"),
        # a small point of the GEMM+ReduceScatter sweep (K = M/16, N = M), arriving row block by row block
        _rs("rs_small", 16, 5, 4096, 4096, 256, "rows"),
        # two-shot GEMM+AllReduce of a down-projection at half the rows
        _ar("ar_two_shot", 8, 0, 8192, 8192, 3584, True),
        # decode: a small batch of tokens through the routed expert layer, bf16 out
        _moe("moe_decode", 64, 8, "bf16"),
        # the expert layer of the baseline tables, from device top-k, fp32 out
        _moe("moe_layer", 4096, 8, "f32"),
        # prefill: a long batch of tokens through the same layer
        _moe("moe_prefill", 16384, 8, "bf16"),
        # token dispatch + grouped GEMM through the reference-named module, tables built by the caller
        _dispatch("dispatch_gemm", 1000, 8),
    ]


def _gemm(name, M, N, K):
    return {"name": name, "op": "gemm", "M": M, "N": N, "K": K}


def _ag(name, world, M, N, K, own):
    return {"name": name, "op": "ag", "world": world, "M": M, "N": N, "K": K, "own": own}


def _rs(name, world, rank, M, N, K, order):
    return {"name": name, "op": "rs", "world": world, "rank": rank, "M": M, "N": N, "K": K, "order": order}


def _ar(name, world, rank, M, N, K, two_shot):
    return {"name": name, "op": "ar", "world": world, "rank": rank, "M": M, "N": N, "K": K, "two_shot": two_shot}


def _moe(name, tokens, ep, out):
    return {"name": name, "op": "moe", "tokens": tokens, "ep": ep, "out": out}


def _dispatch(name, tokens, ep):
    return {"name": name, "op": "dispatch", "tokens": tokens, "ep": ep}


def draw(rng):
    """One more case of the same ranges."""
    def spread(lo, hi, step):
        return step * max(1, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step))

    op = rng.choice(["gemm", "gemm", "ag", "rs", "ar", "moe", "moe", "dispatch"])
    if op == "gemm":
        c = _gemm("", spread(128, 8192, 128), spread(256, 8192, 256), spread(256, 8192, 32))
    elif op == "ag":
        world = rng.choice([2, 4, 8, 16])
        c = _ag("", world, spread(4096, 16384, 256 * world), spread(256, 3584, 256), spread(1024, 8192, 32),
                rng.random() < 0.5)
    elif op == "rs":
        world = rng.choice([2, 4, 8, 16])
        c = _rs("", world, rng.randrange(world), spread(2048, 16384, 256 * world), spread(2048, 8192, 256),
                spread(128, 3584, 32), rng.choice(["random", "rows"]))
    elif op == "ar":
        world = rng.choice([2, 4, 8])
        two = rng.random() < 0.5
        c = _ar("", world, rng.randrange(world), spread(2048, 8192 if two else 4096, 256 * world),
                spread(1024, 8192, 256), spread(256, 3584, 32), two)
    elif op == "moe":
        c = _moe("", spread(8, 16384, 1), rng.choice([8, 16]), rng.choice(["f32", "bf16"]))
    else:
        c = _dispatch("", spread(64, 8192, 1), rng.choice([8, 16]))
    del c["name"]
    return c


# ------------------------------------------------------------------- inputs
def _generator(seed, part):
    return torch.Generator(device=DEV).manual_seed(1000003 * int(seed) + part)


def _randn(shape, seed, part, scale):
    """bf16 N(0, scale^2), drawn in slices so that no large fp32 copy is held."""
    out = torch.empty(shape, dtype=BF16, device=DEV)
    g = _generator(seed, part)
    for piece in out.view(-1).split(1 << 27):
        piece.copy_(torch.randn(piece.numel(), generator=g, device=DEV).mul_(scale))
    return out


def _order(n, seed, part):
    return torch.randperm(n, generator=_generator(seed, part), device=DEV).to(torch.int32)


def _words(n):
    return torch.zeros(n, dtype=torch.int32, device=DEV)


def _matrices(c, seed):
    """A [M, K] and B [K, N] scaled as activations and weights of a trained projection."""
    s = c["K"] ** -0.5
    return _randn((c["M"], c["K"]), seed, 1, s), _randn((c["K"], c["N"]), seed, 2, s)


def _popularity():
    """Expert popularity of the router: Zipf ranks dealt to the experts once (a property of the model)."""
    ranks = np.random.default_rng(6).permutation(EXPERTS) + 1.0
    w = ranks ** -ZIPF
    return w / w.sum()


def _routing(tokens, seed):
    """The router's output on the device: ids int32 and softmax gates float32 [tokens, TOPK]."""
    logp = torch.from_numpy(np.log(_popularity())).to(DEV, torch.float32)
    u = torch.rand((tokens, EXPERTS), generator=_generator(seed, 3), device=DEV).clamp_(1e-7, 1 - 1e-6)
    top, ids = torch.topk(logp - torch.log(-torch.log(u)), TOPK, dim=1)
    return ids.to(torch.int32).contiguous(), torch.softmax(top, dim=1).contiguous()


def _capacity(c):
    """Padded rows of the worst routing of the batch."""
    return (c["tokens"] * TOPK + EXPERTS // c["ep"] * (BLOCK - 1) + BLOCK - 1) // BLOCK * BLOCK


def _expected(c):
    """(routed rows, local experts that get a row) to expect of a batch: an
    expert is among a token's top-k with probability 1 - exp(-x p_e)."""
    p = _popularity()
    lo, hi = 0.0, 1e6
    for _ in range(200):
        x = 0.5 * (lo + hi)
        lo, hi = (x, hi) if (1 - np.exp(-x * p)).sum() < TOPK else (lo, x)
    hit = (1 - np.exp(-x * p))[: EXPERTS // c["ep"]]
    T = c["tokens"]
    return max(1.0, float(T * hit.sum())), max(1.0, float((1 - (1 - hit) ** T).sum()))


def _peer_blocks(c):
    """128-row blocks of one rank's slice."""
    return c["M"] // c["world"] // BLOCK


def _peers(c, seed):
    rows = c["M"] // c["world"] if c["op"] == "rs" or c["two_shot"] else c["M"]
    return _randn((c["world"] - 1, rows, c["N"]), seed, 4, 0.5)


def _reduced(c, seed):
    """The other slices as their owners reduced them, [world-1, M/world, N]."""
    return _randn((c["world"] - 1, c["M"] // c["world"], c["N"]), seed, 5, 1.5)


def prepare(case, seed):
    c = dict(case)
    s = {"case": c}
    op = c["op"]
    if op in ("gemm", "ag", "rs", "ar"):
        s["A"], s["B"] = _matrices(c, seed)
    if op == "gemm":
        s["C"] = torch.empty((c["M"], c["N"]), dtype=BF16, device=DEV)
    elif op == "ag":
        n = c["M"] // BLOCK
        s["epoch"], s["flags"], s["counters"] = 0, _words(n), _words(n)
        s["A_full"] = torch.zeros_like(s["A"])
        s["C"] = torch.empty((c["M"], c["N"]), dtype=BF16, device=DEV)
        order = _order(n, seed, 6)
        s["present"] = 0
        if c["own"]:  # rank 0's own shard is in place; its blocks come first in the order
            s["present"] = n // c["world"]
            s["A_full"][: s["present"] * BLOCK] = s["A"][: s["present"] * BLOCK]
            order = torch.cat([torch.arange(s["present"], dtype=torch.int32, device=DEV),
                               order[order >= s["present"]]])
        s["order"] = order
    elif op == "rs":
        n = (c["world"] - 1) * _peer_blocks(c)
        s["epoch"], s["flags"], s["counters"] = 0, _words(n), _words(n)
        s["peers"] = _peers(c, seed)
        s["recv"] = torch.zeros_like(s["peers"])
        s["sends"] = torch.zeros((c["M"], c["N"]), dtype=BF16, device=DEV)
        s["out"] = torch.empty((c["M"] // c["world"], c["N"]), dtype=BF16, device=DEV)
        s["order"] = (_order(n, seed, 6) if c["order"] == "random"
                      else torch.arange(n, dtype=torch.int32, device=DEV)
                      .view(c["world"] - 1, -1).t().contiguous().view(-1))
    elif op == "ar":
        s["peers"] = _peers(c, seed)
        s["recv"] = torch.zeros_like(s["peers"])
        s["C"] = torch.empty((c["M"], c["N"]), dtype=BF16, device=DEV)
        s["done"] = _words((c["M"] // 256) * (c["N"] // 256))
        if c["two_shot"]:
            n = (c["world"] - 1) * _peer_blocks(c)
            s["reduced"] = _reduced(c, seed)
            s["sends"] = torch.zeros((c["M"], c["N"]), dtype=BF16, device=DEV)
            # the partials of the own slice row block by row block, then the reduced slices
            first = torch.arange(n, dtype=torch.int32, device=DEV).view(c["world"] - 1, -1).t().contiguous().view(-1)
            s["order"] = torch.cat([first, torch.arange(n, 2 * n, dtype=torch.int32, device=DEV)])
            n *= 2
        else:
            n = (c["world"] - 1) * (c["M"] // BLOCK)
            s["order"] = _order(n, seed, 6)
        s["epoch"], s["flags"], s["counters"] = 0, _words(n), _words(n)
    elif op == "moe":
        T, n_local = c["tokens"], EXPERTS // c["ep"]
        s["tokens"] = _randn((T, H), seed, 1, 1.0)
        s["ids"], s["gates"] = _routing(T, seed)
        s["w1"] = _randn((n_local, H, 2 * INTER), seed, 7, H ** -0.5)
        s["w2"] = _randn((n_local, INTER, H), seed, 8, INTER ** -0.5)
        s["act"] = torch.empty((_capacity(c), INTER), dtype=BF16, device=DEV)
        s["ye"] = torch.empty((_capacity(c), H), dtype=BF16, device=DEV)
        s["y"] = torch.empty((T, H), dtype=torch.float32 if c["out"] == "f32" else BF16, device=DEV)
    elif op == "dispatch":
        T, n_local = c["tokens"], EXPERTS // c["ep"]
        s["tokens"] = _randn((T, H), seed, 1, 1.0)
        s["w1"] = _randn((n_local, H, 2 * INTER), seed, 7, H ** -0.5)
        s["module"] = load_module.load("dispatch_gemm")
        ids, gates = _routing(T, seed)
        t = ops.moe_build_indices_dev(ids, gates, 0, n_local)
        s["pull"], s["padded"], s["local_rb"] = (t["pull_indices"], t["padded_tokens_per_expert"],
                                                 t["local_rb_per_expert"])
        s["rows"] = t["R_pad"]
        # rows past this routing's padded row count stay zero
        s["out"] = torch.zeros((_capacity(c), 2 * INTER), dtype=BF16, device=DEV)
    return s


# ------------------------------------------------------------------- one pass
def run(s):
    c = s["case"]
    op = c["op"]
    if op == "gemm":
        return {"C": ops.gemm(s["A"], s["B"], s["C"])}
    if op == "ag":
        s["epoch"] += 1
        ops.ag_gemm(s["A"], s["A_full"], s["B"], s["C"], s["flags"], s["order"], epoch=s["epoch"],
                    stage_counters=s["counters"], n_present=s["present"])
        return {"C": s["C"], "A_full": s["A_full"]}
    if op == "rs":
        s["epoch"] += 1
        ops.gemm_rs(s["A"], s["B"], s["sends"], s["out"], s["peers"], s["recv"], c["world"], c["rank"], s["flags"],
                    s["order"], epoch=s["epoch"], stage_counters=s["counters"])
        return {"out": s["out"], "sends": s["sends"], "recv": s["recv"]}
    if op == "ar":
        s["epoch"] += 1
        if c["two_shot"]:
            ops.gemm_ar_two_shot(s["A"], s["B"], s["C"], s["sends"], s["peers"], s["recv"], s["reduced"], c["world"],
                                 c["rank"], s["flags"], s["order"], epoch=s["epoch"], stage_counters=s["counters"],
                                 done_flags=s["done"])
            return {"C": s["C"], "sends": s["sends"], "recv": s["recv"]}
        ops.gemm_ar(s["A"], s["B"], s["C"], s["peers"], s["recv"], c["world"], s["flags"], s["order"],
                    epoch=s["epoch"], stage_counters=s["counters"], done_flags=s["done"])
        return {"C": s["C"], "recv": s["recv"]}
    if op == "moe":
        t = ops.moe_build_indices_dev(s["ids"], s["gates"], 0, EXPERTS // c["ep"], sync=False)
        ops.moe_ffn_combine(s["tokens"], t["pull_indices"], t["row_weight"], t["owner_offset"], t["slot_to_row"],
                            s["w1"], s["w2"], None, s["act"], s["ye"], s["y"], rb_expert=t["rb_expert"],
                            rb_rows=t["rb_rows"], fuse_dispatch=True, sizes=t["sizes"])
        return {"y": s["y"], "owner_offset": t["owner_offset"]}
    s["module"].moe_dispatch_gemm_fused(
        s["tokens"], None, None, None, s["w1"], s["out"], s["padded"], s["pull"], s["local_rb"], None, None, 0, 0, 0,
        0, 0, 0, 0, 1, 0, c["tokens"], s["rows"], 0, 0, 0, validate_tables=False)
    return {"out": s["out"]}


# ------------------------------------------------------------------- what it takes
def work(case):
    c = case
    if c["op"] in ("gemm", "ag", "rs", "ar"):
        M, N, K = c["M"], c["N"], c["K"]
        b = 2 * (M * K + K * N + M * N)
        if c["op"] == "ag":  # the staged rows are read as shards and written into the gathered matrix
            b += 2 * M * K * (c["world"] - 1) // c["world"] if c["own"] else 2 * M * K
        if c["op"] == "rs":  # the partials of the own slice: read, and written where they arrive
            b += 2 * 2 * (c["world"] - 1) * (M // c["world"]) * N
        if c["op"] == "ar" and c["two_shot"]:  # the same, and the other slices read; their partials are sent
            b += 2 * (2 + 1 + 1) * (c["world"] - 1) * (M // c["world"]) * N
        elif c["op"] == "ar":
            b += 2 * 2 * (c["world"] - 1) * M * N
        return {"bytes": b, "flops": 2 * M * N * K}
    rows, used = _expected(c)
    T = c["tokens"]
    read = min(T, rows) * H * 2
    if c["op"] == "dispatch":
        return {"bytes": read + used * H * 2 * INTER * 2 + rows * 2 * INTER * 2, "flops": 4 * rows * H * INTER}
    out = T * H * (4 if c["out"] == "f32" else 2)
    return {"bytes": read + used * 3 * H * INTER * 2 + T * TOPK * 8 + out, "flops": 6 * rows * H * INTER}


def tolerance(case):
    # One bf16 rounding of an fp32 sum: 1.7e-3 (2-norm) and at most 2^-8 of
    # the value against 64 bits; four times that.  The expert layer rounds
    # its activation and its expert rows to bf16 as well: 2.4e-3 against 64
    # bits at fp32 out, 2.9e-3 at bf16 out, at most 0.04 of the value.
    if case["op"] == "moe":
        return {"rel": 1.2e-2, "max": 0.16}
    return {"rel": 7e-3, "max": 1.6e-2}


# ------------------------------------------------------------------- 64 bits
def exact(case, seed):
    c = case
    d = torch.float64
    if c["op"] in ("gemm", "ag", "rs", "ar"):
        A, B = _matrices(c, seed)
        C = A.to(d) @ B.to(d)
        if c["op"] == "gemm":
            return {"C": C}
        if c["op"] == "ag":
            return {"C": C, "A_full": A}
        peers = _peers(c, seed)
        if c["op"] == "ar" and not c["two_shot"]:
            for p in peers:
                C += p.to(d)
            return {"C": C, "recv": peers}
        rows = c["M"] // c["world"]
        lo, hi = c["rank"] * rows, (c["rank"] + 1) * rows
        own = C[lo:hi].clone()
        for p in peers:
            own += p.to(d)
        C[lo:hi] = 0  # the own rows are not sent
        if c["op"] == "rs":
            return {"out": own, "sends": C, "recv": peers}
        other = _reduced(c, seed).to(d)
        return {"C": torch.cat([*other[: c["rank"]], own, *other[c["rank"]:]]), "sends": C, "recv": peers}
    T, n_local = c["tokens"], EXPERTS // c["ep"]
    tokens = _randn((T, H), seed, 1, 1.0)
    ids, gates = _routing(T, seed)
    w1 = _randn((n_local, H, 2 * INTER), seed, 7, H ** -0.5)
    if c["op"] == "dispatch":
        out = torch.zeros((_capacity(c), 2 * INTER), dtype=d, device=DEV)
        row = 0
        for e in range(n_local):
            t = (ids == e).any(1).nonzero().view(-1)
            out[row:row + t.numel()] = tokens[t].to(d) @ w1[e].to(d)
            row += (t.numel() + BLOCK - 1) // BLOCK * BLOCK
        return {"out": out}
    w2 = _randn((n_local, INTER, H), seed, 8, INTER ** -0.5)
    y = torch.zeros((T, H), dtype=d, device=DEV)
    for e in range(n_local):
        t, k = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            h = tokens[t].to(d) @ w1[e].to(d)
            a = torch.nn.functional.silu(h[:, :INTER]) * h[:, INTER:]
            y.index_add_(0, t, (a @ w2[e].to(d)) * gates[t, k].to(d)[:, None])
    off = torch.zeros(T + 1, dtype=torch.int32, device=DEV)
    off[1:] = ((ids >= 0) & (ids < n_local)).sum(1).cumsum(0)
    return {"y": y, "owner_offset": off}
