"""Performance cases: decode attention as a serving engine calls it, one call
per layer and step, through the package's Python operators.

Two paths, both single-step decode over a paged bf16 cache:

  gqa   binding.gqa_decode_v2 (num_splits=0 is the automatic choice, 8 the
        operator's default) and binding.gqa_decode_v1, head dim 128;
  mla   mla.flash_mla_with_kvcache over the 576-dim latent cache. Its plan
        (get_mla_metadata) is made once per decode step and serves every
        layer of the model, so it belongs to the prepared state.

Request lengths follow from the case alone ("lens": every request the same
length, U[1, S], or FlashMLA's N(S, S/2)); the seed decides which request gets
which length, the tensors' values and the order of the physical blocks.
"""

import math
import os
import random
import sys

import torch

for _p in (os.path.join(os.getcwd(), "mla-decode-kernels_amd", "python"),):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import binding  # noqa: E402
import mla  # noqa: E402

DEVICE = "cuda"
D = 128              # GQA head dim
MLA_D, MLA_DV = 576, 512


def _gqa(name, B, S, Hq, Hkv, bs, lens="uniform", op="v2", num_splits=0):
    return {"name": name, "path": "gqa", "op": op, "B": B, "S": S, "lens": lens, "Hq": Hq,
            "Hkv": Hkv, "block": bs, "num_splits": num_splits}


def _mla(name, B, S, h_q, bs=64, lens="varlen", s_q=1, causal=False, fixed_plan=False):
    return {"name": name, "path": "mla", "B": B, "S": S, "lens": lens, "h_q": h_q, "s_q": s_q,
            "causal": causal, "block": bs, "fixed_plan": fixed_plan}


def listed():
    return [
        # One user, a short prompt: the smallest call, where latency counts.
        _gqa("gqa_b1_s512", 1, 512, 32, 8, 16),
        # One user deep into a long document.
        _gqa("gqa_b1_s32768_h64", 1, 32768, 64, 8, 64),
        # A handful of users at mixed lengths, the operator's default split count.
        _gqa("gqa_b8_ragged_default", 8, 4096, 64, 8, 16, lens="ragged", num_splits=8),
        # A large batch of short chats of an odd length, single-pass operator.
        _gqa("gqa_b128_s777_v1", 128, 777, 32, 8, 16, op="v1"),
        # The representative batch: 32 requests of 8192 tokens (1 GiB of KV).
        _gqa("gqa_b32_s8192", 32, 8192, 32, 8, 16),
        # Wide groups and long contexts (4 GiB of KV).
        _gqa("gqa_b32_s32768_h64", 32, 32768, 64, 8, 64),
        # Continuous batching at its fullest: 128 requests, U[1, 32768].
        _gqa("gqa_b128_ragged", 128, 32768, 32, 8, 16, lens="ragged"),
        # MLA, one user: all 128 heads of one request on one GPU.
        _mla("mla_b1_s4096", 1, 4096, 128, lens="uniform"),
        # One rank of a tensor-parallel group: 16 of the 128 heads, full batch.
        _mla("mla_b128_h16_s4096", 128, 4096, 16),
        # Half the heads, long contexts.
        _mla("mla_b32_h64_s16384", 32, 16384, 64),
        # The benchmark row: 128 heads, 128 requests around 4096 tokens.
        _mla("mla_b128_s4096", 128, 4096, 128),
        # The same with two query tokens per request (speculative decoding).
        _mla("mla_b128_s4096_sq2", 128, 4096, 128, s_q=2, causal=True),
    ]


# Drawn cases stay under the largest listed ones.
_MOST_BYTES, _MOST_FLOPS = 5.0e9, 2.5e11


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        B, S = _log_int(rng, 1, 128), _log_int(rng, 200, 32768)
        lens = rng.choice(["uniform", "ragged", "varlen"])
        if rng.random() < 0.5:
            Hq, Hkv = rng.choice([(32, 8), (64, 8), (32, 8), (64, 8), (16, 8), (40, 8), (8, 8),
                                  (128, 8), (16, 4), (64, 16)])
            # The single-pass operator is for batches that fill the device.
            op, ns = rng.choice([("v2", 0), ("v2", 0), ("v2", 8), ("v1", 0)])
            if op == "v1" and B * Hkv < 256:
                op = "v2"
            case = _gqa("", B, S, Hq, Hkv, rng.choice([16, 64, 32]), lens, op, ns)
        else:
            s_q = rng.choice([1, 1, 2, 4])
            case = _mla("", B, S, rng.choice([16, 32, 64, 128]), rng.choice([64, 64, 32, 16]),
                        lens, s_q, s_q > 1 and rng.random() < 0.7, rng.random() < 0.25)
        del case["name"]
        w = work(case)
        if w["bytes"] <= _MOST_BYTES and w["flops"] <= _MOST_FLOPS:
            return case


def _lengths(case):
    """The batch's request lengths: the same numbers for every seed."""
    B, S, r = case["B"], case["S"], random.Random(case["B"] * 1000003 + case["S"])
    if case["lens"] == "uniform":
        return [S] * B
    if case["lens"] == "ragged":
        return [r.randint(1, S) for _ in range(B)]
    return [max(int(r.gauss(S, S / 2)), case.get("s_q", 1)) for _ in range(B)]


def work(case):
    lens, B = _lengths(case), case["B"]
    total = float(sum(lens))
    index = 4.0 * (B + sum((n + case["block"] - 1) // case["block"] for n in lens))
    if case["path"] == "gqa":
        return {"bytes": total * case["Hkv"] * D * 4 + 2.0 * B * case["Hq"] * D * 2 + index,
                "flops": 4.0 * case["Hq"] * D * total}
    rows = case["s_q"] * case["h_q"]
    return {"bytes": total * MLA_D * 2 + B * rows * ((MLA_D + MLA_DV) * 2.0 + 4.0) + index,
            "flops": 2.0 * rows * total * (MLA_D + MLA_DV)}


def _inputs(case, seed):
    """(q, caches, block_table, seq_lens): N(0, 1) bf16, a pool of 1.25 times
    the blocks in use, handed out in a shuffled order; -1 past each request."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    cpu = torch.Generator().manual_seed(seed)
    lens, bs, B = _lengths(case), case["block"], case["B"]
    lens = [lens[i] for i in torch.randperm(B, generator=cpu).tolist()]
    blocks = [(n + bs - 1) // bs for n in lens]
    pool = sum(blocks) + (sum(blocks) + 3) // 4

    def normal(*shape):
        return torch.empty(*shape, dtype=torch.bfloat16, device=DEVICE).normal_(generator=gen)

    if case["path"] == "gqa":
        q = normal(B, case["Hq"], D)
        caches = [normal(pool, bs, case["Hkv"], D) for _ in range(2)]
    else:
        q = normal(B, case["s_q"], case["h_q"], MLA_D)
        caches = [normal(pool, bs, 1, MLA_D)]
    ids = torch.randperm(pool, generator=cpu).to(torch.int32)
    table = torch.full((B, max(blocks)), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(blocks):
        table[b, :n] = ids[at:at + n]
        at += n
    return (q, caches, table.to(DEVICE), torch.tensor(lens, dtype=torch.int32, device=DEVICE))


def prepare(case, seed):
    q, caches, table, lens = _inputs(case, seed)
    if case["path"] == "gqa":
        args = (q, *caches, table, lens, D ** -0.5)
        if case["op"] == "v1":
            return {"fn": binding.gqa_decode_v1, "args": args}
        return {"fn": binding.gqa_decode_v2, "args": args + (case["num_splits"],)}
    rows = case["s_q"] * case["h_q"]
    # The fixed plan wants the longest request, which an engine knows on its
    # host: it wrote the block table there.
    plan = (mla.get_mla_metadata(lens, rows, 1, max(_lengths(case)), case["block"], 0)
            if case["fixed_plan"] else mla.get_mla_metadata(lens, rows, 1))
    return {"fn": mla.flash_mla_with_kvcache,
            "args": (q, caches[0], table, lens, MLA_DV, *plan, MLA_D ** -0.5, case["causal"])}


def run(state):
    return state["fn"](*state["args"])


def tolerance(case):
    """bf16 outputs of fp32 sums; MLA's softmax weights are bf16 as well."""
    return {"rel": 6e-3} if case["path"] == "gqa" else {"rel": 1e-2}


def exact(case, seed):
    """The same attention in float64, request by request, in plain torch."""
    q, caches, table, lens = _inputs(case, seed)
    bs, f64, outs, lses = case["block"], torch.float64, [], []

    def rows_of(cache, b, n):
        ids = table[b, :(n + bs - 1) // bs].long()
        return cache.index_select(0, ids).flatten(0, 1)[:n]  # [n, heads, dims]

    for b, n in enumerate(lens.tolist()):
        if case["path"] == "gqa":
            k, v = (rows_of(c, b, n).transpose(0, 1).to(f64).contiguous() for c in caches)
            qb = q[b].to(f64).view(case["Hkv"], -1, D)
            kt = k.transpose(1, 2).contiguous()
            p = torch.softmax(torch.matmul(qb, kt) * D ** -0.5, dim=-1)
            outs.append(torch.matmul(p, v).reshape(case["Hq"], D))
            continue
        c = rows_of(caches[0], b, n)[:, 0].to(f64)
        s = torch.matmul(q[b].to(f64).flatten(0, 1), c.t().contiguous()) * MLA_D ** -0.5
        s = s.view(case["s_q"], case["h_q"], n)
        if case["causal"]:
            for i in range(case["s_q"]):
                s[i, :, max(0, n - (case["s_q"] - 1 - i)):] = -math.inf
        lse = torch.logsumexp(s, dim=-1)                         # [s_q, h_q]
        p = torch.exp(s - lse.unsqueeze(-1)).nan_to_num(0.0)
        outs.append(torch.matmul(p.flatten(0, 1), c[:, :MLA_DV].contiguous()).view(
            case["s_q"], case["h_q"], MLA_DV))
        lses.append(lse.t())
    return torch.stack(outs) if case["path"] == "gqa" else (torch.stack(outs), torch.stack(lses))
