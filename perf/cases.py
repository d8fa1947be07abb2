"""The work that a serving program has this package do, as cases that can be timed.

A program that serves a model with this package makes six kinds of calls.  Per layer of a prefill iteration it attends over
the new tokens ("prefill": one GPU holds all keys, maybe behind a context that is cached already; "ring": the sequence is
spread over instances and one KV chunk after the other passes by) and runs the token-wise steps around the attention
("prefill_layer").  Per layer of a decode iteration it attends over the token-indexed KV pool ("decode"; "elastic" where
the context of a request is spread over instances), and at small batches what counts is the whole chain of short calls of
a layer with the slot bookkeeping of the iteration ("decode_layer").

listed() holds ordinary points of these kinds, draw() gives others of the same ranges; lengths come from the case alone,
values and slot numbers from the seed.
"""
import math
import random

import torch

from loongserve_amd import (LongServeMemoryManager, LongServeReqManager, context_attention_fwd, copy_kv_index_to_req,
                            destindex_copy_kv, init_req_to_token_indexes, longserve_token_decode_attention_flash_decoding,
                            ops, prefill_attention_step, rotary_emb_write_kv, simulate)
from loongserve_amd.longserve_cuda_kernels import rms_norm, rotary_emb, silu_and_mul_inplace

DEV = "cuda:0"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
EPS = 1e-5
PAD = 2147483647  # unused entries of the request table


def listed():
    return [
        # one short prompt, MHA with 32 heads: the smallest prefill call, where launches and the host's part count
        dict(name="prefill_1x100", kind="prefill", seqs=1, shortest=100, longest=100, context=0, q_heads=32, kv_heads=32,
             head_dim=128, dtype="f16", result="in_place", kv_write=False, lens=1),
        # a prefill iteration of chat traffic: a batch of short prompts of any length, grouped-query heads
        dict(name="prefill_16_short", kind="prefill", seqs=16, shortest=40, longest=1024, context=0, q_heads=32, kv_heads=8,
             head_dim=128, dtype="f16", result="in_place", kv_write=False, lens=2),
        # one sequence of 2048 tokens as a partial (fp32 output and log-sum-exp) that can be merged with others
        dict(name="prefill_1x2048_partial", kind="prefill", seqs=1, shortest=2048, longest=2048, context=0, q_heads=32,
             kv_heads=32, head_dim=128, dtype="f16", result="partial", kv_write=False, lens=3),
        # a batch of long documents of mixed lengths in bfloat16, K/V rows written to the pool and registered in the pass
        dict(name="prefill_8_long_bf16", kind="prefill", seqs=8, shortest=512, longest=32768, context=0, q_heads=32,
             kv_heads=8, head_dim=128, dtype="bf16", result="in_place", kv_write=True, lens=4),
        # chunked prefill: the next 500 tokens of a request that has 65000 in its context, with the caller's workspace
        dict(name="prefill_chunk_500", kind="prefill", seqs=1, shortest=500, longest=500, context=65000, q_heads=32,
             kv_heads=8, head_dim=128, dtype="f16", result="in_place", kv_write=False, lens=5),
        # a model with heads of 64, a batch of mid-sized prompts
        dict(name="prefill_8_head64", kind="prefill", seqs=8, shortest=1000, longest=3000, context=0, q_heads=32, kv_heads=8,
             head_dim=64, dtype="f16", result="in_place", kv_write=False, lens=6),
        # a long sequence over a ring of instances: 16384 queries of one shard against the KV chunks of four
        dict(name="ring_4x16384", kind="ring", shard=16384, chunks=4, striped=False, q_heads=32, kv_heads=32, dtype="f16"),
        # one user's decode step: a single request, where latency counts
        dict(name="decode_1x2048", kind="decode", batch=1, shortest=2048, longest=2048, q_heads=32, kv_heads=8, dtype="f16",
             lens=7),
        # the decode step of a full batch of long requests, slots scattered over the pool
        dict(name="decode_64_long", kind="decode", batch=64, shortest=4096, longest=32768, q_heads=32, kv_heads=8,
             dtype="f16", lens=8),
        # one layer of a decode iteration of chat traffic with everything around the attention: slots allocated and freed,
        # registered, norms, rotary embedding, K/V write, activation
        dict(name="decode_layer_24", kind="decode_layer", batch=24, shortest=200, longest=4000, q_heads=32, kv_heads=8,
             fused_write=False, lens=9),
        # very long requests whose context is spread over four instances, MHA: partials of the peers merged by the master
        dict(name="elastic_4x131072", kind="elastic", batch=4, shortest=131072, longest=131072, instances=4, q_heads=32,
             kv_heads=32, dtype="f16", lens=10),
        # the token-wise steps of one layer of a large prefill iteration: norms, rotary embedding, K/V write, activation
        dict(name="prefill_layer_16384", kind="prefill_layer", seqs=4, shortest=4096, longest=4096, q_heads=32, kv_heads=32,
             fused_write=True, lens=11),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    heads = rng.choice([(32, 32), (32, 8), (32, 8), (64, 8), (8, 1)])
    kind = rng.choice(["prefill", "prefill", "prefill", "ring", "decode", "decode", "decode_layer", "elastic", "prefill_layer"])
    case = dict(kind=kind, q_heads=heads[0], kv_heads=heads[1], lens=rng.randrange(1 << 20))
    if kind == "prefill":
        sort = rng.choice(["short", "short", "long", "chunk", "head64"])
        case.update(head_dim=128, dtype=rng.choice(["f16", "f16", "bf16"]), result=rng.choice(["in_place", "in_place", "partial"]),
                    kv_write=False, context=0)
        if sort == "short":  # up to some 16k tokens in all
            longest = _log(rng, 50, 2048)
            case.update(seqs=_log(rng, 1, max(1, min(32, 16384 // longest))), shortest=max(1, longest // rng.choice([1, 4, 20])),
                        longest=longest)
        elif sort == "long":
            longest = _log(rng, 4096, 32768)
            case.update(seqs=_log(rng, 1, 6), shortest=max(1, longest // rng.choice([1, 8, 50])), longest=longest,
                        kv_write=rng.random() < 0.5)
        elif sort == "chunk":
            rows = _log(rng, 64, 1024)
            case.update(seqs=rng.choice([1, 1, 2]), shortest=rows, longest=rows, context=_log(rng, 8192, 100000))
        else:
            longest = _log(rng, 100, 4096)
            case.update(head_dim=64, seqs=_log(rng, 1, max(1, min(16, 24576 // longest))), shortest=max(1, longest // rng.choice([1, 3])),
                        longest=longest)
    elif kind == "ring":
        del case["lens"]
        case.update(shard=_log(rng, 1000, 12000), chunks=rng.choice([2, 3, 4]), striped=rng.random() < 0.5,
                    dtype=rng.choice(["f16", "bf16"]))
    elif kind == "decode":
        longest = _log(rng, 128, 65536)
        case.update(batch=_log(rng, 1, max(1, min(256, 1500000 // longest))), shortest=max(1, longest // rng.choice([1, 8, 64])),
                    longest=longest, dtype=rng.choice(["f16", "bf16"]))
    elif kind == "decode_layer":
        longest = _log(rng, 64, 8192)
        case.update(batch=_log(rng, 1, max(1, min(128, 200000 // longest))), shortest=max(2, longest // rng.choice([1, 8])),
                    longest=longest, fused_write=rng.random() < 0.5)
    elif kind == "elastic":
        longest = _log(rng, 4096, 131072)
        case.update(batch=_log(rng, 1, max(1, min(16, 524288 // longest))), shortest=max(64, longest // rng.choice([1, 4])),
                    longest=longest, instances=rng.choice([2, 3, 4]), dtype=rng.choice(["f16", "bf16"]))
    else:
        longest = _log(rng, 100, 8192)
        case.update(seqs=_log(rng, 1, max(1, min(32, 20000 // longest))), shortest=max(1, longest // rng.choice([1, 4])),
                    longest=longest, fused_write=rng.random() < 0.5)
    need = work(case)
    return case if need["flops"] < 1.4e13 and need["bytes"] < 8.5e9 else draw(rng)  # no dearer than the largest listed ones


def _lengths(case):
    """The lengths of the case's sequences, log-uniform between its bounds."""
    rng = random.Random(case["lens"])
    return [_log(rng, case["shortest"], case["longest"]) for _ in range(case.get("seqs") or case["batch"])]


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _starts(lengths):
    at, out = 0, []
    for n in lengths:
        out.append(at)
        at += n
    return out


def _inter(case):
    """Width of the feed-forward block beside these heads, in the proportion of 11008 to 4096."""
    return case["q_heads"] * 128 * 43 // 16


class _Inputs:
    """Seeded inputs: activations and cached rows are N(0, 1) * 0.5."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV).manual_seed(seed)

    def values(self, shape, dtype=torch.float16, scale=0.5):
        return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, scale, generator=self.gen)

    def permutation(self, n):
        return torch.randperm(n, generator=self.gen, device=DEV)

    def angles(self, positions, head_dim):
        """cos and sin of the rotary embedding at these positions."""
        inv = 1.0 / (10000.0 ** (torch.arange(0, head_dim, 2, device=DEV, dtype=torch.float32) / head_dim))
        a = positions.float()[:, None] * inv[None, :]
        return a.cos().half(), a.sin().half()


def _positions(lengths):
    return torch.cat([torch.arange(n, device=DEV) for n in lengths])


def _prepare_prefill(case, inp):
    lengths, dtype = _lengths(case), DTYPES[case["dtype"]]
    hq, hkv, d, ctx = case["q_heads"], case["kv_heads"], case["head_dim"], case["context"]
    kv_lengths = [n + ctx for n in lengths]
    tokens = sum(lengths)
    s = dict(q=inp.values((tokens, hq, d), dtype), kv=inp.values((sum(kv_lengths), 2 * hkv, d), dtype))
    s["k"], s["v"] = s["kv"][:, :hkv], s["kv"][:, hkv:]
    s["where"] = (_i32(_starts(lengths)), _i32(lengths), _i32([ctx] * len(lengths)), _i32(_starts(kv_lengths)), _i32(kv_lengths),
                  _i32([0] * len(lengths)), 1, max(lengths))
    s["tokens"], s["workspace"] = tokens, None
    if case["result"] == "in_place":
        s["o"] = torch.empty_like(s["q"])
        s["m"] = torch.empty((tokens, hq), dtype=torch.float32, device=DEV)
        s["l"] = torch.empty_like(s["m"])
        if ctx:  # scratch for the cuts of the keys, kept by the program
            cuts = ops.kv_split_count(len(lengths), hq, max(lengths), s["k"].shape[0], hkv)
            s["workspace"] = torch.empty((cuts * tokens * hq * (d + 1),), dtype=torch.float32, device=DEV)
    if case["kv_write"]:
        s["pool"] = torch.zeros((tokens * 3 // 2, 2 * hkv, d), dtype=dtype, device=DEV)
        s["slots"] = inp.permutation(s["pool"].shape[0])[:tokens].to(torch.int32)
        s["table"] = torch.full((len(lengths) + 2, max(lengths)), PAD, dtype=torch.int32, device=DEV)
        s["b_req_idx"] = _i32([len(lengths) + 1 - i for i in range(len(lengths))])
    return s


def _run_prefill(s, case):
    if case["result"] == "partial":
        out = list(prefill_attention_step(s["q"], s["k"], s["v"], *s["where"], total_q_len=s["tokens"]))
    else:
        # the state starts over in every layer; how a step is split between m and l is the kernel's own, o is what the layer uses
        s["m"].fill_(float("-inf"))
        s["l"].zero_()
        context_attention_fwd(s["q"], s["k"], s["v"], s["o"], *s["where"], s["m"], s["l"], total_q_len=s["tokens"],
                              workspace=s["workspace"])
        out = [s["o"]]
    if case["kv_write"]:
        destindex_copy_kv(s["kv"], s["slots"], s["pool"])
        init_req_to_token_indexes(s["table"], s["b_req_idx"], s["where"][1], s["slots"], s["where"][0], s["where"][7])
        out += [s["pool"], s["table"]]
    return out


def _prepare_ring(case, inp):
    dtype, n, hq, hkv, peers = DTYPES[case["dtype"]], case["shard"], case["q_heads"], case["kv_heads"], case["chunks"]
    last = peers - 1
    s = dict(q=inp.values((n, hq, 128), dtype), o=torch.empty((n, hq, 128), dtype=dtype, device=DEV),
             m=torch.empty((n, hq), dtype=torch.float32, device=DEV), l=torch.empty((n, hq), dtype=torch.float32, device=DEV))
    first = (lambda j: j) if case["striped"] else (lambda j: j * n)
    s["chunks"] = [simulate.KVChunk(inp.values((n, 2 * hkv, 128), dtype), _i32([0]), _i32([n]), _i32([first(j)]))
                   for j in [last] + list(range(last))]  # the local chunk is the first to be attended
    s["where"] = (_i32([0]), _i32([n]), _i32([first(last)]), peers if case["striped"] else 1, n, hkv)
    return s


def _run_ring(s, case):
    return [simulate.ring_prefill(s["q"], s["chunks"], *s["where"], s["o"], s["m"], s["l"])[0]]


def _table(lengths, slots):
    """A request table over these slots; requests stand in it in reverse order, with a gap."""
    rows = len(lengths) + 3
    table = torch.full((rows, max(lengths)), PAD, dtype=torch.int32, device=DEV)
    order = [rows - 1 - i for i in range(len(lengths))]
    for row, at, n in zip(order, _starts(lengths), lengths):
        table[row, :n] = slots[at:at + n]
    return table, _i32(order)


def _prepare_decode(case, inp):
    lengths, dtype = _lengths(case), DTYPES[case["dtype"]]
    hq, hkv, batch, longest = case["q_heads"], case["kv_heads"], case["batch"], max(lengths)
    slots = max(65536, 2 * sum(lengths))
    s = dict(q=inp.values((batch, hq, 128), dtype), kv=inp.values((slots, 2 * hkv, 128), dtype), longest=longest)
    s["k"], s["v"] = s["kv"][:, :hkv], s["kv"][:, hkv:]
    s["table"], s["b_req_idx"] = _table(lengths, inp.permutation(slots)[:sum(lengths)].to(torch.int32))
    s["b_seq_len"], s["block"] = _i32(lengths), simulate.decode_block_seq(longest)
    s["mid_o"] = torch.empty((longest // s["block"] + 1, batch, hq, 128), dtype=torch.float32, device=DEV)
    s["mid_lse"] = torch.empty(s["mid_o"].shape[:3], dtype=torch.float32, device=DEV)
    return s


def _decode(s, case):
    return longserve_token_decode_attention_flash_decoding(
        s["q"], s["table"], s["b_req_idx"], s["b_seq_len"], s["mid_o"], s["mid_lse"], case["batch"], s["longest"],
        case["q_heads"], 128, s["k"], s["v"], s["block"])


def _run_decode(s, case):
    return list(_decode(s, case))


def _prepare_decode_layer(case, inp):
    lengths = [n + 1 for n in _lengths(case)]  # with the new token
    hq, hkv, batch, longest = case["q_heads"], case["kv_heads"], case["batch"], max(lengths)
    hidden, total = hq * 128, sum(lengths) - batch
    size = max(65536, 2 * total)
    mem = LongServeMemoryManager(size, torch.float16, hkv, 128, 1)
    req = LongServeReqManager(batch + 8, longest + 64, mem)
    mem.kv_buffer.normal_(0.0, 0.5, generator=inp.gen)
    # a pool in use: half of it is taken, by these requests and by others that have left, and what is free lies scattered
    held = mem.alloc(size)[inp.permutation(size)]
    mem.free(held[total:total + size // 2].contiguous())
    s = dict(mem=mem, req=req, table=req.req_to_token_indexs, pool=mem.kv_buffer[0], longest=longest)
    s["b_req_idx"] = req.alloc(batch).to(torch.int32)
    init_req_to_token_indexes(s["table"], s["b_req_idx"], _i32([n - 1 for n in lengths]), held[:total])
    s["b_seq_len"] = _i32(lengths)
    s["k"], s["v"] = s["pool"][:, :hkv], s["pool"][:, hkv:]
    s["hidden"], s["ffn_in"] = inp.values((batch, hidden), scale=1.0), inp.values((batch, hidden), scale=1.0)
    s["w"], s["w2"] = inp.values((hidden,)), inp.values((hidden,))
    s["q"], s["kv"] = inp.values((batch, hq, 128)), inp.values((batch, 2 * hkv, 128))
    s["gate_up"] = inp.values((batch, 2 * _inter(case)))
    s["cos"], s["sin"] = inp.angles(s["b_seq_len"] - 1, 128)
    s["block"] = simulate.decode_block_seq(longest)
    s["mid_o"] = torch.empty((longest // s["block"] + 1, batch, hq, 128), dtype=torch.float32, device=DEV)
    s["mid_lse"] = torch.empty(s["mid_o"].shape[:3], dtype=torch.float32, device=DEV)
    s["hkv"] = hkv
    return s


def _run_decode_layer(s, case):
    slots = s["mem"].alloc(case["batch"])
    if not case["fused_write"]:
        copy_kv_index_to_req(s["table"], s["b_req_idx"], s["b_seq_len"], slots)
    x = rms_norm(s["hidden"], s["w"], EPS)
    if case["fused_write"]:
        rotary_emb_write_kv(s["q"], s["kv"], s["cos"], s["sin"], slots, s["pool"], s["table"], s["b_req_idx"], s["b_seq_len"],
                            decode=True)
    else:
        rotary_emb(s["q"], s["kv"][:, :s["hkv"]], s["cos"], s["sin"])
        destindex_copy_kv(s["kv"], slots, s["pool"])
    o, lse = _decode(s, case)
    y = rms_norm(s["ffn_in"], s["w2"], EPS)
    silu_and_mul_inplace(s["gate_up"])
    s["mem"].free(slots)  # the requests are done: the next pass starts from the same pool
    return [slots, x, s["q"], s["kv"], o, lse, y, s["gate_up"], s["pool"], s["table"], s["mem"].mem_state]


def _shares(n, parts):
    """n tokens in contiguous ranges over the instances."""
    return [n * (j + 1) // parts - n * j // parts for j in range(parts)]


def _prepare_elastic(case, inp):
    lengths, dtype, hkv = _lengths(case), DTYPES[case["dtype"]], case["kv_heads"]
    s = dict(q=inp.values((case["batch"], case["q_heads"], 128), dtype), hkv=hkv, instances=[], kept={})
    for j in range(case["instances"]):
        held = [_shares(n, case["instances"])[j] for n in lengths]
        slots = sum(held) * 5 // 4
        table, rows = _table(held, inp.permutation(slots)[:sum(held)].to(torch.int32))
        s["instances"].append(simulate.DecodeInstance(inp.values((slots, 2 * hkv, 128), dtype), table, rows, _i32(held), max(held)))
    return s


def _run_elastic(s, case):
    return list(simulate.multi_instance_decode(s["q"], s["instances"], s["hkv"], workspace=s["kept"]))


def _prepare_prefill_layer(case, inp):
    lengths, hq, hkv = _lengths(case), case["q_heads"], case["kv_heads"]
    tokens, hidden = sum(lengths), hq * 128
    s = dict(lengths=_i32(lengths), starts=_i32(_starts(lengths)), longest=max(lengths), hkv=hkv)
    s["hidden"], s["ffn_in"] = inp.values((tokens, hidden), scale=1.0), inp.values((tokens, hidden), scale=1.0)
    s["w"], s["w2"] = inp.values((hidden,)), inp.values((hidden,))
    s["q"], s["kv"] = inp.values((tokens, hq, 128)), inp.values((tokens, 2 * hkv, 128))
    s["gate_up"] = inp.values((tokens, 2 * _inter(case)))
    s["cos"], s["sin"] = inp.angles(_positions(lengths), 128)
    s["pool"] = torch.zeros((tokens * 3 // 2 + 8, 2 * hkv, 128), dtype=torch.float16, device=DEV)
    s["slots"] = inp.permutation(s["pool"].shape[0])[:tokens].to(torch.int32)
    s["table"] = torch.full((len(lengths) + 2, max(lengths)), PAD, dtype=torch.int32, device=DEV)
    s["b_req_idx"] = _i32([len(lengths) + 1 - i for i in range(len(lengths))])
    return s


def _run_prefill_layer(s, case):
    x = rms_norm(s["hidden"], s["w"], EPS)
    if case["fused_write"]:
        rotary_emb_write_kv(s["q"], s["kv"], s["cos"], s["sin"], s["slots"], s["pool"], s["table"], s["b_req_idx"], s["lengths"],
                            s["starts"], s["longest"])
    else:
        rotary_emb(s["q"], s["kv"][:, :s["hkv"]], s["cos"], s["sin"])
        destindex_copy_kv(s["kv"], s["slots"], s["pool"])
        init_req_to_token_indexes(s["table"], s["b_req_idx"], s["lengths"], s["slots"], s["starts"], s["longest"])
    y = rms_norm(s["ffn_in"], s["w2"], EPS)
    silu_and_mul_inplace(s["gate_up"])
    return [x, s["q"], s["kv"], y, s["gate_up"], s["pool"], s["table"]]


_KINDS = {
    "prefill": (_prepare_prefill, _run_prefill),
    "ring": (_prepare_ring, _run_ring),
    "decode": (_prepare_decode, _run_decode),
    "decode_layer": (_prepare_decode_layer, _run_decode_layer),
    "elastic": (_prepare_elastic, _run_elastic),
    "prefill_layer": (_prepare_prefill_layer, _run_prefill_layer),
}


def prepare(case, seed):
    return case, _KINDS[case["kind"]][0](case, _Inputs(seed))


def run(state):
    case, s = state
    return _KINDS[case["kind"]][1](s, case)


def _token_wise_bytes(case, tokens):
    """Two norms, the activation, the rotation of q and k in place, a K/V row read and written to the pool."""
    hq, hkv = case["q_heads"], case["kv_heads"]
    return tokens * (2 * 2 * hq * 128 * 2 + 3 * _inter(case) * 2 + 2 * hq * 256 + 2 * hkv * 256 + 2 * hkv * 256 + 2 * hkv * 256
                     + 2 * 64 * 2 + 2 * 4)


def work(case):
    """Every input read once, every output written once; 4 * head_dim flops per query head and visible (query, key) pair."""
    kind, hq, hkv = case["kind"], case["q_heads"], case["kv_heads"]
    if kind == "prefill":
        lengths, d, ctx = _lengths(case), case["head_dim"], case["context"]
        tokens, keys = sum(lengths), sum(lengths) + ctx * len(lengths)
        pairs = sum(n * ctx + n * (n + 1) // 2 for n in lengths)
        out = 4 if case["result"] == "partial" else 2
        b = tokens * hq * (d * 2 + d * out + (4 if case["result"] == "partial" else 8)) + keys * 2 * hkv * d * 2
        b += tokens * (2 * hkv * d * 2 + 8) if case["kv_write"] else 0
        return {"bytes": b, "flops": 4 * d * hq * pairs}
    if kind == "ring":
        n, chunks = case["shard"], case["chunks"]
        diagonal = n * (n + 1) // 2  # (the last instance of a striped ring sees m + 1 keys of every chunk)
        pairs = diagonal * chunks if case["striped"] else diagonal + (chunks - 1) * n * n
        return {"bytes": n * hq * (2 * 256 + 8) + chunks * n * 2 * hkv * 256, "flops": 512 * hq * pairs}
    if kind == "decode_layer":
        lengths = [n + 1 for n in _lengths(case)]
        tokens, batch = sum(lengths), case["batch"]
        size = max(65536, 2 * (tokens - batch))
        b = tokens * (2 * hkv * 256 + 4) + batch * hq * (256 + 512 + 4) + _token_wise_bytes(case, batch)
        return {"bytes": b + size * 4 + batch * 24, "flops": 512 * hq * tokens}
    if kind in ("decode", "elastic"):
        tokens = sum(_lengths(case))
        out = 512 if kind == "decode" else 256
        return {"bytes": tokens * (2 * hkv * 256 + 4) + case["batch"] * hq * (256 + out + 4), "flops": 512 * hq * tokens}
    return {"bytes": _token_wise_bytes(case, sum(_lengths(case))), "flops": 0}


def tolerance(case):
    """Products of 16-bit values summed in fp32: what remains is the rounding of the probabilities and of the result."""
    if case.get("dtype") == "bf16":
        return {"rel": 1e-2}
    return {"rel": 2e-3}
