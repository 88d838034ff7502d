"""The decode batches by which the speed of this framework is measured, from the smallest call to the largest.

A case is one decode batch: a prefix tree over a paged KV cache, the head geometry, the element type and the public
entry point that serves it. `listed()` names the cases, `draw(rng)` gives more of the same ranges, `prepare` makes what a
program holds before the call, `run` is one call (or one decode step of several layers), `work` and `tolerance` say what
the call cannot do without and how far two correct implementations at this precision lie apart.

The fields of a case:
  tree      "n1,...,nk_l1,...,lk": level i has n_i nodes of l_i tokens, request r lies below node r * n_i // n_k of level i;
            the last length may be a range "lo-hi" (every request's own tail, drawn evenly). "forest:b,r" is a forest of b
            requests below r roots with random depths, fan-outs and lengths (pat_amd.workloads.forest)
  shape     seed of the lengths (which requests are long); the contents come from prepare's own seed
  heads, kv_heads, dim, dtype, page
  call      "tree": prefix_attn_with_kvcache(q, k, v, tree, scale, out), the plan in hand as between a step's layers
            "table": the same with the plan's tables passed one by one
            "step": a decode step from the batch's metadata on: plan, upload and the attention of `layers` layers
  lse       whether the log-sum-exp is asked for
  stacked   K and V are the two halves of one tensor, as serving engines allocate them, or two tensors
"""
import math
import random
from types import SimpleNamespace

import numpy as np
import torch

from pat_amd import PrefixTree, PrefixTreeCPP, prefix_attn_with_kvcache, workloads
from pat_amd.vllm_decode import DecodePlan, decode_attention

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}

# No case, drawn or listed, has more than this to do in one pass.
MOST_KV_BYTES = 540_000_000        # per layer
MOST_FLOPS = 71e9                  # per layer
MOST_STEP_BYTES = 2_750_000_000    # over the layers of a step


def _case(name, tree, heads, kv_heads, dim, dtype, page, call="tree", lse=False, stacked=False, layers=1, shape=0):
    case = {"name": name} if name else {}
    case.update(tree=tree, shape=shape, heads=heads, kv_heads=kv_heads, dim=dim, dtype=dtype, page=page, call=call,
                lse=lse, stacked=stacked, layers=layers)
    return case


def listed():
    return [
        # a handful of short chats behind one system prompt on a small model: launches and latency are all there is
        _case("chats-8", "1,8_256,32", 8, 8, 64, "fp16", 16),
        # one user alone with a 4k context: the whole chip for one request's KV
        _case("single-4k", "1_4096", 32, 8, 128, "bf16", 16, stacked=True),
        # a few dozen users of one assistant on a model without grouped heads; odd lengths
        _case("assistant-24", "1,24_784,33-300", 32, 32, 128, "fp16", 16, lse=True, shape=5),
        # the benchmark's headline: an 8B model's layer, 64 requests behind a 2048-token system prompt
        _case("prompt-64", "1,64_2048,64-512", 32, 8, 128, "bf16", 16),
        # three levels: system prompt, tenant prompt, conversation
        _case("levels-128", "1,8,128_1024,512,128-1024", 32, 8, 128, "fp16", 16),
        # an irregular forest (search over prompts), head_dim 64, no grouped heads
        _case("forest-256", "forest:256,16", 16, 16, 64, "fp16", 16),
        # one long document and 32 questions, a 70B model's layer
        _case("document-32", "1,32_16384,256-2048", 64, 8, 128, "bf16", 16),
        # nothing shared: plain paged decode at full memory traffic
        _case("unshared-32", "32_4096", 64, 8, 128, "bf16", 16),
        # offline evaluation: a thousand short items behind one few-shot prompt
        _case("fewshot-1024", "1,1024_2048,32", 64, 8, 128, "fp16", 32),
        # a deep tree with many requests, two query heads per KV head
        _case("deep-512", "1,4,16,512_1024,256,128,32", 16, 8, 128, "fp16", 32),
        # the tables passed one by one, ragged batch, pages of 48 tokens, two KV heads (a tensor-parallel slice)
        _case("tables-37", "1,5,37_2976,480,17-900", 16, 2, 128, "bf16", 48, call="table", lse=True, shape=7),
        # a whole decode step of an 8B model: metadata -> plan -> 32 layers
        _case("step-64", "1,64_2048,64-512", 32, 8, 128, "bf16", 16, call="step", stacked=True, layers=32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        heads, kv_heads = rng.choice([(8, 8), (16, 16), (32, 32), (16, 8), (16, 2), (32, 8), (64, 8)])
        dim = rng.choice([64, 128, 128, 128])
        page = rng.choice([16, 16, 16, 32, 48, 64])
        dtype = rng.choice(["fp16", "bf16"])
        call = rng.choice(["tree", "tree", "tree", "table", "step"])
        layers = _log_int(rng, 2, 32) if call == "step" else 1
        batch = _log_int(rng, 1, 1024)
        kind = rng.choice(["flat", "flat", "levels", "levels", "unshared", "forest"])
        if kind == "forest" and page == 16 and batch >= 16:
            tree = "forest:%d,%d" % (batch, max(1, batch // rng.choice([8, 12, 16])))
        else:
            lo = _log_int(rng, 1, 1024)
            tail = "%d-%d" % (lo, lo * rng.choice([1, 2, 4, 8]))
            whole = lambda n: page * max(1, n // page)  # noqa: E731  shared nodes are whole blocks
            if kind == "unshared" or batch < 4:
                counts, lens = [batch], ["%d-%d" % (whole(64 + 4 * lo), 64 + 6 * lo + page)]
            elif kind == "flat":
                counts, lens = [1, batch], [str(whole(_log_int(rng, 128, 16384))), tail]
            else:
                middle = max(2, batch // rng.choice([3, 8, 16]))
                counts, lens = [1, middle, batch], [str(whole(_log_int(rng, 128, 8192))), str(whole(_log_int(rng, 64, 1024))), tail]
                if middle >= 8 and rng.random() < 0.4:
                    counts.insert(1, 2), lens.insert(1, str(whole(_log_int(rng, 64, 512))))
            tree = ",".join(map(str, counts)) + "_" + ",".join(lens)
        case = _case(None, tree, heads, kv_heads, dim, dtype, page, call=call, lse=rng.random() < 0.3 and call != "step",
                     stacked=call == "step" or rng.random() < 0.5, layers=layers, shape=rng.randrange(1 << 20))
        nodes, _, lens = _layout(case)
        kv = sum(nodes) * _token_bytes(case)
        if kv <= MOST_KV_BYTES and kv * layers <= MOST_STEP_BYTES and _flops(case, lens) <= MOST_FLOPS:
            return case


def _token_bytes(case):
    return case["kv_heads"] * case["dim"] * 2 * 2


def _flops(case, lens):
    return 4.0 * case["dim"] * case["heads"] * sum(lens)


def _layout(case):
    """(tokens of every node, every request's block ids, every request's length): block ids not yet shuffled."""
    page = case["page"]
    if case["tree"].startswith("forest:"):
        batch, roots = map(int, case["tree"][7:].split(","))
        w = workloads.forest("forest", batch, roots, case["heads"], case["kv_heads"], case["dim"], DTYPES[case["dtype"]], case["shape"])
        return w.tree["node_tokens"], w.rows, w.seq_lens
    counts, lens = case["tree"].split("_")
    counts, lens = [int(c) for c in counts.split(",")], lens.split(",")
    rng = random.Random(case["shape"])
    batch, nodes, at = counts[-1], [], 0
    rows, total = [[] for _ in range(batch)], [0] * batch
    for count, length in zip(counts, lens):
        lo, hi = (int(x) for x in (length.split("-") if "-" in length else (length, length)))
        first = len(nodes)
        nodes += [rng.randint(lo, hi) for _ in range(count)]
        blocks = []
        for n in nodes[first:]:
            blocks.append(list(range(at, at + -(-n // page))))
            at += -(-n // page)
        for r in range(batch):
            rows[r] += blocks[r * count // batch]
            total[r] += nodes[first + r * count // batch]
    return nodes, rows, total


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    dtype, page, hq, hkv, dim = DTYPES[case["dtype"]], case["page"], case["heads"], case["kv_heads"], case["dim"]
    _, rows, lens = _layout(case)
    batch, layers = len(rows), case["layers"]
    # physical blocks are scattered over the cache, as an allocator leaves them after a while
    num_blocks = 1 + max(max(r) for r in rows)
    place = np.random.default_rng(seed).permutation(num_blocks).astype(np.int32)
    rows = [place[r] for r in rows]
    table = torch.zeros(batch, max(len(r) for r in rows), dtype=torch.int32)
    for i, r in enumerate(rows):
        table[i, :len(r)] = torch.from_numpy(r)

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=dev, dtype=dtype)

    state = SimpleNamespace(call=case["call"], scale=1.0 / math.sqrt(dim), lse=None)
    if case["call"] == "step":
        state.kv = [randn(2, num_blocks, page, hkv, dim) for _ in range(layers)]
        state.q, state.out = randn(layers, batch, hq, dim), torch.empty(layers, batch, hq, dim, device=dev, dtype=dtype)
        state.meta = SimpleNamespace(num_prefills=0, num_decode_tokens=batch, seq_lens=lens, block_tables=table.to(dev),
                                     block_tables_cpu=table, block_size=page, nheads=hq, nheads_kv=hkv, max_decode_query_len=1)
        return state
    if case["stacked"]:
        state.k, state.v = randn(2, num_blocks, page, hkv, dim)
    else:
        state.k, state.v = randn(num_blocks, page, hkv, dim), randn(num_blocks, page, hkv, dim)
    state.q = randn(batch, 1, hq, dim)
    state.out = torch.empty_like(state.q)
    if case["lse"]:
        state.lse = torch.empty(batch, hq, device=dev)
    if case["call"] == "table":
        tree = PrefixTree(page)
        tree.build_radix_tree(lens, [r.tolist() for r in rows])
        state.info = tree.pack_schedule(MNWs=None, HRatio=hq // hkv, kvHead=hkv)
        state.info.to_tensor(device=dev)
    else:
        state.tree = PrefixTreeCPP(page)
        state.tree.build_radix_tree(lens, table)
        state.tree.pack_schedule(None, hq // hkv, hkv)
        state.tree.kernel_info.to_gpu(dev)
    return state


def run(state):
    if state.call == "step":
        plan = DecodePlan.from_metadata(state.meta)
        for layer, kv in enumerate(state.kv):
            decode_attention(state.q[layer], kv, plan, state.scale, state.out[layer])
        return state.out
    if state.call == "table":
        i = state.info
        prefix_attn_with_kvcache(state.q, state.k, state.v, i.num_split_per_seq, i.q_tables, i.block_tables, i.num_seqs_per_CTAs,
                                 i.CTA_ranks, i.kv_in_CTAs, i.MNWs, i.max_split_per_seq, i.max_seqs_in_CTA, i.max_blocks_in_CTA,
                                 state.scale, state.out, None, softmax_lse=state.lse)
    else:
        prefix_attn_with_kvcache(state.q, state.k, state.v, state.tree, state.scale, state.out, softmax_lse=state.lse)
    return state.out if state.lse is None else {"out": state.out, "lse": state.lse}


def work(case):
    """Every K and V token of the tree read once, the queries read and the rows written once; a multiplication and an
    addition per query head, token and dimension for the scores and again for the weighted sum."""
    nodes, rows, lens = _layout(case)
    q = len(rows) * case["heads"] * case["dim"] * 2
    lse = len(rows) * case["heads"] * 4 if case["lse"] else 0
    return {"bytes": case["layers"] * (sum(nodes) * _token_bytes(case) + 2 * q + lse), "flops": case["layers"] * _flops(case, lens)}


def tolerance(case):
    # Against the same attention in 64 bits the listed cases are off by up to rel 2.9e-4, max 1.3e-3 (fp16) and rel 2.3e-3,
    # max 8.7e-3 (bf16): the rounding of the probabilities and of the result. Four times that.
    return {"rel": 1e-2, "max": 0.035} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 5.2e-3}
