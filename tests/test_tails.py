"""Tails: the few tokens a request has behind a box of 17..64 rows, walked by that box's workgroup instead of one of their own
(PAT_BUCKET_TAILS in include/pat_amd.h). The planner's tables on the CPU; on the GPU the kernel against the oracle, and that one
request's tail stays out of the others' rows."""
import ctypes as C
import math
import random

import pytest
import torch

from oracle import attn_oracle as ao
from pat_amd import PrefixTreeCPP, _lib, prefix_attn_with_kvcache, workloads

TOL = {torch.float16: 2e-3, torch.bfloat16: 1.6e-2}


def _batch(seqs, prefix, tails, heads, d, dtype, page, seed=0):
    """`seqs` requests behind one prefix (a list: behind its parts, an even share of the requests each)."""
    r = random.Random(seed + seqs)
    parts = prefix if isinstance(prefix, list) else [prefix]
    rows, lens, nxt = [], [], 0
    nodes = []
    for p in parts:
        nodes.append(list(range(nxt, nxt + p // page)))
        nxt += p // page
    for s in range(seqs):
        node = nodes[s * len(nodes) // seqs]
        n = r.randint(*tails)
        need = -(-n // page)
        rows.append(node + list(range(nxt, nxt + need)))
        nxt += need
        lens.append(len(node) * page + n)
    return workloads.Workload("tails", heads[0], heads[1], d, dtype, page, lens, rows, nxt, 0, seed)


def _plan(w):
    tree = PrefixTreeCPP(w.page_size)
    tree.build_radix_tree(w.seq_lens, w.padded_table())
    tree.pack_schedule(None, w.heads // w.kv_heads, w.kv_heads)
    return tree


def _flat_layout(w):
    """pat_flat_plan and its buffer for the batch, through the C ABI."""
    lib = _lib.load()
    handle = C.c_void_p()
    assert lib.pat_tree_create(w.page_size, C.byref(handle)) == 0
    table = w.padded_table().contiguous()
    lens = (C.c_int32 * w.batch)(*w.seq_lens)
    assert lib.pat_tree_build(handle, lens, C.cast(table.data_ptr(), _lib.i32p), table.shape[0], table.shape[1]) == 0
    assert lib.pat_tree_pack(handle, None, 0, w.heads // w.kv_heads, w.kv_heads, 0, None) == 0
    flat = _lib.FlatPlan()
    assert lib.pat_tree_flat_plan(handle, C.byref(flat), None, 0) == 0
    buf = torch.full((flat.total,), -99, dtype=torch.int32)
    assert lib.pat_tree_flat_plan(handle, C.byref(flat), buf.data_ptr(), flat.total) == 0
    lib.pat_tree_destroy(handle)
    return flat, buf


@pytest.mark.parametrize("seqs,prefix,tails,heads,page", [
    (64, 640, (1, 32), (32, 8), 16),        # pairs, tails of two tile labels
    (38, 640, (20, 32), (32, 8), 16),       # six requests over: a box of 24 rows of another label
    (67, 512, (9, 16), (16, 8), 16),        # three over: a box of 6 rows, whose tails are nobody's
    (130, [256, 512], (1, 60), (8, 8), 64),
    (40, 640, (60, 120), (32, 8), 16),      # some too long: the others in a launch bucket of their own
    (40, 640, (65, 120), (32, 8), 16),      # all too long
])
def test_planner_tables(seqs, prefix, tails, heads, page):
    w = _batch(seqs, prefix, tails, heads, 128, torch.float16, page)
    flat, buf = _flat_layout(w)
    n = flat.num_launch_buckets
    holds = [i for i in range(n) if flat.tails >> (8 + i) & 1]
    tables = [i for i in range(n) if (flat.tails & 0xffffffff) >> (20 + i) & 1]
    if tails[0] > 64:
        assert flat.tails == 0
        return
    assert holds and tables
    view = lambda off, *shape: buf[off:off + math.prod(shape)].view(*shape)  # noqa: E731
    launch = flat.launch
    boxes = view(flat.num_boxes_per_seq, w.batch)
    claimed, counts = {}, None
    for i in tables:
        f = launch[i]
        assert f.mnw[0] > 16
        at = f.kv + f.num_boxes + 2 * f.num_items
        t = view(at, f.num_boxes, f.max_seqs)
        counts = view(at + f.num_boxes * f.max_seqs, w.batch)
        q, ns = view(f.q_table, f.num_boxes, f.max_seqs), view(f.num_seqs, f.num_boxes)
        for b in range(f.num_boxes):
            for j in range(f.max_seqs):
                e = int(t[b, j])
                if e < 0:
                    continue
                leaf = launch[e >> 27]
                row = e & ((1 << 27) - 1)
                assert j < ns[b] and e >> 27 in holds and row < leaf.num_boxes
                assert int(buf[leaf.q_table + row * leaf.max_seqs]) == int(q[b, j]) and int(buf[leaf.num_seqs + row]) == 1
                assert (e >> 27, row) not in claimed
                claimed[e >> 27, row] = int(q[b, j])
    assert sorted(claimed) == [(i, r) for i in holds for r in range(launch[i].num_boxes)]       # each tail once, all of them
    of_seq = torch.zeros(w.batch, dtype=torch.int32)
    for s in claimed.values():
        of_seq[s] += 1
    assert torch.equal(counts, boxes - of_seq) and int(counts.min()) >= 1 and int(counts.max()) == flat.tails & 0xff
    # a sequence's boxes are numbered 0.. in the launch copies, tails behind the others
    seen = [set() for _ in range(w.batch)]
    for i in range(n):
        f = launch[i]
        q, sl, ns = view(f.q_table, f.num_boxes, f.max_seqs), view(f.q_slot, f.num_boxes, f.max_seqs), view(f.num_seqs, f.num_boxes)
        for b in range(f.num_boxes):
            for j in range(int(ns[b])):
                s, o = int(q[b, j]), int(sl[b, j])
                assert o not in seen[s] and (o >= counts[s]) == (i in holds)
                seen[s].add(o)
    assert [sorted(x) for x in seen] == [list(range(int(c))) for c in boxes]
    # the scheduler-order tables know nothing of this
    tree = _plan(w)
    for b in range(flat.num_buckets):
        f = flat.buckets[b]
        assert torch.equal(view(f.q_slot, f.num_boxes, f.max_seqs), tree.kernel_info.slot_tables[b])


def _tail_args(tall, tails, heads, kv_heads, d, batch, page, most=1):
    b = (_lib.FwdBucket * 2)()
    for i, (m, boxes, seqs, tokens, flags, items) in enumerate([tall, tails]):
        b[i].q_table = b[i].block_table = b[i].num_seqs = b[i].rank = b[i].kv = b[i].q_slot = 0x10000
        b[i].mnw[:] = [m, 128, 4 if m == 64 else 1]
        b[i].num_boxes, b[i].max_seqs, b[i].max_blocks, b[i].num_items = boxes, seqs, tokens // page, items
        b[i].q_table_stride, b[i].block_table_stride, b[i].flags = seqs, tokens // page, flags
    a = _lib.FwdArgs()
    a.dtype, a.batch, a.seqlen_q, a.heads, a.kv_heads = _lib.PAT_DTYPE_F16, batch, 1, heads, kv_heads
    a.head_dim, a.page_size, a.num_pages = d, page, 1 << 16
    a.q = a.k = a.v = a.out = a.num_split_per_seq = 0x10000
    a.q_stride = a.o_stride = (C.c_int64 * 3)(heads * d, heads * d, d)
    a.k_stride = a.v_stride = (C.c_int64 * 3)(page * kv_heads * d, kv_heads * d, d)
    a.max_split_per_seq, a.max_seqs_in_box, a.max_blocks_in_box, a.softmax_scale = 2, tall[2], tall[3] // page, 0.1
    a.num_buckets, a.buckets = 2, C.cast(b, C.POINTER(_lib.FwdBucket))
    a._keep = b
    return a


def test_launch_rule(tuning):
    lib, g = _lib.load(), _lib.FwdGeometry()
    both = _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_ITEMS
    leaf = _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_TAIL | 1 << _lib.PAT_TAIL_BOXES_SHIFT

    def geometry(a):
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        return bool(g.flags & _lib.PAT_GEOMETRY_TAILS), g.num_slots, g.num_workgroups

    def many(tall_flags, leaf_flags, tokens=32):       # 1024 requests of 32 tokens over 2048 at 64/8 heads
        return _tail_args((64, 128, 8, 2048, both | tall_flags, 64), (16, 1024, 1, tokens, leaf_flags, 0), 64, 8, 128, 1024, 32)

    assert geometry(many(_lib.PAT_BUCKET_TAILS, leaf)) == (True, 1, 512)
    for a in (many(0, leaf), many(_lib.PAT_BUCKET_TAILS, _lib.PAT_BUCKET_EVEN), many(_lib.PAT_BUCKET_TAILS, leaf, 96),
              many(_lib.PAT_BUCKET_TAILS, leaf & 0xff)):       # not both flags, too wide, no count of the other boxes
        assert geometry(a)[0] is False
    need = C.c_size_t()
    assert lib.pat_fwd_workspace_bytes(C.byref(many(_lib.PAT_BUCKET_TAILS, leaf)), C.byref(need)) == 0
    records = need.value
    tuning(pairs=_lib.PAT_TAILS_NEVER)
    assert geometry(many(_lib.PAT_BUCKET_TAILS, leaf)) == (False, 2, 2560)
    assert lib.pat_fwd_workspace_bytes(C.byref(many(_lib.PAT_BUCKET_TAILS, leaf)), C.byref(need)) == 0 and need.value > 60 * records
    # two rows per sequence, tall boxes cut: a merge all the same, sixteen tails a wave
    few = _tail_args((64, 16, 32, 1408, _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_TAILS, 0), (16, 512, 1, 32, leaf, 0), 16, 8, 128, 512, 32)
    tuning()
    assert geometry(few)[0] is False
    tuning(pairs=_lib.PAT_TAILS_ALWAYS)
    assert geometry(few)[0] is True and g.tall_rows == 32
    tuning(pairs=_lib.PAT_TAILS_ALWAYS, tall_rows=16)          # (the form that has no tails)
    assert geometry(few)[0] is False


# ---- on the GPU ------------------------------------------------------------------------------------------
def _run(tree, w, q, k, v, scale, out=None, lse=None):
    out = torch.empty_like(q) if out is None else out
    lse = torch.empty((w.batch, w.heads), dtype=torch.float32, device=q.device) if lse is None else lse
    out.fill_(float("nan"))
    lse.fill_(float("nan"))
    prefix_attn_with_kvcache(q, k, v, tree, scale, out, softmax_lse=lse)
    torch.cuda.synchronize()
    return out, lse


def _close(name, out, lse, ref, dtype):
    err = (out.float().cpu() - ref[0].float()).abs().max().item()
    lerr = ((lse.cpu() - ref[1]).abs() / ref[1].abs().clamp_min(1.0)).max().item()
    print(f"[parity] {name}: max|out - ref| = {err:.3e}, LSE rel = {lerr:.3e}", flush=True)
    assert err <= TOL[dtype] and lerr <= 1e-4, name


@pytest.mark.gpu
@pytest.mark.parametrize("seqs,prefix,tails,heads,d,dtype,page,tune,scale", [
    (32, 256, (1, 64), (64, 8), 128, torch.float16, 16, dict(), 0.09),              # pairs, uncut: straight to `out`; one and two steps
    (64, 640, (31, 33), (32, 8), 128, torch.bfloat16, 16, dict(pairs=1), 0.09),     # steps of 1, 31 and 32 tokens
    (64, 640, (16, 17), (32, 8), 64, torch.float16, 16, dict(pairs=2), -0.1),       # a box a workgroup: two waves share the rows
    (38, 640, (1, 48), (32, 8), 128, torch.float16, 48, dict(), 0.09),              # a box of 24 rows; pages of 48
    (67, 512, (1, 16), (16, 8), 128, torch.bfloat16, 16, dict(), 0.09),             # tails that are nobody's beside the others
    (130, 1040, (1, 64), (8, 8), 64, torch.bfloat16, 16, dict(tall_chunk_tokens=256), 0.1),   # 64 sequences a box, pieces take their tails in turn
    (64, 1680, (1, 60), (16, 8), 128, torch.float16, 16, dict(tall_chunk_tokens=544, equalize_chunks=0), 0.09),   # tiles handed over apart
    (64, [256, 512, 2048, 128], (33, 64), (64, 8), 128, torch.bfloat16, 32, dict(), 0.0),     # boxes of 2 to 32 super-steps; scale 0
    (48, 528, (1, 3), (16, 16), 64, torch.float16, 16, dict(pairs=1), 0.1),         # rows of one sequence each
])
def test_against_the_oracle(seqs, prefix, tails, heads, d, dtype, page, tune, scale, tuning, monkeypatch):
    print(f"[case] tails: {seqs} x ({prefix} + {tails}), heads {heads}, d {d}, page {page}, {tune}", flush=True)
    monkeypatch.setenv("PAT_WHOLE_SEQUENCES", "0")
    w = _batch(seqs, prefix, tails, heads, d, dtype, page)
    q, k, v = w.tensors(torch.device("cuda:0"))
    ref = ao.paged_attention_ref(q.cpu(), k.cpu(), v.cpu(), w.rows, w.seq_lens, scale)
    for switch in (_lib.PAT_TAILS_ALWAYS, _lib.PAT_TAILS_NEVER):
        tuning(**{**dict(tall_rows=32), **tune, "pairs": tune.get("pairs", 0) | switch})
        tree = _plan(w)
        tree.kernel_info.to_gpu(q.device)
        out, lse = _run(tree, w, q, k, v, scale)
        assert [g["tails"] for g in tree.kernel_info._launch_geometries] == [switch == _lib.PAT_TAILS_ALWAYS]
        _close(f"switch {switch}", out, lse, ref, dtype)


@pytest.mark.gpu
def test_a_tail_stays_out_of_the_other_rows(tuning, monkeypatch):
    # infinite and NaN values in one request's tail make its own rows NaN and leave every other row as it was, to the bit
    print("[case] NaN and infinite values in one request's tail", flush=True)
    monkeypatch.setenv("PAT_WHOLE_SEQUENCES", "0")
    w = _batch(64, 640, (5, 40), (32, 8), 128, torch.float16, 16)
    q, k, v = w.tensors(torch.device("cuda:0"))
    tuning(tall_rows=32, pairs=_lib.PAT_TAILS_ALWAYS)
    tree = _plan(w)
    tree.kernel_info.to_gpu(q.device)
    clean, lse0 = _run(tree, w, q, k, v, 0.09)
    assert bool(torch.isfinite(clean).all())
    for victim, cache, value in ((7, k, float("nan")), (30, v, float("inf")), (63, v, float("nan"))):
        page = w.rows[victim][40]                   # the first block of its tail
        kept = cache[page].clone()
        cache[page] = value
        out, lse = _run(tree, w, q, k, v, 0.09)
        cache[page] = kept
        others = [s for s in range(w.batch) if s != victim]
        assert torch.equal(out[others], clean[others]) and torch.equal(lse[others], lse0[others])
        assert not bool(torch.isfinite(out[victim]).any())


@pytest.mark.gpu
def test_growing_in_place_and_capture(tuning, monkeypatch):
    # tails grow in their own bucket between steps, into spare columns of its table; a captured launch reads the tables as they
    # are at each replay and does without tails
    print("[case] tails that grow, eager and captured", flush=True)
    monkeypatch.setenv("PAT_WHOLE_SEQUENCES", "0")
    dev = torch.device("cuda:0")
    w = _batch(64, 640, (17, 24), (64, 8), 128, torch.float16, 32)
    q, k, v = w.tensors(dev)
    tuning(tall_rows=32, pairs=_lib.PAT_TAILS_ALWAYS)
    tree = _plan(w)
    info = tree.kernel_info
    info.to_gpu(dev)
    out, lse = torch.empty_like(q), torch.empty(w.batch, w.heads, device=dev)
    _run(tree, w, q, k, v, 0.09, out, lse)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        prefix_attn_with_kvcache(q, k, v, tree, 0.09, out, softmax_lse=lse)
    lt = info.launch_tables()
    leaves = [i for i, ns in enumerate(lt["num_seqs_per_CTAs"]) if int(ns.max()) == 1]
    lens = list(w.seq_lens)
    for step in range(3):
        held = info._items_hold()
        for i in leaves:
            lt["kv_in_CTAs"][i].add_(1)
        if held:
            info._hold_items()
        lens = [n + 1 for n in lens]
        ref = ao.paged_attention_ref(q.cpu(), k.cpu(), v.cpu(), w.rows, lens, 0.09)
        _run(tree, w, q, k, v, 0.09, out, lse)
        assert [g["tails"] for g in info._launch_geometries] == [True]
        _close(f"eager, step {step}", out, lse, ref, w.dtype)
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        _close(f"replay, step {step}", out, lse, ref, w.dtype)
    # a write that nobody vouches for: the launch goes box by box
    for i in leaves:
        lt["kv_in_CTAs"][i].sub_(1)
    _run(tree, w, q, k, v, 0.09, out, lse)
    assert [g["tails"] for g in info._launch_geometries] == [False]
    _close("after a write of somebody else", out, lse,
           ao.paged_attention_ref(q.cpu(), k.cpu(), v.cpu(), w.rows, [n - 1 for n in lens], 0.09), w.dtype)


def test_not_taken_where_a_merge_follows_all_the_same(tuning):
    # the rule counts a merge that tails save: not an `out` that the split kernel may not store to, nor one kept from it
    lib, g = _lib.load(), _lib.FwdGeometry()
    leaf = _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_TAIL | 1 << _lib.PAT_TAIL_BOXES_SHIFT

    def tails(**other):
        a = _tail_args((64, 128, 8, 2048, _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_ITEMS | _lib.PAT_BUCKET_TAILS, 64), (16, 1024, 1, 32, leaf, 0),
                       64, 8, 128, 1024, 32)
        for name, value in other.items():
            setattr(a, name, value)
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        return bool(g.flags & _lib.PAT_GEOMETRY_TAILS)

    assert tails() is True
    assert tails(out=0x10004) is False
    assert tails(o_stride=(C.c_int64 * 3)(64 * 130, 64 * 130, 130)) is False
    tuning(direct_out=0)
    assert tails() is False
    tuning(pairs=_lib.PAT_TAILS_ALWAYS)      # (asked for, they are walked by the tall workgroups and merged)
    assert tails(out=0x10004) is True


def test_an_item_count_that_is_none_is_refused():
    # the tails table is found behind so many items, with or without their own flag
    lib = _lib.load()
    leaf = _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_TAIL | 1 << _lib.PAT_TAIL_BOXES_SHIFT
    for items, ok in ((0, True), (64, True), (128, True), (-1, False), (129, False)):
        a = _tail_args((64, 128, 8, 2048, _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_TAILS, items), (16, 1024, 1, 32, leaf, 0), 64, 8, 128, 1024, 32)
        assert (lib.pat_fwd_validate(C.byref(a)) == 0) is ok, items


def test_lines_of_the_rule(tuning):
    lib, g = _lib.load(), _lib.FwdGeometry()
    leaf = _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_TAIL | 1 << _lib.PAT_TAIL_BOXES_SHIFT

    def tails(items, tokens, shared=1248, d=128, heads=(64, 8), page=16):         # boxes of 64 rows in twos, and an end a request
        seqs = 64 * heads[1] // heads[0]
        a = _tail_args((64, 2 * items, seqs, shared, _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_ITEMS | _lib.PAT_BUCKET_TAILS, items),
                       (16, 2 * items * seqs, 1, tokens, leaf, 0), *heads, d, 2 * items * seqs, page)
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        return bool(g.flags & _lib.PAT_GEOMETRY_TAILS)

    tuning()
    # more than four steps a wave: not where up to an eighth of the CUs have two workgroups (256, 264, 288, 296 and 512 workgroups)
    assert [tails(n, 64) for n in (32, 33, 36, 37, 64)] == [True, False, False, True, True]
    assert tails(33, 32) is True                                                                # four steps
    # tall boxes that leave CUs idle and would be cut: not where they are long
    assert tails(23, 16, shared=384) and not tails(18, 64, shared=1504) and not tails(16, 32, shared=4096)
    # many ends a wave
    assert not tails(8, 16, shared=768, heads=(16, 16))
    # a launch that would be in the 16-row form, which rounds less: where the ends and the merge alone pay, not for the form's sake
    for shared, taken in ((384, True), (64, False)):
        tuning(pairs=_lib.PAT_TAILS_NEVER)
        assert tails(23, 16, shared=shared, d=64) is False and g.tall_rows == 16
        tuning()
        assert tails(23, 16, shared=shared, d=64) is taken
