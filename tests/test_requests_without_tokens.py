"""Requests of length 0 sit in no box of a plan: their rows come out as zeros with LSE -inf whatever form the launch takes. A launch
that stores `out` from the split kernel has nobody to write them, so it is not taken for such a batch (PAT_BUCKET_UNBOXED, or fewer
places in the boxes than requests). Host side on the CPU; on the GPU the rows, into buffers of NaN."""
import ctypes as C
import random

import pytest
import torch

from oracle import attn_oracle as ao
from pat_amd import PrefixTreeCPP, _lib, prefix_attn_with_kvcache, workloads

TOL = {torch.float16: 2e-3, torch.bfloat16: 1.6e-2}


def _batch(shared, lens, heads, d, dtype, page):
    """Requests of `lens` tokens behind `shared` common ones; a length of 0 is a request without any token at all."""
    node = list(range(shared // page))
    rows, nxt = [], len(node)
    for n in lens:
        need = -(-n // page)
        rows.append(node + list(range(nxt, nxt + need)) if n else [0])
        nxt += need
    total = [len(node) * page + n if n else 0 for n in lens]
    return workloads.Workload("without-tokens", heads[0], heads[1], d, dtype, page, total, rows, max(nxt, 1), 0, 3)


def _launch_args(w):
    """pat_fwd_args of the plan's launch copies at made-up addresses, tails and items handed over; and the flat plan."""
    lib, handle, flat = _lib.load(), C.c_void_p(), _lib.FlatPlan()
    assert lib.pat_tree_create(w.page_size, C.byref(handle)) == 0
    table = w.padded_table().contiguous()
    lens = (C.c_int32 * w.batch)(*w.seq_lens)
    assert lib.pat_tree_build(handle, lens, C.cast(table.data_ptr(), _lib.i32p), table.shape[0], table.shape[1]) == 0
    assert lib.pat_tree_pack(handle, None, 0, w.heads // w.kv_heads, w.kv_heads, 0, None) == 0
    assert lib.pat_tree_flat_plan(handle, C.byref(flat), None, 0) == 0
    lib.pat_tree_destroy(handle)
    n, base, word = flat.num_launch_buckets, 1 << 20, flat.tails & 0xffffffff
    b = (_lib.FwdBucket * n)()
    for i in range(n):
        f = flat.launch[i]
        for name in ("q_table", "q_slot", "block_table", "num_seqs", "rank", "kv"):
            setattr(b[i], name, base + 4 * getattr(f, name))
        b[i].mnw[:] = list(f.mnw)
        b[i].num_boxes, b[i].max_seqs, b[i].max_blocks, b[i].num_items = f.num_boxes, f.max_seqs, f.max_blocks, f.num_items
        b[i].q_table_stride, b[i].block_table_stride = max(f.max_seqs, 1), max(f.max_blocks, 1)
        b[i].flags = f.flags | (_lib.PAT_BUCKET_ITEMS if f.num_items else 0)
        b[i].flags |= (_lib.PAT_BUCKET_TAIL | (word & 0xff) << _lib.PAT_TAIL_BOXES_SHIFT) if word >> (8 + i) & 1 else 0
        b[i].flags |= _lib.PAT_BUCKET_TAILS if word >> (20 + i) & 1 else 0
    a, d = _lib.FwdArgs(), w.head_dim
    a.dtype, a.batch, a.seqlen_q, a.heads, a.kv_heads = _lib.PAT_DTYPE_F16, w.batch, 1, w.heads, w.kv_heads
    a.head_dim, a.page_size, a.num_pages = d, w.page_size, w.num_blocks
    a.q = a.k = a.v = a.out = base
    a.num_split_per_seq = base + 4 * flat.num_boxes_per_seq
    a.q_stride = a.o_stride = (C.c_int64 * 3)(w.heads * d, w.heads * d, d)
    a.k_stride = a.v_stride = (C.c_int64 * 3)(w.page_size * w.kv_heads * d, w.kv_heads * d, d)
    a.max_split_per_seq, a.softmax_scale = flat.max_boxes_per_seq, 0.1
    a.num_buckets, a.buckets = n, C.cast(b, C.POINTER(_lib.FwdBucket))
    a._keep = b
    return a, flat


def _merge_form(a):
    g = _lib.FwdGeometry()
    assert _lib.load().pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
    return g, (g.flags >> _lib.PAT_GEOMETRY_MERGE_SHIFT) & 7


@pytest.mark.parametrize("shared,lens,heads", [
    (2048, [32] * 1023, (64, 8)),       # tails by the rule
    (384, [1, 2, 3, 4] * 92, (64, 8)),  # the same, short
    (0, [320] * 40, (32, 8)),           # nothing shared, whole boxes
    (0, [690] * 5 + [600], (32, 32)),   # pieces of double length that leave one
])
@pytest.mark.parametrize("at", [None, 0, 5])
def test_a_merge_follows(shared, lens, heads, at, tuning):
    # without an empty request these launches write `out` themselves, with one they do not
    tuning()
    if at is not None:
        lens = lens[:at] + [0] + lens[at:]
    w = _batch(shared, lens, heads, 128, torch.float16, 32)
    a, flat = _launch_args(w)
    flags = [flat.launch[i].flags & _lib.PAT_BUCKET_UNBOXED for i in range(flat.num_launch_buckets)]
    assert all(flags) if at is not None else not any(flags)
    assert (_merge_form(a)[1] != 0) == (at is not None)
    # sizes alone tell it too where nothing is shared (the tables handed over one by one, without flags)
    if shared == 0:
        for i in range(a.num_buckets):
            a._keep[i].flags = 0
        assert (_merge_form(a)[1] != 0) == (at is not None)


@pytest.mark.gpu
@pytest.mark.parametrize("name,shared,lens,heads,d,dtype,page,switch,tails", [
    ("tails, forced", 640, (64, 5, 40), (32, 8), 128, torch.float16, 16, _lib.PAT_TAILS_ALWAYS, True),
    ("tails, forced, pieces", 1680, (48, 1, 60), (16, 8), 128, torch.bfloat16, 16, _lib.PAT_TAILS_ALWAYS, True),
    ("tails but for them", 384, (369, 1, 4), (64, 8), 64, torch.float16, 16, 0, False),
    ("unshared", 0, (40, 300, 320), (32, 8), 128, torch.bfloat16, 16, 0, False),
    ("unshared, head_dim 64", 0, (64, 100, 200), (8, 8), 64, torch.float16, 32, 0, False),
    ("pieces of double length", 0, (6, 600, 690), (32, 32), 128, torch.float16, 16, 0, False),
    ("eight waves asked for", 0, (8, 288, 288), (8, 8), 128, torch.float16, 16, _lib.PAT_WAVES_8, False),
])
@pytest.mark.parametrize("form", ["tree", "table"])
def test_rows_of_empty_requests(name, shared, lens, heads, d, dtype, page, switch, tails, form, tuning, monkeypatch):
    print(f"[case] requests without tokens: {name}, {form} form", flush=True)
    monkeypatch.setenv("PAT_WHOLE_SEQUENCES", "0")
    r = random.Random(lens[0])
    own = [r.randint(lens[1], lens[2]) for _ in range(lens[0])]
    empty = [0, lens[0] // 2, lens[0] + 2]
    for at in empty:
        own.insert(at, 0)
    w = _batch(shared, own, heads, d, dtype, page)
    q, k, v = w.tensors(torch.device("cuda:0"))
    full = [i for i in range(w.batch) if i not in empty]
    ref_out, ref_lse = ao.paged_attention_ref(q[full].cpu(), k.cpu(), v.cpu(), [w.rows[i] for i in full], [w.seq_lens[i] for i in full], 0.09)
    tuning(pairs=switch, **(dict(tall_rows=32) if tails else {}), **(dict(tall_chunk_tokens=544, equalize_chunks=0) if "pieces" in name and tails else {}))
    tree = PrefixTreeCPP(page)
    tree.build_radix_tree(w.seq_lens, w.padded_table())
    tree.pack_schedule(None, w.heads // w.kv_heads, w.kv_heads)
    i = tree.kernel_info
    i.to_gpu(q.device)
    out = torch.full_like(q, float("nan"))
    lse = torch.full((w.batch, w.heads), float("nan"), dtype=torch.float32, device=q.device)
    for _ in range(2):    # (the second call finds the first one's partial rows in the workspace)
        out.fill_(float("nan"))
        lse.fill_(float("nan"))
        if form == "tree":
            prefix_attn_with_kvcache(q, k, v, tree, 0.09, out, softmax_lse=lse)
        else:
            prefix_attn_with_kvcache(q, k, v, i.num_split_per_seq, i.q_tables, i.block_tables, i.num_seqs_per_CTAs, i.CTA_ranks, i.kv_in_CTAs,
                                     i.MNWs, i.max_split_per_seq, i.max_seqs_in_CTA, i.max_blocks_in_CTA, 0.09, out, None, softmax_lse=lse)
        torch.cuda.synchronize()
        if form == "tree":
            assert [g["tails"] for g in i._launch_geometries] == [tails]
        assert bool((out[empty] == 0).all()) and bool((lse[empty] == float("-inf")).all())
        err = (out[full].float().cpu() - ref_out.float()).abs().max().item()
        lerr = ((lse[full].cpu() - ref_lse).abs() / ref_lse.abs().clamp_min(1.0)).max().item()
        print(f"[parity] {err:.3e} {lerr:.3e}", flush=True)
        assert err <= TOL[dtype] and lerr <= 1e-4
