"""Lists: workgroups that walk several private boxes of one step each (32-row form, head_dim 128). When they are taken, and the
results at list ends, part lists, unfilled slots and lengths of a step."""
import ctypes as C
import random

import pytest
import torch

from oracle import attn_oracle as ao
from pat_amd import PrefixTreeCPP, _lib, prefix_attn_with_kvcache, workloads

EVEN = _lib.PAT_BUCKET_EVEN


def _args(tall, short, heads, kv_heads, batch, page, d=128):
    """(tile, boxes, sequences, tokens, flags) of two buckets, fake addresses."""
    b = (_lib.FwdBucket * 2)()
    for i, (m, boxes, seqs, tokens, flags) in enumerate([tall, short]):
        b[i].q_table = b[i].block_table = b[i].num_seqs = b[i].rank = b[i].kv = b[i].q_slot = 0x10000
        b[i].mnw[:] = [m, 128, 4 if m == 64 else 1]
        b[i].num_boxes, b[i].max_seqs, b[i].max_blocks, b[i].flags = boxes, seqs, tokens // page, flags
        b[i].q_table_stride, b[i].block_table_stride = seqs, tokens // page
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

    def geometry(a):
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        return bool(g.flags & _lib.PAT_GEOMETRY_LISTS), g.num_workgroups

    def batch(requests, end, **other):      # `requests` of 1408 tokens in boxes of 32 and an end each, 16/8 heads
        return _args((64, requests // 32, 32, 1408, EVEN), (16, requests, 1, end, EVEN), 16, 8, requests, 32, **other)

    assert geometry(batch(512, 32)) == (True, 512)
    assert geometry(batch(512, 64))[0] is False             # two steps
    assert geometry(batch(512, 32, d=64))[0] is False       # three places per CU
    assert geometry(batch(320, 32))[0] is False             # 1.75 times what fits at once it is not
    tuning(pairs=_lib.PAT_LISTS_NEVER)
    assert geometry(batch(512, 32)) == (False, 1280)
    tuning(pairs=_lib.PAT_LISTS_ALWAYS)
    assert geometry(batch(320, 32))[0] is True
    tuning(pairs=_lib.PAT_LISTS_ALWAYS, tall_rows=16)
    assert geometry(batch(320, 32))[0] is False


@pytest.mark.gpu
@pytest.mark.parametrize("seqs,prefix,ends,heads,dtype,page,chunk", [
    (131, 640, (1, 32), (32, 8), torch.float16, 16, 0),       # lists of two, the last of one box; two pages a box
    (515, 320, (31, 32), (16, 8), torch.bfloat16, 32, 0),     # lists of four; three requests that are no tall box's
    (290, 1040, (1, 16), (16, 16), torch.float16, 16, 256),   # the tall boxes in pieces: every box leaves slots unfilled
    (1801, 272, (1, 16), (8, 8), torch.bfloat16, 16, 0),      # lists of eight, more than fits at once
])
def test_against_the_oracle(seqs, prefix, ends, heads, dtype, page, chunk, tuning, monkeypatch):
    print(f"[case] lists: {seqs} x ({prefix} + {ends}), heads {heads}, page {page}, pieces of {chunk}", flush=True)
    monkeypatch.setenv("PAT_WHOLE_SEQUENCES", "0")
    r = random.Random(seqs)
    shared = prefix // page
    rows, lens, nxt = [], [], shared
    for s in range(seqs):
        n = r.randint(*ends)
        rows.append(list(range(shared)) + list(range(nxt, nxt + -(-n // page))))
        nxt += -(-n // page)
        lens.append(shared * page + n)
    w = workloads.Workload("lists", heads[0], heads[1], 128, dtype, page, lens, rows, nxt, 0, 3)
    q, k, v = w.tensors(torch.device("cuda:0"))
    ref_out, ref_lse = ao.paged_attention_ref(q.cpu(), k.cpu(), v.cpu(), rows, lens, 0.09)
    for lists in (True, False):
        tuning(tall_rows=32, tall_chunk_tokens=chunk, pairs=_lib.PAT_TAILS_NEVER | (_lib.PAT_LISTS_ALWAYS if lists else _lib.PAT_LISTS_NEVER))
        tree = PrefixTreeCPP(page)
        tree.build_radix_tree(lens, w.padded_table())
        tree.pack_schedule(None, heads[0] // heads[1], heads[1])
        tree.kernel_info.to_gpu(q.device)
        out = torch.full_like(q, float("nan"))
        lse = torch.full((w.batch, w.heads), float("nan"), dtype=torch.float32, device=q.device)
        for _ in range(2):    # (the second call finds the first one's partial rows in the workspace)
            prefix_attn_with_kvcache(q, k, v, tree, 0.09, out, softmax_lse=lse)
        torch.cuda.synchronize()
        assert [g["lists"] for g in tree.kernel_info._launch_geometries] == [lists]
        err = (out.float().cpu() - ref_out.float()).abs().max().item()
        lerr = ((lse.cpu() - ref_lse).abs() / ref_lse.abs().clamp_min(1.0)).max().item()
        print(f"[parity] lists {lists}: {err:.3e} {lerr:.3e}", flush=True)
        assert err <= (2e-3 if dtype == torch.float16 else 1.6e-2) and lerr <= 1e-4
    # NaN in one request's end stays its own
    tuning(tall_rows=32, tall_chunk_tokens=chunk, pairs=_lib.PAT_TAILS_NEVER | _lib.PAT_LISTS_ALWAYS)
    tree.pack_schedule(None, heads[0] // heads[1], heads[1])
    tree.kernel_info.to_gpu(q.device)
    prefix_attn_with_kvcache(q, k, v, tree, 0.09, out, softmax_lse=lse)
    victim = seqs // 2
    v[rows[victim][shared]] = float("nan")
    got = torch.empty_like(out)
    prefix_attn_with_kvcache(q, k, v, tree, 0.09, got)
    others = [s for s in range(seqs) if s != victim]
    assert torch.equal(got[others], out[others]) and not bool(torch.isfinite(got[victim]).any())


def test_static_launch_box_by_box_keeps_the_switches(tuning):
    # a launch with boxes in twos that its scratch does not hold is made box by box, and is otherwise the launch that was asked for. This one
    # is too large either way, and the error names the bytes: records of lists are fewer
    lib = _lib.load()
    a = _args((64, 128, 32, 1408, EVEN | _lib.PAT_BUCKET_ITEMS), (16, 4096, 1, 32, EVEN), 64, 32, 4096, 32)
    a._keep[0].num_items = 64
    sizes = []
    for lists in (_lib.PAT_LISTS_ALWAYS, _lib.PAT_LISTS_NEVER):
        switch = lists | _lib.PAT_STREAM_V_NEVER
        need = C.c_size_t()
        tuning(tall_rows=32, pairs=switch | _lib.PAT_TAILS_NEVER | 2)
        assert lib.pat_fwd_workspace_bytes(C.byref(a), C.byref(need)) == 0 and need.value > lib.pat_fwd_static_scratch_bytes()
        tuning(tall_rows=32, pairs=switch | 1)
        assert lib.pat_fwd_launch_static(C.byref(a), None) == -6, _lib.last_error()
        assert f"needs {need.value} bytes" in _lib.last_error()
        sizes.append(need.value)
    assert sizes[0] < sizes[1]


def test_boxes_without_blocks_are_no_lists(tuning):
    # (the record kernel divides by a list's pages per box)
    lib, g = _lib.load(), _lib.FwdGeometry()
    tuning(pairs=_lib.PAT_LISTS_ALWAYS)
    for end, lists in ((0, False), (32, True)):
        assert lib.pat_fwd_geometry_of(C.byref(_args((64, 16, 32, 1408, EVEN), (16, 512, 1, end, EVEN), 16, 8, 512, 32)), C.byref(g)) == 0
        assert bool(g.flags & _lib.PAT_GEOMETRY_LISTS) is lists


def test_lists_only_where_they_leave_nothing_waiting(tuning):
    # the lines of the rule: half the places left by the others, 2.25 times what fits at once
    lib, g = _lib.load(), _lib.FwdGeometry()

    def lists(boxes, requests):       # tall boxes in two pieces each, 8 kv heads: 16 workgroups a box; ends: two workgroups a request
        a = _args((64, boxes, 32, 1408, EVEN), (16, requests, 1, 32, EVEN), 16, 8, requests, 32)
        tuning(pairs=_lib.PAT_LISTS_NEVER, tall_rows=32)
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0 and g.num_workgroups == 16 * boxes + 2 * requests
        tuning(tall_rows=32)
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        return bool(g.flags & _lib.PAT_GEOMETRY_LISTS)

    assert lists(16, 448) and not lists(16, 447)        # 1152 workgroups
    assert lists(16, 600) and not lists(17, 600)        # 256 others
