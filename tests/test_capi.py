"""libpat_amd loads, exports every symbol include/pat_amd.h declares, and its GPU-free entry
points (argument validation, launch geometry, workspace size) behave. No kernel is launched."""
import ctypes as C
import os
import re

import pytest
import torch

from pat_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_functions():
    text = open(os.path.join(ROOT, "include", "pat_amd.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(pat_[a-z_0-9]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    names = _declared_functions()
    assert len(names) >= 15
    for name in names:
        assert hasattr(lib, name), f"libpat_amd.so does not export {name}"
    assert sorted(_lib.SYMBOLS) == names       # the ctypes table covers the header, no more, no less
    assert lib.pat_abi_version() == 4


def _args(**over):
    """A well-formed pat_fwd_args with fake (never dereferenced) device addresses."""
    fake = 0x10000
    b = (_lib.FwdBucket * 2)()
    for i, (m, boxes, seqs, blocks) in enumerate([(64, 4, 16, 128), (16, 64, 1, 32)]):
        b[i].q_table = b[i].block_table = b[i].num_seqs = b[i].rank = b[i].kv = fake
        b[i].q_table_stride, b[i].block_table_stride = seqs, blocks
        b[i].num_boxes, b[i].max_seqs, b[i].max_blocks = boxes, seqs, blocks
        b[i].mnw[0], b[i].mnw[1], b[i].mnw[2] = m, 128, 4 if m == 64 else 1
    a = _lib.FwdArgs()
    a.dtype, a.batch, a.seqlen_q, a.heads, a.kv_heads = _lib.PAT_DTYPE_BF16, 64, 1, 32, 8
    a.head_dim, a.page_size, a.num_pages = 128, 16, 4096
    a.q = a.k = a.v = a.out = a.num_split_per_seq = fake
    a.q_stride = (C.c_int64 * 3)(4096, 4096, 128)
    a.k_stride = (C.c_int64 * 3)(16 * 8 * 128, 8 * 128, 128)
    a.v_stride = (C.c_int64 * 3)(16 * 8 * 128, 8 * 128, 128)
    a.o_stride = (C.c_int64 * 3)(4096, 4096, 128)
    a.max_split_per_seq, a.max_seqs_in_box, a.max_blocks_in_box = 2, 16, 128
    a.softmax_scale = 0.088
    a.num_buckets, a.buckets = 2, C.cast(b, C.POINTER(_lib.FwdBucket))
    a._keep = b
    for k, v in over.items():
        setattr(a, k, v)
    return a


def test_validate_accepts_headline_shape():
    lib = _lib.load()
    assert lib.pat_fwd_validate(C.byref(_args())) == 0


@pytest.mark.parametrize("field,value,needle", [
    ("dtype", 7, "only support fp16 and bf16"),
    ("max_split_per_seq", 33, "only supports up to 32 splits"),
    ("max_split_per_seq", 0, "no case that a seq has no block"),
    ("head_dim", 96, "head_size_og must be 64 / 128"),
    ("page_size", 24, "divisible by 16"),
    ("kv_heads", 5, "must divide number of heads"),
    ("kv_heads", 2, "hq/hkv = 1, 2, 4, 8"),
    ("batch", 0, "batch size must be positive"),
    ("seqlen_q", 2, "decode only"),
    ("q", 0, "non-null"),
    ("num_buckets", 13, "between 1 and 12"),
])
def test_validate_rejects(field, value, needle):
    lib = _lib.load()
    rc = lib.pat_fwd_validate(C.byref(_args(**{field: value})))
    assert rc == _lib.PAT_ERR_INVALID
    assert needle in _lib.last_error()
    with pytest.raises(RuntimeError):
        _lib.check(rc)


def test_validate_rejects_bad_bucket_and_strides():
    lib = _lib.load()
    a = _args()
    a.buckets[0].mnw[0] = 48
    assert lib.pat_fwd_validate(C.byref(a)) == _lib.PAT_ERR_INVALID and "tile_q" in _lib.last_error()
    a = _args()
    a.k_stride = (C.c_int64 * 3)(16 * 8 * 128 + 4, 8 * 128, 128)
    assert lib.pat_fwd_validate(C.byref(a)) == _lib.PAT_ERR_INVALID and "multiples of 8" in _lib.last_error()
    a = _args()
    a.v_stride = (C.c_int64 * 3)(1 << 30, 8 * 128, 128)          # blocks 2^30 elements apart
    assert lib.pat_fwd_validate(C.byref(a)) == _lib.PAT_ERR_INVALID and "2^30 elements apart" in _lib.last_error()
    a = _args()
    a.k_stride = (C.c_int64 * 3)(1 << 29, 1 << 25, 128)          # a 16-token block spanning 2^29 elements
    assert lib.pat_fwd_validate(C.byref(a)) == _lib.PAT_ERR_INVALID and "span less than 1 GiB" in _lib.last_error()
    a = _args()
    a.buckets[1].max_seqs = 32      # 32 sequences x 4 heads per kv head > 64 rows
    a.buckets[1].q_table_stride = 32
    assert lib.pat_fwd_validate(C.byref(a)) == _lib.PAT_ERR_INVALID and "64 rows" in _lib.last_error()
    a = _args()
    a.buckets[1].max_seqs = 8       # 8 sequences x 4 heads = 32 rows in a bucket labelled tile_q 16
    a.buckets[1].q_table_stride = 8
    assert lib.pat_fwd_validate(C.byref(a)) == _lib.PAT_ERR_INVALID and "than its bucket's tile_q" in _lib.last_error()
    a.buckets[1].mnw[0] = 32        # ... which a tile_q 32 bucket holds
    assert lib.pat_fwd_validate(C.byref(a)) == 0


def test_geometry_and_workspace_are_consistent():
    lib = _lib.load()
    a = _args()
    g = _lib.FwdGeometry()
    assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0
    assert g.chunk_tokens % 32 == 0 and g.tall_chunk_tokens % 32 == 0
    # the whole launch is resident at two workgroups per CU: the tall boxes take the 32-row form and are cut
    # until there are about three tall workgroups per eight CUs: 3 pieces; the 64 boxes of up to 512 tokens
    # run a kv head per wave on 256-token pieces (2 per box, 2 head groups)
    assert g.tall_rows == 32
    per_box = [3, 2]
    assert -(-128 * 16 // g.tall_chunk_tokens) == per_box[0]
    assert g.chunks_per_rank == max(per_box)
    assert g.num_slots == g.chunks_per_rank * 2
    assert g.num_workgroups == 8 * 4 * per_box[0] + 64 * per_box[1] * (8 // 4)
    need = C.c_size_t()
    assert lib.pat_fwd_workspace_bytes(C.byref(a), C.byref(need)) == 0
    rows = 64 * 32 * g.num_slots
    assert need.value >= rows * 128 * 4 + rows * 4
    # launching without a workspace is refused before any GPU call
    a.workspace, a.workspace_bytes = 0, 0
    assert lib.pat_fwd_launch(C.byref(a), None) == _lib.PAT_ERR_WORKSPACE


def test_single_slot_launch_needs_no_workspace(tuning):
    # no sequence in two boxes (max_split_per_seq 1), every box one chunk, a box per CU and kv head:
    # the launch writes `out` from its first kernel (csrc/api.h:230-238) and, given the plan's
    # launch records, needs no scratch
    lib = _lib.load()
    fake = 0x10000

    def plan(boxes, blocks, **over):
        b = (_lib.FwdBucket * 1)()
        b[0].q_table = b[0].block_table = b[0].num_seqs = b[0].rank = b[0].kv = fake
        b[0].q_table_stride, b[0].block_table_stride = 1, blocks
        b[0].num_boxes, b[0].max_seqs, b[0].max_blocks = boxes, 1, blocks
        b[0].mnw[0], b[0].mnw[1], b[0].mnw[2] = 16, 128, 1
        kw = dict(batch=boxes, max_split_per_seq=1, max_seqs_in_box=1, max_blocks_in_box=blocks, num_buckets=1,
                  buckets=C.cast(b, C.POINTER(_lib.FwdBucket)), records=fake)
        kw.update(over)
        a = _args(**kw)
        a._keep = b
        g, need = _lib.FwdGeometry(), C.c_size_t()
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0
        assert lib.pat_fwd_workspace_bytes(C.byref(a), C.byref(need)) == 0
        return g, need.value

    tuning()
    g, need = plan(64, 100)                       # 64 boxes of 1600 tokens, 8 kv heads: 512 workgroups
    assert (g.chunks_per_rank, g.num_slots, need) == (1, 1, 0)
    g, need = plan(64, 100, out=fake + 2)         # `out` not 8-byte aligned: the two-kernel route
    assert g.num_slots == 1 and need > 0
    g, need = plan(64, 100, max_split_per_seq=2)  # some sequence sits in two boxes
    assert need > 0
    g, need = plan(16, 100)                       # 128 workgroups: cutting the boxes fills the device
    assert g.chunks_per_rank > 1 and need > 0
    g, need = plan(64, 200)                       # 3200 tokens: longer than a chunk can be
    assert g.chunks_per_rank > 1 and need > 0
    tuning(direct_out=0)
    g, need = plan(64, 100)
    assert g.num_slots == 1 and need > 0
    # without prebuilt records the launch writes them into its workspace: one per workgroup
    tuning()
    g, need = plan(64, 100, records=0)
    rec = C.c_size_t()
    a = _args()
    assert need > 0 and need % 256 == 0 and need >= g.num_workgroups * 64


def test_record_buffer_sizes_and_errors_without_a_gpu():
    lib = _lib.load()
    a = _args()
    g, need, rec = _lib.FwdGeometry(), C.c_size_t(), C.c_size_t()
    assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0
    assert lib.pat_fwd_records_bytes(C.byref(a), C.byref(rec)) == 0
    # a record: 32-byte header, sequence id and slot per sequence of the widest box (16), page ids of the
    # longest piece, rounded up to 64 bytes
    pages = max(g.chunk_tokens, g.tall_chunk_tokens) // 16
    assert rec.value >= g.num_workgroups * (32 + 2 * 16 * 4 + 4)
    assert rec.value <= 256 + g.num_workgroups * ((32 + 2 * 16 * 4 + pages * 4 + 63) // 64 * 64)
    # the launch's own workspace holds the partial results and, without prebuilt records, the records
    assert lib.pat_fwd_workspace_bytes(C.byref(a), C.byref(need)) == 0
    with_records = C.c_size_t()
    b = _args(records=0x20000)
    assert lib.pat_fwd_workspace_bytes(C.byref(b), C.byref(with_records)) == 0
    assert need.value == with_records.value + rec.value
    tag = C.c_uint64()
    assert lib.pat_fwd_build_records(C.byref(a), None, 0, C.byref(tag), None) == _lib.PAT_ERR_INVALID
    assert lib.pat_fwd_build_records(C.byref(a), C.c_void_p(0x10000), 16, C.byref(tag), None) == _lib.PAT_ERR_WORKSPACE
    assert lib.pat_fwd_build_records(C.byref(a), C.c_void_p(0x10010), rec.value, C.byref(tag), None) == _lib.PAT_ERR_WORKSPACE
    # records whose tag does not belong to this launch are refused before any GPU call
    b.workspace, b.workspace_bytes, b.records_bytes, b.records_tag = 0x100000, with_records.value, rec.value, 12345
    assert lib.pat_fwd_launch(C.byref(b), None) == _lib.PAT_ERR_INVALID and "launch records" in _lib.last_error()


def test_static_scratch_and_slot_buffer_sizes_without_a_gpu():
    lib = _lib.load()
    assert lib.pat_fwd_static_scratch_bytes() == 64 << 20
    a = _args()
    need = C.c_size_t()
    assert lib.pat_fwd_slots_bytes(C.byref(a), C.byref(need)) == 0
    # one count per sequence + one ordinal per q_table entry, each piece 256-byte aligned
    assert need.value == 256 + 256 + 256     # 64 counts, 4 x 16 and 64 x 1 entries
    offsets = (C.c_int64 * 2)()
    assert lib.pat_fwd_derive_slots(C.byref(a), None, 0, offsets, None) == _lib.PAT_ERR_INVALID
    assert lib.pat_fwd_derive_slots(C.byref(a), C.c_void_p(0x10000), 16, offsets, None) == _lib.PAT_ERR_WORKSPACE
    # a launch whose partial results exceed the built-in scratch is refused before any GPU call
    big = _args(batch=4096, max_split_per_seq=32)
    assert lib.pat_fwd_workspace_bytes(C.byref(big), C.byref(need)) == 0 and need.value > (64 << 20)
    assert lib.pat_fwd_launch_static(C.byref(big), None) == _lib.PAT_ERR_WORKSPACE
    assert "built-in scratch" in _lib.last_error()


def test_tuning_round_trip(tuning):
    lib = _lib.load()
    tuning(chunk_tokens=256, direct_out=0)
    t = _lib.FwdTuning()
    assert lib.pat_fwd_get_tuning(C.byref(t)) == 0
    assert (t.chunk_tokens, t.tall_chunk_tokens, t.head_per_wave_tokens, t.direct_out) == (256, 0, -1, 0)
    g = _lib.FwdGeometry()
    assert lib.pat_fwd_geometry_of(C.byref(_args()), C.byref(g)) == 0 and g.chunk_tokens == 256
    # the form of the tall path: chosen per launch unless set
    for rows in (32, 16):
        tuning(tall_rows=rows)
        assert lib.pat_fwd_geometry_of(C.byref(_args()), C.byref(g)) == 0 and g.tall_rows == rows
    tuning(tall_rows=16)
    assert lib.pat_fwd_geometry_of(C.byref(_args()), C.byref(g)) == 0
    assert -(-128 * 16 // g.tall_chunk_tokens) == 4      # the 16-row form: a tall workgroup per two CUs


def test_tree_handles_and_errors():
    lib = _lib.load()
    h = C.c_void_p()
    assert lib.pat_tree_create(0, C.byref(h)) == _lib.PAT_ERR_INVALID
    assert lib.pat_tree_create(16, C.byref(h)) == 0
    view = _lib.PlanView()
    assert lib.pat_tree_plan(h, C.byref(view)) == _lib.PAT_ERR_INVALID and "no plan" in _lib.last_error()
    assert lib.pat_tree_num_nodes(h) == 1
    nv = _lib.NodeView()
    assert lib.pat_tree_node(h, 5, C.byref(nv)) == _lib.PAT_ERR_INDEX
    lib.pat_tree_destroy(h)


def test_baseline_workspace_and_errors_without_a_gpu():
    lib = _lib.load()
    fake = 0x10000
    a = _lib.BaselineArgs()
    a.dtype, a.batch, a.heads, a.kv_heads, a.head_dim = _lib.PAT_DTYPE_F16, 32, 64, 8, 128
    a.page_size, a.num_pages, a.max_blocks = 16, 8192, 256
    a.q = a.k = a.v = a.out = a.block_table = a.seq_lens = fake
    a.q_stride = (C.c_int64 * 3)(8192, 8192, 128)
    a.o_stride = (C.c_int64 * 3)(8192, 8192, 128)
    a.k_stride = (C.c_int64 * 3)(16 * 8 * 128, 8 * 128, 128)
    a.v_stride = (C.c_int64 * 3)(16 * 8 * 128, 8 * 128, 128)
    a.block_table_stride, a.softmax_scale = 256, 0.088
    need = C.c_size_t()
    assert lib.pat_paged_decode_baseline_workspace_bytes(C.byref(a), C.byref(need)) == 0
    # partial rows of 4096-token requests (>= 2 chunks) plus the three per-request tables
    assert need.value >= 32 * 64 * 2 * (128 + 1) * 4 + 3 * 32 * 4
    assert lib.pat_paged_decode_baseline_launch(C.byref(a), None) == _lib.PAT_ERR_WORKSPACE
    a.max_blocks = 0
    assert lib.pat_paged_decode_baseline_workspace_bytes(C.byref(a), C.byref(need)) == _lib.PAT_ERR_INVALID
    assert "max_blocks" in _lib.last_error()
    a.max_blocks, a.kv_heads = 256, 5
    assert lib.pat_paged_decode_baseline_workspace_bytes(C.byref(a), C.byref(need)) == _lib.PAT_ERR_INVALID


def test_form_of_the_tall_path_follows_the_launch():
    """32-row tiles when the whole launch is resident at two workgroups per CU or its long tall boxes
    outweigh the short ones; the 16-row form (a third resident workgroup per CU) otherwise."""
    lib = _lib.load()
    g = _lib.FwdGeometry()

    def form(tall_boxes, tall_blocks, short_boxes, short_blocks, batch):
        a = _args(batch=batch)
        b = a._keep
        b[0].num_boxes, b[0].max_blocks, b[0].block_table_stride = tall_boxes, tall_blocks, tall_blocks
        b[1].num_boxes, b[1].max_blocks, b[1].block_table_stride = short_boxes, short_blocks, short_blocks
        a.max_blocks_in_box = max(tall_blocks, short_blocks)
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        return g.tall_rows, g.num_workgroups

    assert form(4, 128, 64, 32, 64)[0] == 32            # the headline batch: everything resident at once
    assert form(16, 64, 128, 64, 128)[0] == 16          # a 3-level tree: 1024-token leaves outweigh the tall boxes
    assert form(24, 171, 32, 128, 32)[0] == 32          # a 16k prefix in 2736-token tall boxes over 2048-token suffixes
    assert form(128, 8, 1024, 2, 1024)[0] == 16         # many short tall boxes over a thousand 32-token leaves
    assert form(0, 128, 512, 64, 512)[0] == 16          # no tall box at all

    # items of two boxes: hundreds of two- to five-page boxes at 2 kv heads wait for places (32-row form 6-9 % slower), a few
    # workgroups of four heads each do not (9 % faster); head_dim 64, where the 32-row form costs no place, without items
    def form_of(buckets, heads, kv_heads, d, batch):
        a = _args(batch=batch, heads=heads, kv_heads=kv_heads, head_dim=d)
        a.q_stride = a.o_stride = (C.c_int64 * 3)(heads * d, heads * d, d)
        a.k_stride = a.v_stride = (C.c_int64 * 3)(16 * kv_heads * d, kv_heads * d, d)
        bs = (_lib.FwdBucket * len(buckets))()
        for b, (tile, boxes, seqs, tokens, flags, items) in zip(bs, buckets):
            b.q_table = b.block_table = b.num_seqs = b.rank = b.kv = 0x10000
            b.mnw[0], b.mnw[1], b.mnw[2] = tile, 64, 4
            b.num_boxes, b.max_seqs, b.max_blocks, b.flags, b.num_items = boxes, seqs, tokens // 16, flags, items
            b.q_table_stride, b.block_table_stride = seqs, tokens // 16
        a.num_buckets, a.buckets, a.max_blocks_in_box = len(bs), C.cast(bs, C.POINTER(_lib.FwdBucket)), 400
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        return g.tall_rows, bool(g.flags & _lib.PAT_GEOMETRY_PAIRS), g.num_slots

    both = _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_ITEMS
    assert form_of([(64, 97, 8, 400, both, 49), (16, 1, 1, 448, 1, 0), (16, 108, 1, 80, 1, 0), (16, 387, 1, 64, 0, 0),
                    (16, 281, 1, 32, 0, 0)], 16, 2, 128, 777)[:2] == (16, False)
    assert form_of([(64, 25, 8, 512, both, 13), (16, 198, 1, 32, 1, 0)], 64, 8, 128, 198)[:2] == (32, True)
    assert form_of([(64, 12, 16, 3968, 0, 0), (32, 1, 6, 3968, 0, 0), (16, 102, 1, 1776, 0, 0)], 32, 8, 64, 102)[:2] == (32, False)


def _bucket_args(buckets, heads, kv_heads, d, batch, page):
    """Args of a launch of (tile, boxes, sequences, tokens, flags, items) buckets, fake addresses."""
    a = _args(batch=batch, heads=heads, kv_heads=kv_heads, head_dim=d, page_size=page)
    a.q_stride = a.o_stride = (C.c_int64 * 3)(heads * d, heads * d, d)
    a.k_stride = a.v_stride = (C.c_int64 * 3)(page * kv_heads * d, kv_heads * d, d)
    bs = (_lib.FwdBucket * len(buckets))()
    for b, (tile, boxes, seqs, tokens, flags, items) in zip(bs, buckets):
        b.q_table = b.block_table = b.num_seqs = b.rank = b.kv = 0x10000
        b.mnw[0], b.mnw[1], b.mnw[2] = tile, 64, 4
        b.num_boxes, b.max_seqs, b.max_blocks, b.flags, b.num_items = boxes, seqs, tokens // page, flags, items
        b.q_table_stride, b.block_table_stride = seqs, tokens // page
    a.num_buckets, a.buckets, a.max_blocks_in_box, a._keep = len(bs), C.cast(bs, C.POINTER(_lib.FwdBucket)), 400, bs
    return a


def test_one_long_short_box_does_not_multiply_every_rows_slots():
    """The few requests that a node's tall boxes leave over keep the whole shared length in a box of <= 16 rows; how it is
    cut sets the partial slots of all rows. Pairs and the 1024-token bound on its pieces cut such boxes finer only where
    no row gets more slots for it."""
    lib, g, need = _lib.load(), _lib.FwdGeometry(), C.c_size_t()
    even, both = _lib.PAT_BUCKET_EVEN, _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_ITEMS
    cases = [  # (args, slots of a row)
        (_bucket_args([(64, 83, 8, 1152, both, 42), (16, 1, 2, 1152, even, 0), (16, 596, 1, 96, 0, 0), (16, 70, 1, 48, 0, 0)], 64, 8, 128, 666, 48), 2),
        (_bucket_args([(64, 27, 16, 3888, both, 14), (16, 1, 1, 3984, even, 0), (16, 32, 1, 96, 0, 0), (16, 269, 1, 96, 0, 0),
                       (16, 131, 1, 48, 0, 0)], 32, 8, 128, 433, 48), 6),
        (_bucket_args([(64, 6, 64, 6880, both, 3), (16, 1, 6, 6880, even, 0), (16, 390, 1, 32, 0, 0)], 16, 16, 128, 390, 16), 12),
        (_bucket_args([(64, 61, 8, 2176, even, 0), (16, 1, 1, 2304, even, 0), (16, 488, 1, 128, even, 0)], 64, 8, 128, 489, 16), 4),
    ]
    for a, slots in cases:
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        assert g.num_slots == slots
        assert lib.pat_fwd_workspace_bytes(C.byref(a), C.byref(need)) == 0 and need.value <= lib.pat_fwd_static_scratch_bytes()
    # pieces of 1024 tokens where the tall boxes have as many anyway
    a = _bucket_args([(64, 24, 8, 2736, even, 0), (16, 32, 1, 2048, 0, 0)], 64, 8, 128, 32, 16)
    assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0 and (g.chunk_tokens, g.chunks_per_rank) == (1024, 2)


def test_tall_boxes_are_cut_by_what_a_workgroup_takes_ends_included():
    lib, g, need = _lib.load(), _lib.FwdGeometry(), C.c_size_t()
    even, both = _lib.PAT_BUCKET_EVEN, _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_ITEMS

    def plan(max_split, *args):
        a = _bucket_args(*args)
        a.max_split_per_seq = max_split
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        assert lib.pat_fwd_workspace_bytes(C.byref(a), C.byref(need)) == 0
        return g

    # in two: the chain of 352 tokens alone is shorter than the launch, with the workgroup's ends it is not
    assert plan(3, [(64, 1, 24, 352, even, 0), (16, 3, 8, 992, even, 0), (16, 24, 8, 512, 0, 0)], 16, 8, 128, 24, 16).tall_chunk_tokens == 256
    assert plan(2, [(64, 53, 8, 1440, both, 27), (16, 1, 1, 1472, even, 0), (16, 424, 1, 32, even, 0)], 64, 8, 64, 425, 32).tall_chunk_tokens == 768
    # not in two: 34 slots a row are past the 32 that the merge requests at once with four waves, and one piece is put at less than that
    assert plan(17, [(32, 16, 10, 336, even, 0), (16, 10, 8, 48, 0, 0)], 16, 8, 128, 10, 48).num_slots == 17
    # ... but in 384-token pieces where those of 32 slots would be more than twice as long
    assert plan(3, [(64, 1, 33, 8096, even, 0), (32, 1, 17, 864, even, 0), (16, 1, 16, 864, even, 0), (16, 33, 1, 32, 0, 0)], 8, 8, 64, 33, 32).tall_chunk_tokens == 384
    # a forest of nine boxes per request: fewer pieces than its chains call for, so that the partial rows stay in bounds
    plan(9, [(64, 2, 7, 3216, 0, 0), (64, 9, 7, 816, 0, 0), (32, 6, 4, 480, 0, 0), (16, 13, 2, 512, 0, 0), (16, 43, 2, 384, 0, 0),
             (16, 24, 2, 128, 0, 0)], 64, 8, 128, 66, 16)
    assert g.num_slots == 18 and need.value <= 48 << 20


@pytest.mark.parametrize("force", [0, 32])
def test_pieces_too_long_for_the_32_row_form_take_the_other(force, tuning):
    # 64 pieces a box at most, so a box of more than 64 x 4096 tokens is cut into pieces longer than that form takes
    lib, g = _lib.load(), _lib.FwdGeometry()
    if force:
        tuning(tall_rows=force)
    for tokens, rows in ((64 * 4096, 32), (64 * 4096 + 64, 16)):
        a = _bucket_args([(64, 2, 16, tokens, _lib.PAT_BUCKET_ITEMS, 1), (16, 32, 1, 64, 0, 0)], 32, 8, 128, 32, 64)
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        assert g.tall_rows == rows and g.chunks_per_rank <= 64 and not (rows == 16 and g.flags & _lib.PAT_GEOMETRY_PAIRS)


@pytest.mark.skipif(torch.cuda.is_available(), reason="would launch on fake addresses")
def test_static_launch_that_only_fits_box_by_box_is_not_refused():
    # records of items hold twice the sequences: 65.8 MiB with the boxes in twos, 64.0 one by one
    lib, need = _lib.load(), C.c_size_t()
    a = _bucket_args([(64, 8, 64, 7744, _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_ITEMS, 4), (16, 482, 1, 64, 0, 0)], 32, 32, 128, 482, 64)
    assert lib.pat_fwd_workspace_bytes(C.byref(a), C.byref(need)) == 0 and need.value > lib.pat_fwd_static_scratch_bytes()
    assert lib.pat_fwd_launch_static(C.byref(a), None) == _lib.PAT_ERR_HIP      # (got past the check: there is no GPU here)


@pytest.mark.parametrize("tile,boxes,seqs,tokens,heads,kv_heads,d,even,whole", [
    (16, 24, 1, 640, 32, 8, 128, True, False), (16, 27, 1, 768, 64, 8, 128, True, False), (16, 26, 1, 624, 8, 8, 64, True, False),
    (16, 20, 1, 896, 16, 8, 128, False, False), (16, 30, 1, 1152, 8, 8, 128, False, False), (16, 31, 1, 896, 16, 8, 128, False, False),   # ragged: one long box, maybe
    (64, 1, 16, 640, 32, 8, 128, True, False), (64, 30, 8, 1920, 64, 8, 128, True, False), (64, 28, 8, 1536, 64, 8, 128, True, False),   # requests with one table
    (16, 3, 1, 736, 16, 8, 128, True, False), (16, 8, 1, 1344, 16, 16, 128, True, False), (16, 1, 1, 4096, 32, 8, 128, True, False),
    (16, 64, 1, 2048, 32, 8, 128, True, True), (16, 8, 1, 512, 8, 8, 128, True, True), (16, 32, 1, 1152, 8, 8, 128, False, True),
])
def test_boxes_of_one_request_each_walked_whole_or_cut(tile, boxes, seqs, tokens, heads, kv_heads, d, even, whole):
    # one slot a row, written by the split kernel, for short boxes and where there is one per CU and kv head; longer ones of small
    # launches are cut, whatever their rows and whether or not the bucket is even
    lib, g = _lib.load(), _lib.FwdGeometry()
    a = _bucket_args([(tile, boxes, seqs, tokens, _lib.PAT_BUCKET_EVEN if even else 0, 0)], heads, kv_heads, d, boxes * seqs, 16)
    a.max_split_per_seq = 1
    assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
    assert (g.num_slots == 1) == whole, g.num_slots


@pytest.mark.parametrize("buckets,heads,kv_heads,d,workgroups", [
    ([(16, 24, 1, 272, 0, 0), (16, 3, 1, 128, 0, 0)], 16, 8, 128, 600),                                  # 24 WGs on four waves each, 6 on a head per wave
    ([(16, 24, 1, 272, 0, 0), (16, 3, 1, 96, 0, 0)], 16, 8, 128, 582),                                   # three steps: a head per wave
    ([(64, 3, 64, 192, 0, 0), (16, 1, 1, 192, 0, 0), (16, 206, 1, 80, 0, 0)], 8, 8, 128, 444),
    ([(64, 1, 32, 1696, 0, 0), (32, 2, 16, 480, 0, 0), (16, 23, 1, 256, 0, 0), (16, 8, 1, 128, 0, 0), (16, 2, 1, 64, 0, 0)], 16, 8, 128, 476),   # would queue
])
def test_few_boxes_of_several_steps_stay_on_four_waves(buckets, heads, kv_heads, d, workgroups):
    # ... in launches that are resident all the same
    lib, g = _lib.load(), _lib.FwdGeometry()
    a = _bucket_args(buckets, heads, kv_heads, d, 25, 16)
    a.max_split_per_seq = 4
    assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
    assert g.num_workgroups == workgroups, (g.num_workgroups, g.tall_rows)


def test_switches_in_one_field_do_not_leak_into_each_other(tuning, monkeypatch):
    # pat_fwd_tuning.pairs: 0..2, and two bits about V; other values, and other values of the environment variables, are automatic
    lib, g, t = _lib.load(), _lib.FwdGeometry(), _lib.FwdTuning()
    items = _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_ITEMS

    def flags(boxes, short):
        a = _bucket_args([(64, boxes, 8, 2048, items, boxes // 2), (16, 64, 1, short, _lib.PAT_BUCKET_EVEN, 0)], 64, 8, 128, 8 * boxes, 16)
        a.max_split_per_seq = 2
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        return bool(g.flags & _lib.PAT_GEOMETRY_PAIRS), bool(g.flags & _lib.PAT_GEOMETRY_STREAM_V)

    tuning(pairs=0)
    large, small = flags(16, 2048), flags(4, 64)      # (pairs and V past the caches pay, neither does)
    assert large == (True, True) and small == (False, False)
    for value in (-1, -2, -3, 3, 16, 17, 18, 20, 1 << 30):
        tuning(pairs=value)
        assert (flags(16, 2048), flags(4, 64)) == (large, small), value
    tuning(pairs=2 | _lib.PAT_STREAM_V_NEVER)
    assert flags(16, 2048) == (False, False)
    tuning(pairs=1 | _lib.PAT_STREAM_V_ALWAYS)
    assert flags(4, 64) == (True, True)
    for pairs, stream, want in (("1", "2", 1 | 8), ("4", "", 0), ("8", "1", 4), ("-1", "", 0), ("7", "3", 0), ("2", "1", 2 | 4)):
        monkeypatch.setenv("PAT_PAIRS", pairs)
        monkeypatch.setenv("PAT_STREAM_V", stream)
        assert lib.pat_fwd_set_tuning(None) == 0 and lib.pat_fwd_get_tuning(C.byref(t)) == 0
        assert t.pairs == want, (pairs, stream)


@pytest.mark.skipif(torch.cuda.is_available(), reason="would launch on fake addresses")
def test_static_launch_box_by_box_with_the_switch_out_of_range(tuning):
    # the second geometry, without boxes in twos, is asked for by a value of its own: -1 with two bits replaced would be automatic again
    lib = _lib.load()
    tuning(pairs=-1)
    a = _bucket_args([(64, 8, 64, 7744, _lib.PAT_BUCKET_EVEN | _lib.PAT_BUCKET_ITEMS, 4), (16, 482, 1, 64, 0, 0)], 32, 32, 128, 482, 64)
    assert lib.pat_fwd_launch_static(C.byref(a), None) == _lib.PAT_ERR_HIP      # (past the check of the size: there is no GPU here)


@pytest.mark.parametrize("slots,rows,d,form", [
    (8, 16383, 128, 1), (8, 16384, 128, 2), (9, 3640, 128, 3), (9, 3641, 128, 1), (32, 1024, 64, 3), (32, 1032, 64, 1),
    (33, 868, 128, 4), (33, 872, 128, 5), (64, 896, 64, 4), (64, 904, 64, 5), (64, 448, 128, 4), (64, 456, 128, 6), (65, 8, 64, 6),
    (65, 768, 128, 6), (65, 776, 128, 5), (320, 3072, 64, 5), (40, 3072, 128, 5), (40, 3080, 128, 1), (34, 4096, 64, 1), (320, 8192, 128, 1),
])
def test_the_merge_kernels_form_by_slots_and_rows(slots, rows, d, form, tuning):
    # (rows of 8 heads each but where the line is not at a multiple of 8)
    lib, g = _lib.load(), _lib.FwdGeometry()
    heads = next(h for h in (8, 4, 1) if rows % h == 0)
    tuning(chunk_tokens=32, head_per_wave_long_wgs=1 << 40, equalize_chunks=0)
    splits = next(s for s in range(1, 33) if slots % s == 0 and slots // s <= 64)
    a = _bucket_args([(16, rows // heads, 1, 32 * (slots // splits), 0, 0)], heads, heads, d, rows // heads, 16)
    a.max_split_per_seq = splits
    assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
    assert g.num_slots == slots and (g.flags >> _lib.PAT_GEOMETRY_MERGE_SHIFT) & 7 == form, (g.num_slots, g.flags >> 8)


@pytest.mark.parametrize("buckets,heads,kv_heads,d,workgroups", [
    ([(16, 1, 1, 1536, 1, 0), (16, 3, 1, 384, 1, 0), (16, 5, 1, 112, 0, 0), (16, 16, 1, 64, 0, 0), (16, 14, 1, 32, 1, 0)], 16, 16, 128, 204),
    ([(16, 3, 1, 528, 1, 0), (16, 5, 1, 128, 0, 0), (16, 6, 1, 64, 0, 0), (16, 4, 1, 32, 0, 0)], 32, 32, 128, 216),
    ([(16, 9, 1, 336, 1, 0), (16, 4, 1, 112, 0, 0), (16, 1, 1, 64, 0, 0)], 32, 32, 128, 184),     # the long ones run a head per wave too, on two pieces
    ([(16, 2, 1, 144, 0, 0), (16, 14, 1, 128, 0, 0), (16, 15, 1, 64, 0, 0), (16, 11, 1, 32, 0, 0)], 16, 16, 128, 360),     # nothing longer that would share a CU
    ([(16, 1, 1, 144, 0, 0), (16, 49, 1, 128, 0, 0), (16, 30, 1, 64, 0, 0), (16, 21, 1, 32, 0, 0)], 8, 8, 128, 208),       # 49 x 8 are more than a workgroup per CU
])
def test_few_boxes_of_several_steps_where_a_launch_has_a_workgroup_per_cu(buckets, heads, kv_heads, d, workgroups):
    # ... it does not get more for them beside a longer box
    lib, g = _lib.load(), _lib.FwdGeometry()
    a = _bucket_args(buckets, heads, kv_heads, d, sum(b[1] for b in buckets), 16)
    a.max_split_per_seq = 2 if len(buckets) == 3 else 1
    assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
    assert g.num_workgroups == workgroups, (g.num_workgroups, g.tall_rows)
