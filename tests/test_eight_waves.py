"""Single-slot launches of few workgroups run eight waves per workgroup: when they do, and the results at the edges of the waves' steps."""
import ctypes as C
import math

import pytest
import torch

from oracle import attn_oracle as ao
from pat_amd import PrefixTreeCPP, _lib, prefix_attn_with_kvcache, workloads


def _args(requests, tokens, heads, kv_heads, d, page=16):
    b = (_lib.FwdBucket * 1)()
    b[0].q_table = b[0].block_table = b[0].num_seqs = b[0].rank = b[0].kv = 0x10000
    b[0].mnw[:] = [16, 128, 1]
    b[0].num_boxes, b[0].max_seqs, b[0].max_blocks = requests, 1, tokens // page
    b[0].q_table_stride, b[0].block_table_stride = 1, tokens // page
    a = _lib.FwdArgs()
    a.dtype, a.batch, a.seqlen_q, a.heads, a.kv_heads = _lib.PAT_DTYPE_F16, requests, 1, heads, kv_heads
    a.head_dim, a.page_size, a.num_pages = d, page, 1 << 16
    a.q = a.k = a.v = a.out = a.num_split_per_seq = 0x10000
    a.q_stride = a.o_stride = (C.c_int64 * 3)(heads * d, heads * d, d)
    a.k_stride = a.v_stride = (C.c_int64 * 3)(page * kv_heads * d, kv_heads * d, d)
    a.max_split_per_seq, a.max_seqs_in_box, a.max_blocks_in_box, a.softmax_scale = 1, 1, tokens // page, 0.1
    a.num_buckets, a.buckets = 1, C.cast(b, C.POINTER(_lib.FwdBucket))
    a._keep = b
    return a


@pytest.mark.parametrize("requests,tokens,heads,d,eight", [
    (8, 288, (8, 8), 64, True), (8, 256, (8, 8), 64, False),          # more than eight steps
    (20, 384, (8, 8), 64, True), (21, 384, (8, 8), 64, False),        # 160 workgroups at most ...
    (20, 384, (8, 8), 128, True), (20, 400, (8, 8), 128, False),      # ... at head_dim 128 for boxes of up to twelve steps,
    (8, 512, (8, 8), 128, True), (9, 512, (8, 8), 128, False),        # 64 for longer ones
    (8, 528, (8, 8), 64, False),                                      # cut into pieces: a merge follows
])
def test_launch_rule(requests, tokens, heads, d, eight, tuning):
    lib, g = _lib.load(), _lib.FwdGeometry()
    for switch, want in ((0, eight), (_lib.PAT_WAVES_4, False), (_lib.PAT_WAVES_8, tokens <= 512)):
        tuning(pairs=switch)
        assert lib.pat_fwd_geometry_of(C.byref(_args(requests, tokens, *heads, d)), C.byref(g)) == 0, _lib.last_error()
        assert bool(g.flags & _lib.PAT_GEOMETRY_WAVES_8) == want, switch


@pytest.mark.gpu
@pytest.mark.parametrize("heads,d,dtype,page", [((8, 8), 64, torch.float16, 16), ((16, 2), 128, torch.bfloat16, 48),
                                                ((32, 8), 128, torch.float16, 32), ((16, 8), 64, torch.bfloat16, 64)])
def test_against_the_oracle(heads, d, dtype, page, tuning, monkeypatch):
    print(f"[case] eight waves, heads {heads}, d {d}, {dtype}, page {page}", flush=True)
    monkeypatch.setenv("PAT_WHOLE_SEQUENCES", "1")
    dev = torch.device("cuda:0")
    # waves without a step, a last step of one token, one and two steps per wave and one token more
    lens = [n for n in (1, 31, 33, 224, 255, 256, 257, 288, 480, 511, 512) if -(-n // page) * page <= 512]
    rows, nxt = [], 0
    for n in lens:
        rows.append(list(range(nxt, nxt + -(-n // page))))
        nxt += -(-n // page)
    w = workloads.Workload("eight", heads[0], heads[1], d, dtype, page, lens, rows, nxt, 0, 2)
    q, k, v = w.tensors(dev)
    ref_out, ref_lse = ao.paged_attention_ref(q.cpu(), k.cpu(), v.cpu(), rows, lens)
    for switch in (_lib.PAT_WAVES_8, _lib.PAT_WAVES_4):
        tuning(pairs=switch)
        tree = PrefixTreeCPP(page)
        tree.build_radix_tree(lens, w.padded_table())
        tree.pack_schedule(None, heads[0] // heads[1], heads[1])
        tree.kernel_info.to_gpu(dev)
        out = torch.full_like(q, float("nan"))
        lse = torch.full((w.batch, w.heads), float("nan"), dtype=torch.float32, device=dev)
        prefix_attn_with_kvcache(q, k, v, tree, 1.0 / math.sqrt(d), out, softmax_lse=lse)
        torch.cuda.synchronize()
        assert [g["waves"] for g in tree.kernel_info._launch_geometries] == [8 if switch == _lib.PAT_WAVES_8 else 4]
        err = (out.float().cpu() - ref_out.float()).abs().max().item()
        lerr = ((lse.cpu() - ref_lse).abs() / ref_lse.abs().clamp_min(1.0)).max().item()
        print(f"[parity] {err:.3e} {lerr:.3e}", flush=True)
        assert err <= (2e-3 if dtype == torch.float16 else 1.6e-2) and lerr <= 1e-4


@pytest.mark.parametrize("requests,tokens,heads,d,want", [
    (8, 2240, (64, 8), 128, (8, 192, 3)),     # 384 workgroups of 384 tokens: 192 of 768
    (16, 512, (16, 16), 128, None),           # (whole: nothing to merge)
    (12, 768, (16, 16), 128, (8, 192, 1)),    # two pieces become one
    (4, 1152, (8, 8), 128, None), (4, 1280, (8, 8), 128, (8, 160, 5)),    # 288 workgroups are too few, 320 not
    (5, 1280, (8, 8), 128, (8, 200, 5)), (8, 832, (8, 8), 128, None),     # 400 still, 448 not
    (12, 2048, (64, 8), 128, None),           # 288 would be left
    (8, 2240, (64, 8), 64, None),             # head_dim 64
])
def test_double_pieces_rule(requests, tokens, heads, d, want, tuning):
    lib, g, a = _lib.load(), _lib.FwdGeometry(), _args(requests, tokens, *heads, d)
    tuning(pairs=_lib.PAT_WAVES_4)
    assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0 and not g.flags & _lib.PAT_GEOMETRY_WAVES_8
    four = (4, g.num_workgroups, g.num_slots)
    tuning()
    assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
    assert (8 if g.flags & _lib.PAT_GEOMETRY_WAVES_8 else 4, g.num_workgroups, g.num_slots) == (want or four)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,heads,dtype,page,direct", [
    ([2239, 1, 767, 768, 769, 2240, 1537, 800], (64, 8), torch.float16, 16, False),        # pieces unfilled, of one token and full
    ([1280, 1249, 33, 1025], (8, 8), torch.bfloat16, 16, False),
    ([1000, 1279, 257, 31, 256], (16, 8), torch.float16, 32, False),
    ([767, 768, 1, 33, 736, 500, 255, 256, 384, 385, 640, 700], (16, 16), torch.bfloat16, 48, True),    # one piece: straight to `out`
])
def test_double_pieces_against_the_oracle(lens, heads, dtype, page, direct, tuning, monkeypatch):
    print(f"[case] double pieces, {lens}, heads {heads}, {dtype}, page {page}", flush=True)
    monkeypatch.setenv("PAT_WHOLE_SEQUENCES", "1")
    rows, nxt = [], 0
    for n in lens:
        rows.append(list(range(nxt, nxt + -(-n // page))))
        nxt += -(-n // page)
    w = workloads.Workload("double", heads[0], heads[1], 128, dtype, page, lens, rows, nxt, 0, 4)
    q, k, v = w.tensors(torch.device("cuda:0"))
    ref_out, ref_lse = ao.paged_attention_ref(q.cpu(), k.cpu(), v.cpu(), rows, lens)
    for switch in (0, _lib.PAT_WAVES_4):
        tuning(pairs=switch)
        tree = PrefixTreeCPP(page)
        tree.build_radix_tree(lens, w.padded_table())
        tree.pack_schedule(None, heads[0] // heads[1], heads[1])
        tree.kernel_info.to_gpu(q.device)
        out = torch.full_like(q, float("nan"))
        lse = torch.full((w.batch, w.heads), float("nan"), dtype=torch.float32, device=q.device)
        for _ in range(2):    # (the second call finds the first one's partial rows in the workspace)
            prefix_attn_with_kvcache(q, k, v, tree, 1.0 / math.sqrt(128), out, softmax_lse=lse)
        torch.cuda.synchronize()
        assert [(g["waves"], g["num_slots"] == 1) for g in tree.kernel_info._launch_geometries] == [(8, direct) if switch == 0 else (4, False)]
        err = (out.float().cpu() - ref_out.float()).abs().max().item()
        lerr = ((lse.cpu() - ref_lse).abs() / ref_lse.abs().clamp_min(1.0)).max().item()
        print(f"[parity] {err:.3e} {lerr:.3e}", flush=True)
        assert err <= (2e-3 if dtype == torch.float16 else 1.6e-2) and lerr <= 1e-4


def test_the_launcher_refuses_what_it_has_no_instance_for(tmp_path):
    # asked of the launcher itself, which answers before anything touches a GPU: combinations that no launch rule makes
    import os
    import shutil
    import subprocess
    _lib.load()
    here = os.path.dirname(os.path.abspath(_lib.__file__))
    src, so = tmp_path / "probe.cc", tmp_path / "probe.so"
    src.write_text("""
#include "hip/fwd_params.hpp"
#include <cstring>
struct ihipStream_t;
namespace pat { int launch_split(bool bf16, int head_dim, ihipStream_t* stream, const SplitParams& params); }
extern "C" int probe(int head_dim, int direct, int waves, int rows, int lists, int tail_pages, int stream_v) {
  pat::SplitParams p;
  std::memset(&p, 0, sizeof(p));
  p.direct = direct; p.waves = waves; p.tall_rows = rows; p.list_boxes = lists; p.tail_pages = tail_pages; p.stream_v = stream_v;
  return pat::launch_split(false, head_dim, nullptr, p);
}
""")
    subprocess.run([shutil.which("g++") or "c++", "-std=c++17", "-shared", "-fPIC", f"-I{here}/csrc", f"-I{os.path.dirname(here)}/include", str(src), "-o", str(so),
                    f"-L{here}", "-lpat_amd", f"-Wl,-rpath,{here}", "-Wl,--allow-shlib-undefined"], check=True)
    probe = C.CDLL(str(so)).probe
    for case in [(64, 0, 8, 16, 0, 0, 0),                                                                  # eight waves and partial rows at head_dim 64
                 (128, 1, 8, 16, 0, 0, 1), (128, 0, 8, 32, 0, 2, 0), (128, 0, 8, 32, 4, 0, 0), (128, 1, 5, 16, 0, 0, 0),
                 (64, 0, 4, 32, 4, 0, 0), (128, 0, 4, 16, 4, 0, 0), (128, 1, 4, 32, 4, 0, 0),              # lists: head_dim 128, 32-row form, partial rows
                 (128, 0, 4, 32, 4, 2, 0), (128, 0, 4, 32, 4, 0, 1),
                 (128, 1, 4, 16, 0, 2, 0), (128, 1, 4, 32, 0, 2, 1)]:                                      # tails: 32-row form, V through the caches
        assert probe(*case) == 1, case                                                                     # hipErrorInvalidValue


def test_double_pieces_are_for_requests_of_one_box(tuning):
    # requests that sit in several boxes are merged all the same, and longer pieces lose there
    lib, g = _lib.load(), _lib.FwdGeometry()
    for most, eight in ((1, True), (2, False), (3, False)):
        a = _args(8, 2240, 64, 8, 128)
        a.max_split_per_seq = most
        tuning()
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0, _lib.last_error()
        assert bool(g.flags & _lib.PAT_GEOMETRY_WAVES_8) is eight
        got = (g.num_workgroups, g.num_slots)
        tuning(pairs=_lib.PAT_WAVES_4)
        assert lib.pat_fwd_geometry_of(C.byref(a), C.byref(g)) == 0
        assert (got == (g.num_workgroups, g.num_slots)) is not eight
