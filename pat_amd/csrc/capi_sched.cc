// extern "C" surface of the scheduler (declared in include/pat_amd.h).
#include <algorithm>
#include <array>
#include <climits>
#include <cstdint>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "capi_error.hpp"
#include "pat_amd.h"
#include "sched/radix_plan.hpp"

namespace {
// A flat plan as far as it is laid out before its contents are written: the layout, the boxes' launch order, the launch buckets they
// fall into, and the tables that exist in the launch copies only.
struct FlatPlan {
  struct Part { int parent, lo, hi, width; };   // boxes lo..hi of a bucket's launch order
  pat_flat_plan layout;
  std::vector<std::vector<int32_t>> order;      // per bucket
  std::vector<Part> parts;                      // the launch buckets
  std::vector<std::vector<int32_t>> items;      // per launch bucket: boxes of one node in twos
  std::vector<std::vector<int32_t>> tails;      // per launch bucket, where a bucket holds tails: PAT_BUCKET_TAILS
  std::vector<std::vector<int32_t>> slot;       // per bucket, there too: q_slot with the tails behind all other boxes
  std::vector<int32_t> without;                 // ... and the boxes per sequence that are no tails
};
}  // namespace

struct pat_tree {
  int block_size;
  std::unique_ptr<pat::RadixPlanner> planner;
  std::vector<int32_t> child_scratch;
  // Between the call that asks how large the flat plan is and the one that writes it (half of the two was laying it out again).
  // Both are const calls: whoever uses it takes it away, and a call that finds nothing lays it out itself.
  mutable std::unique_ptr<FlatPlan> flat;
  mutable std::mutex flat_mutex;
};

namespace pat {
thread_local std::string g_last_error;
int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}
}  // namespace pat

namespace {
template <typename F>
int guarded(F&& f) {
  try {
    f();
    return PAT_OK;
  } catch (const pat::SchedError& e) {
    return pat::fail(e.code, e.msg);
  } catch (const std::bad_alloc&) {
    return pat::fail(PAT_ERR_INVALID, "out of host memory");
  } catch (const std::exception& e) {
    return pat::fail(PAT_ERR_INVALID, e.what());
  }
}
}  // namespace

// The planner, for calls that change the tree or its plan.
static pat::RadixPlanner& edit(pat_tree* tree) {
  tree->flat.reset();
  return *tree->planner;
}

extern "C" {

const char* pat_last_error(void) { return pat::g_last_error.c_str(); }
int pat_abi_version(void) { return PAT_ABI_VERSION; }

int pat_tree_create(int32_t block_size, pat_tree** out) {
  if (out == nullptr) return pat::fail(PAT_ERR_INVALID, "pat_tree_create: out is NULL");
  if (block_size <= 0) return pat::fail(PAT_ERR_INVALID, "block_size must be positive");
  return guarded([&] {
    auto* t = new pat_tree;
    t->block_size = block_size;
    t->planner.reset(new pat::RadixPlanner(block_size));
    *out = t;
  });
}

void pat_tree_destroy(pat_tree* tree) { delete tree; }

int pat_tree_build_rows(pat_tree* tree, const int32_t* seq_lens, const int32_t* flat_blocks,
                        const int64_t* row_offsets, int32_t num_seqs) {
  if (tree == nullptr) return pat::fail(PAT_ERR_INVALID, "tree is NULL");
  if (num_seqs < 0) return pat::fail(PAT_ERR_INVALID, "num_seqs must be >= 0");
  if (num_seqs > 0 && (seq_lens == nullptr || row_offsets == nullptr))
    return pat::fail(PAT_ERR_INVALID, "seq_lens / row_offsets is NULL");
  for (int i = 0; i < num_seqs; ++i)
    if (row_offsets[i + 1] < row_offsets[i])
      return pat::fail(PAT_ERR_INVALID, "row_offsets must be non-decreasing");
  if (num_seqs > 0 && row_offsets[num_seqs] > row_offsets[0] && flat_blocks == nullptr)
    return pat::fail(PAT_ERR_INVALID, "flat_blocks is NULL");
  return guarded([&] {
    // A tree is built once per batch; building again starts from an empty tree.
    tree->planner.reset(new pat::RadixPlanner(tree->block_size));
    edit(tree).build(seq_lens, flat_blocks, row_offsets, num_seqs);
  });
}

int pat_tree_build(pat_tree* tree, const int32_t* seq_lens, const int32_t* table,
                   int32_t num_seqs, int32_t max_blocks) {
  if (tree == nullptr) return pat::fail(PAT_ERR_INVALID, "tree is NULL");
  if (num_seqs < 0 || max_blocks < 0)
    return pat::fail(PAT_ERR_INVALID, "num_seqs / max_blocks must be >= 0");
  if (num_seqs > 0 && (seq_lens == nullptr || (table == nullptr && max_blocks > 0)))
    return pat::fail(PAT_ERR_INVALID, "seq_lens / block_table is NULL");
  const int bs = tree->block_size;
  std::vector<int64_t> offsets((size_t)num_seqs + 1, 0);
  std::vector<int32_t> flat;
  for (int i = 0; i < num_seqs; ++i) {
    if (seq_lens[i] < 0) return pat::fail(PAT_ERR_INVALID, "seq_lens must be >= 0");
    const int64_t used = ((int64_t)seq_lens[i] + bs - 1) / bs;
    if (used > max_blocks)
      return pat::fail(PAT_ERR_INVALID, "seq_lens[" + std::to_string(i) + "] needs " +
                                            std::to_string(used) + " blocks but block_table has " +
                                            std::to_string(max_blocks) + " columns");
    const int32_t* row = table + (int64_t)i * max_blocks;
    flat.insert(flat.end(), row, row + used);
    offsets[(size_t)i + 1] = (int64_t)flat.size();
  }
  return pat_tree_build_rows(tree, seq_lens, flat.data(), offsets.data(), num_seqs);
}

int pat_tree_append(pat_tree* tree, int32_t seq_len, const int32_t* blocks, int32_t num_blocks) {
  if (tree == nullptr) return pat::fail(PAT_ERR_INVALID, "tree is NULL");
  if (seq_len < 0 || num_blocks < 0) return pat::fail(PAT_ERR_INVALID, "seq_len / num_blocks must be >= 0");
  if (num_blocks > 0 && blocks == nullptr) return pat::fail(PAT_ERR_INVALID, "blocks is NULL");
  return guarded([&] { edit(tree).append(seq_len, blocks, num_blocks); });
}

int pat_tree_remove(pat_tree* tree, int32_t seq) {
  if (tree == nullptr) return pat::fail(PAT_ERR_INVALID, "tree is NULL");
  return guarded([&] { edit(tree).remove(seq); });
}

int pat_tree_grow(pat_tree* tree, int32_t seq, int32_t new_len, const int32_t* more_blocks, int32_t num_more) {
  if (tree == nullptr) return pat::fail(PAT_ERR_INVALID, "tree is NULL");
  if (num_more > 0 && more_blocks == nullptr) return pat::fail(PAT_ERR_INVALID, "more_blocks is NULL");
  return guarded([&] { edit(tree).grow(seq, new_len, more_blocks, num_more); });
}

int pat_tree_num_seqs(const pat_tree* tree) {
  if (tree == nullptr) return pat::fail(PAT_ERR_INVALID, "tree is NULL");
  return tree->planner->num_seqs();
}

int pat_tree_pack(pat_tree* tree, const int32_t* mnws, int32_t n_mnws, int32_t hratio,
                  int32_t kv_heads, int32_t use_compute_model, const pat_sched_opts* opts) {
  if (tree == nullptr) return pat::fail(PAT_ERR_INVALID, "tree is NULL");
  if (n_mnws > 0 && mnws == nullptr) return pat::fail(PAT_ERR_INVALID, "mnws is NULL");
  return guarded(
      [&] { edit(tree).pack(mnws, n_mnws, hratio, kv_heads, use_compute_model != 0, opts); });
}

int pat_tree_naive_schedule(pat_tree* tree, int32_t hratio) {
  if (tree == nullptr) return pat::fail(PAT_ERR_INVALID, "tree is NULL");
  return guarded([&] { edit(tree).naive(hratio); });
}

int pat_tree_plan(const pat_tree* tree, pat_plan_view* out) {
  if (tree == nullptr || out == nullptr) return pat::fail(PAT_ERR_INVALID, "tree / out is NULL");
  const pat::Plan& p = tree->planner->plan();
  if (!p.valid) return pat::fail(PAT_ERR_INVALID, "no plan: call pat_tree_pack first");
  out->num_buckets = (int32_t)p.views.size();
  out->batch = (int32_t)p.num_split_per_seq.size();
  out->buckets = p.views.data();
  out->num_split_per_seq = p.num_split_per_seq.data();
  out->max_split_per_seq = p.max_split;
  out->max_seqs_in_box = p.max_seqs_in_box;
  out->max_blocks_in_box = p.max_blocks_in_box;
  out->num_boxes_per_seq = p.num_boxes_per_seq.data();
  out->max_boxes_per_seq = p.max_boxes;
  return PAT_OK;
}

// Lays out the flat form of a plan.
static int lay_out(const pat::Plan& p, int page, FlatPlan& f) {
  const int nb = (int)p.buckets.size();
  if (nb > PAT_MAX_FLAT_BUCKETS)
    return pat::fail(PAT_ERR_INVALID, "the flat plan holds at most 12 buckets");
  constexpr int kGrowthBlocks = 8;
  pat_flat_plan* layout = &f.layout;
  std::memset(layout, 0, sizeof(*layout));
  layout->num_buckets = nb;
  layout->batch = (int32_t)p.num_split_per_seq.size();
  layout->max_split_per_seq = p.max_split;
  layout->max_boxes_per_seq = p.max_boxes;
  layout->max_seqs_in_box = p.max_seqs_in_box;
  layout->max_blocks_in_box = p.max_blocks_in_box;

  // launch order and parts of every bucket
  using Part = FlatPlan::Part;
  auto& order = f.order;
  auto& parts = f.parts;
  order.resize((size_t)nb);
  int spare = PAT_MAX_FLAT_BUCKETS - nb;

  // Tails: boxes of one sequence, up to PAT_MAX_TAIL_TOKENS wide, whose sequence also sits in a box of more than 16 rows. A launch may
  // have that box's workgroup walk them too (PAT_BUCKET_TAILS). Of several such boxes the shortest takes the tail.
  struct Claim { int bucket = -1, box = -1, j = 0; };
  std::vector<Claim> claim((size_t)layout->batch);   // per sequence: where its tail may go
  std::vector<std::vector<char>> is_tail((size_t)nb);
  bool any_tail = false;
  auto may_hold_tails = [&](const pat::Bucket& bk) {
    return bk.mnw[0] <= 16 && bk.max_seqs == 1 && (int64_t)bk.max_blocks * page <= PAT_MAX_TAIL_TOKENS;
  };
  const bool look = std::any_of(p.buckets.begin(), p.buckets.end(), may_hold_tails);
  for (int b = 0; b < nb && look; ++b) {
    const pat::Bucket& bk = p.buckets[(size_t)b];
    if (bk.mnw[0] <= 16) continue;
    for (size_t box = 0; box < bk.kv.size(); ++box)
      for (int j = 0; j < bk.q_len[box]; ++j) {
        const int32_t s = bk.q_table[box * (size_t)bk.max_seqs + (size_t)j];
        if (s < 0 || s >= layout->batch) continue;
        Claim& c = claim[(size_t)s];
        if (c.bucket < 0 || bk.kv[box] <= p.buckets[(size_t)c.bucket].kv[(size_t)c.box]) c = {b, (int)box, j};
      }
  }
  {
    std::vector<char> taken((size_t)layout->batch, 0);
    for (int b = 0; b < nb; ++b) {
      const pat::Bucket& bk = p.buckets[(size_t)b];
      is_tail[(size_t)b].assign(bk.kv.size(), 0);
      if (!may_hold_tails(bk)) continue;
      for (size_t box = 0; box < bk.kv.size(); ++box) {
        const int32_t s = bk.q_table[box];
        if (bk.q_len[box] != 1 || s < 0 || s >= layout->batch || claim[(size_t)s].bucket < 0 || taken[(size_t)s]) continue;
        taken[(size_t)s] = is_tail[(size_t)b][box] = 1;
        any_tail = true;
      }
    }
  }

  for (int b = 0; b < nb; ++b) {
    const pat::Bucket& bk = p.buckets[(size_t)b];
    const int n = (int)bk.kv.size();
    auto& ord = order[(size_t)b];
    ord.resize((size_t)n);
    for (int i = 0; i < n; ++i) ord[(size_t)i] = i;
    std::stable_sort(ord.begin(), ord.end(), [&](int32_t x, int32_t y) { return bk.kv[(size_t)x] > bk.kv[(size_t)y]; });
    int cut = 0;
    if (spare > 0 && n >= 4) {
      const int32_t widest = bk.kv[(size_t)ord[0]];
      int k = 0;
      while (k < n && bk.kv[(size_t)ord[(size_t)k]] > widest / 2) ++k;
      if (k > 0 && k <= n / 4) { cut = k; --spare; }
    }
    // a bucket of which only some boxes are tails: those in a launch bucket of their own, behind the others
    const auto& tail = is_tail[(size_t)b];
    const int n_tail = (int)std::count(tail.begin(), tail.end(), 1);
    if (n_tail > 0 && n_tail < n && cut == 0 && spare > 0) {
      std::stable_partition(ord.begin(), ord.end(), [&](int32_t x) { return !tail[(size_t)x]; });
      --spare;
      parts.push_back({b, 0, n - n_tail, bk.max_blocks});
      parts.push_back({b, n - n_tail, n, bk.max_blocks});
    } else if (cut == 0) {
      parts.push_back({b, 0, n, bk.max_blocks});
    } else {
      parts.push_back({b, 0, cut, bk.max_blocks});
      int32_t longest = 1;
      for (int i = cut; i < n; ++i) longest = std::max(longest, bk.block_len[(size_t)ord[(size_t)i]]);
      parts.push_back({b, cut, n, std::min<int32_t>(bk.max_blocks, longest + kGrowthBlocks)});
    }
  }
  layout->num_launch_buckets = (int32_t)parts.size();

  // Boxes of one node (same blocks, different sequences) in twos, for launches that serve two of them with one
  // workgroup. Only buckets of more than 16 rows, and only boxes of several sequences: a box of one sequence may be
  // grown in place between decode steps.
  auto& items = f.items;
  items.resize(parts.size());
  for (size_t i = 0; i < parts.size(); ++i) {
    const Part& pt = parts[i];
    const pat::Bucket& bk = p.buckets[(size_t)pt.parent];
    if (bk.mnw[0] <= 16) continue;
    const auto& ord = order[(size_t)pt.parent];
    std::map<std::array<int32_t, 3>, int32_t> open;   // (first block, last block, tokens) -> item that waits for its second box
    bool any = false;
    for (int at = pt.lo; at < pt.hi; ++at) {
      const size_t box = (size_t)ord[(size_t)at];
      const int32_t len = bk.block_len[box];
      const int32_t* blocks = bk.block_table.data() + box * (size_t)bk.max_blocks;
      if (bk.num_seqs[box] > 1 && len > 0) {
        const std::array<int32_t, 3> key{blocks[0], blocks[len - 1], bk.kv[box]};
        const auto it = open.find(key);
        if (it != open.end()) {
          const size_t first = (size_t)ord[(size_t)(pt.lo + items[i][(size_t)it->second * 2])];
          if (bk.block_len[first] == len &&
              std::memcmp(bk.block_table.data() + first * (size_t)bk.max_blocks, blocks, (size_t)len * sizeof(int32_t)) == 0) {
            items[i][(size_t)it->second * 2 + 1] = at - pt.lo;
            open.erase(it);
            any = true;
            continue;
          }
        }
        open[key] = (int32_t)(items[i].size() / 2);
      }
      items[i].push_back(at - pt.lo);
      items[i].push_back(-1);
    }
    if (!any) items[i].clear();
  }

  // The launch buckets that hold nothing but tails, and per box of more than 16 rows the tails of its sequences there: launch
  // bucket << 27 | row, -1 = none.
  auto& tails = f.tails;
  tails.resize(parts.size());
  if (any_tail) {
    std::vector<char> tail_part(parts.size(), 0);
    auto& slot = f.slot;
    auto& without = f.without;
    any_tail = false;
    std::vector<std::vector<std::array<int32_t, 2>>> place((size_t)nb);   // plan box -> (launch bucket, row)
    for (int b = 0; b < nb; ++b) place[(size_t)b].resize(p.buckets[(size_t)b].kv.size());
    for (size_t i = 0; i < parts.size(); ++i) {
      const Part& pt = parts[i];
      const auto& ord = order[(size_t)pt.parent];
      bool all = pt.hi > pt.lo;
      for (int at = pt.lo; at < pt.hi; ++at) {
        place[(size_t)pt.parent][(size_t)ord[(size_t)at]] = {(int32_t)i, at - pt.lo};
        all = all && is_tail[(size_t)pt.parent][(size_t)ord[(size_t)at]];
      }
      tail_part[i] = all;
      any_tail = any_tail || all;
    }
    if (any_tail) {
      for (size_t i = 0; i < parts.size(); ++i) {
        if (!tail_part[i]) continue;
        const Part& pt = parts[i];
        const pat::Bucket& bk = p.buckets[(size_t)pt.parent];
        for (int at = pt.lo; at < pt.hi; ++at) {
          const Claim& c = claim[(size_t)bk.q_table[(size_t)order[(size_t)pt.parent][(size_t)at]]];
          const auto& where = place[(size_t)c.bucket][(size_t)c.box];
          const pat::Bucket& tall = p.buckets[(size_t)c.bucket];
          auto& t = tails[(size_t)where[0]];
          if (t.empty()) t.assign((size_t)(parts[(size_t)where[0]].hi - parts[(size_t)where[0]].lo) * (size_t)tall.max_seqs, -1);
          t[(size_t)where[1] * (size_t)tall.max_seqs + (size_t)c.j] = (int32_t)i << 27 | (at - pt.lo);
        }
      }
      // ordinals of a sequence's boxes with the tails behind all others: a launch that has no slots for tails leaves the last ones out
      std::vector<int32_t> seen((size_t)layout->batch, 0);
      slot.resize((size_t)nb);
      for (int b = 0; b < nb; ++b) slot[(size_t)b].assign(p.buckets[(size_t)b].q_slot.size(), 0);
      for (int pass = 0; pass < 2; ++pass) {
        for (int b = 0; b < nb; ++b) {
          const pat::Bucket& bk = p.buckets[(size_t)b];
          for (size_t box = 0; box < bk.kv.size(); ++box) {
            if ((int)tail_part[(size_t)place[(size_t)b][box][0]] != pass) continue;
            for (int j = 0; j < bk.q_len[box]; ++j) {
              const size_t e = box * (size_t)bk.max_seqs + (size_t)j;
              slot[(size_t)b][e] = seen.at((size_t)bk.q_table[e])++;
            }
          }
        }
        if (pass == 0) without = seen;
      }
      uint32_t word = (uint32_t)*std::max_element(without.begin(), without.end());
      for (size_t i = 0; i < parts.size(); ++i) word |= (tail_part[i] ? 1u << (8 + i) : 0u) | (!tails[i].empty() ? 1u << (20 + i) : 0u);
      layout->tails = (int32_t)word;
    }
  }

  // offsets
  int64_t at = 0;
  auto take = [&](int64_t n) { const int64_t o = at; at += n; return o; };
  layout->num_split_per_seq = take(layout->batch);
  layout->num_boxes_per_seq = take(layout->batch);
  auto place = [&](pat_flat_bucket& f, const pat::Bucket& bk, int rows, int width, int parent, int first) {
    std::memcpy(f.mnw, bk.mnw, sizeof(f.mnw));
    f.num_boxes = rows; f.max_seqs = bk.max_seqs; f.max_blocks = width; f.parent = parent; f.first = first;
    f.flags = 0;
    f.q_table = take((int64_t)rows * bk.max_seqs);
    f.q_slot = take((int64_t)rows * bk.max_seqs);
    f.block_table = take((int64_t)rows * width);
    f.num_seqs = take(rows); f.rank = take(rows); f.kv = take(rows);
  };
  for (int b = 0; b < nb; ++b) {
    const pat::Bucket& bk = p.buckets[(size_t)b];
    place(layout->buckets[b], bk, (int)bk.kv.size(), bk.max_blocks, b, 0);
    layout->launch_order[b] = take((int64_t)bk.kv.size());
  }
  for (size_t i = 0; i < parts.size(); ++i) {
    const Part& pt = parts[i];
    place(layout->launch[i], p.buckets[(size_t)pt.parent], pt.hi - pt.lo, pt.width, pt.parent, pt.lo);
    layout->launch[i].num_items = (int32_t)(items[i].size() / 2);
    take((int64_t)items[i].size());   // (right behind kv, the last table of the bucket)
    if (!tails[i].empty()) take((int64_t)tails[i].size() + layout->batch);
  }
  // hints: a bucket is even when no box is shorter than 3/4 of its widest one
  auto even = [&](const pat::Bucket& bk, const int32_t* ord, int lo, int hi) {
    int32_t widest = 0, shortest = INT32_MAX;
    for (int i = lo; i < hi; ++i) {
      const int32_t t = bk.kv[(size_t)(ord ? ord[i] : i)];
      widest = std::max(widest, t); shortest = std::min(shortest, t);
    }
    return hi > lo && (int64_t)shortest * 4 >= (int64_t)widest * 3 ? PAT_BUCKET_EVEN : 0;
  };
  const int unboxed = std::find(p.num_boxes_per_seq.begin(), p.num_boxes_per_seq.end(), 0) != p.num_boxes_per_seq.end() ? PAT_BUCKET_UNBOXED : 0;
  for (int b = 0; b < nb; ++b)
    layout->buckets[b].flags = even(p.buckets[(size_t)b], nullptr, 0, (int)p.buckets[(size_t)b].kv.size());
  for (size_t i = 0; i < parts.size(); ++i)
    layout->launch[i].flags = even(p.buckets[(size_t)parts[i].parent], order[(size_t)parts[i].parent].data(), parts[i].lo, parts[i].hi) | unboxed;
  layout->total = at;
  return PAT_OK;
}

static int flat_plan_impl(const pat_tree* tree, pat_flat_plan* layout, int32_t* dst, int64_t capacity) {
  if (tree == nullptr || layout == nullptr) return pat::fail(PAT_ERR_INVALID, "tree / layout is NULL");
  const pat::Plan& p = tree->planner->plan();
  if (!p.valid) return pat::fail(PAT_ERR_INVALID, "no plan: call pat_tree_pack first");
  std::unique_ptr<FlatPlan> f;
  {
    const std::lock_guard<std::mutex> lock(tree->flat_mutex);
    f = std::move(tree->flat);
  }
  if (!f) {
    f = std::make_unique<FlatPlan>();
    if (int rc = lay_out(p, tree->block_size, *f)) return rc;
  }
  *layout = f->layout;
  if (dst == nullptr || capacity < layout->total) {
    const std::lock_guard<std::mutex> lock(tree->flat_mutex);
    tree->flat = std::move(f);
    return dst == nullptr ? PAT_OK : pat::fail(PAT_ERR_INVALID, "flat plan: buffer too small");
  }
  const auto& order = f->order;

  // contents
  std::copy(p.num_split_per_seq.begin(), p.num_split_per_seq.end(), dst + layout->num_split_per_seq);
  std::copy(p.num_boxes_per_seq.begin(), p.num_boxes_per_seq.end(), dst + layout->num_boxes_per_seq);
  auto rows_to = [&](int32_t* out, const std::vector<int32_t>& table, int src_width, int width,
                     const int32_t* ord, int lo, int hi) {
    for (int i = lo; i < hi; ++i) {
      const int32_t* row = table.data() + (size_t)(ord ? ord[i] : i) * (size_t)src_width;
      std::copy(row, row + width, out + (size_t)(i - lo) * (size_t)width);
    }
  };
  auto vec_to = [&](int32_t* out, const std::vector<int32_t>& v, const int32_t* ord, int lo, int hi) {
    for (int i = lo; i < hi; ++i) out[i - lo] = v[(size_t)(ord ? ord[i] : i)];
  };
  auto fill = [&](const pat_flat_bucket& to, const pat::Bucket& bk, const std::vector<int32_t>& q_slot, const int32_t* ord, int lo, int hi) {
    rows_to(dst + to.q_table, bk.q_table, bk.max_seqs, bk.max_seqs, ord, lo, hi);
    rows_to(dst + to.q_slot, q_slot, bk.max_seqs, bk.max_seqs, ord, lo, hi);
    rows_to(dst + to.block_table, bk.block_table, bk.max_blocks, to.max_blocks, ord, lo, hi);
    vec_to(dst + to.num_seqs, bk.num_seqs, ord, lo, hi);
    vec_to(dst + to.rank, bk.rank, ord, lo, hi);
    vec_to(dst + to.kv, bk.kv, ord, lo, hi);
  };
  for (int b = 0; b < layout->num_buckets; ++b) {
    const pat::Bucket& bk = p.buckets[(size_t)b];
    fill(layout->buckets[b], bk, bk.q_slot, nullptr, 0, (int)bk.kv.size());
    std::copy(order[(size_t)b].begin(), order[(size_t)b].end(), dst + layout->launch_order[b]);
  }
  for (size_t i = 0; i < f->parts.size(); ++i) {
    const FlatPlan::Part& pt = f->parts[i];
    const pat::Bucket& bk = p.buckets[(size_t)pt.parent];
    fill(layout->launch[i], bk, layout->tails != 0 ? f->slot[(size_t)pt.parent] : bk.q_slot, order[(size_t)pt.parent].data(), pt.lo, pt.hi);
    int32_t* behind = std::copy(f->items[i].begin(), f->items[i].end(), dst + layout->launch[i].kv + layout->launch[i].num_boxes);
    if (!f->tails[i].empty())
      std::copy(f->without.begin(), f->without.end(), std::copy(f->tails[i].begin(), f->tails[i].end(), behind));
  }
  return PAT_OK;
}

int pat_tree_flat_plan(const pat_tree* tree, pat_flat_plan* layout, int32_t* dst, int64_t capacity) {
  int rc = PAT_OK;
  const int thrown = guarded([&] { rc = flat_plan_impl(tree, layout, dst, capacity); });
  return thrown ? thrown : rc;
}

int pat_tree_num_nodes(const pat_tree* tree) {
  if (tree == nullptr) return pat::fail(PAT_ERR_INVALID, "tree is NULL");
  return (int)tree->planner->nodes().size();
}

int pat_tree_node(const pat_tree* tree, int32_t node, pat_node_view* out) {
  if (tree == nullptr || out == nullptr) return pat::fail(PAT_ERR_INVALID, "tree / out is NULL");
  const auto& nodes = tree->planner->nodes();
  if (node < 0 || (size_t)node >= nodes.size())
    return pat::fail(PAT_ERR_INDEX, "node index out of range");
  const pat::RadixNode& n = nodes[(size_t)node];
  out->parent = n.parent;
  out->num_seqs = n.num_seqs;
  out->num_tokens = n.num_tokens;
  out->num_seq_ids = (int32_t)n.seq_ids.size();
  out->num_blocks = (int32_t)n.blocks.size();
  out->num_children = (int32_t)n.child_ids.size();
  out->seq_ids = n.seq_ids.data();
  out->block_ids = n.blocks.data();
  out->child_ids = n.child_ids.data();
  return PAT_OK;
}

}  // extern "C"
