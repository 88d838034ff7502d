// Merge kernel for gfx950: combines the partial outputs of one (sequence, query head)
// into the final attention row.
//
// Contract (the reference's gather_kernel, csrc/pat_fwd_kernel.h:314-467): with
// partial results (O_i, LSE_i), LSE = M + ln(sum_i e^(LSE_i - M)), M = max_i LSE_i and
// out = sum_i e^(LSE_i - LSE) * O_i, cast to the output type; the final LSE is natural
// log of the scaled-logit sum.
//
// One wave64 per (sequence, head). The row's slot LSEs are read once, up to 4 per lane,
// and stay in registers (slots no workgroup filled hold -inf and get weight 0); then each
// lane accumulates head_dim/64 columns over the filled slots, whose rows are fetched in
// batches of 16 independent loads. That is a chain of three memory round trips (split count,
// LSEs, partial rows), which is what the kernel's run time consists of; launches with up to 8
// slots per row make it one: slot addresses do not depend on the split count, so everything is
// requested at once and what turns out unused is dropped (measured: 0.3-0.8 us less per launch;
// with 16 rows requested blindly the extra registers and reads cost what the round trips save).
// Two more forms stand below: a half-wave per row where rows are many and slots few, a workgroup per row where
// slots are many (9 and more) and rows few. In all of them a slot is empty where its LSE is -inf, and nowhere else: a NaN (from
// a NaN in Q or K, or an infinite score) is a filled slot, and makes the row NaN as it makes one that is not cut up.
#include <hip/hip_runtime.h>

#include "fwd_params.hpp"

namespace pat {

// u / d with m = ceil(2^32 / d) (0 for d = 1), any 32-bit u: the product is the quotient or one more.
__device__ __forceinline__ unsigned divide(unsigned u, unsigned d, unsigned m) {
  if (m == 0) return u;
  const unsigned q = __umulhi(u, m);
  return q * d > u ? q - 1 : q;
}

// Which (sequence, head) is row u of workgroup list `xcd`? Workgroups are dealt to the 8 XCDs round-robin, and the
// split kernel's launch order put every partial row of kv head h through the L2 of XCD h mod 8
// (where most of it still sits): with a multiple of 8 kv heads, workgroup b serves heads of the kv
// heads = b mod 8, so the rows are found in its own L2. A matter of speed only. Otherwise there is one list.
// (32-bit arithmetic with a multiplier from the host: batch x heads x slots is below 2^31, and a 64-bit division
// by an argument is 150 instructions ahead of the first load)
__device__ __forceinline__ void row_of(unsigned u, unsigned xcd, int per_list, unsigned per_list_magic, int mapping, int& s, int& hq) {
  s = (int)divide(u, (unsigned)per_list, per_list_magic);
  const int local = (int)u - s * per_list;
  const int group = mapping & 255;
  if (mapping & 256) {
    const int gshift = 31 - __builtin_clz(group);            // group: 1, 2, 4 or 8
    hq = (((int)xcd + 8 * (local >> gshift)) << gshift) + (local & (group - 1));   // kv head (xcd + 8 i), head g of its group
  } else {
    hq = local;
  }
}

// The leading arguments of the kernels, all that stands ahead of their first memory reads: 14 dwords, preloaded into
// SGPRs with the wave; the rest of `p` arrives by load meanwhile.
//   rows_per_list   rows a list holds; per_list: those of one sequence, with its multiplier (0 for 1)
//   mapping         query heads per kv head, + 256 where there are eight lists, one per XCD
#define MERGE_ROWS                                                                                                      \
  const int32_t* __restrict__ num_split_per_seq, const float* __restrict__ lse_part, const float* __restrict__ o_part, \
      const int num_slots, const int chunks_per_rank, const int max_split, const int heads, const int rows_per_list,   \
      const int per_list, const unsigned per_list_magic, const int mapping
template <typename T, int D>
__global__ void __launch_bounds__(256) pat_merge_kernel(MERGE_ROWS, const MergeParams p) {
  constexpr int CPL = D / 64;   // columns per lane
  constexpr int kRegs = 4;      // LSE registers per lane: up to 256 slots stay in registers
  constexpr int kBatch = 16;    // partial rows fetched together
  constexpr int kSpec = 8;      // launches with up to this many slots per row fetch every slot's row at once
  const int lane = threadIdx.x & 63;
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned u = (mapping & 256 ? blockIdx.x >> 3 : blockIdx.x) * 4 + wave;
  if (u >= (unsigned)rows_per_list) return;
  int s, hq;
  row_of(u, blockIdx.x & 7, per_list, per_list_magic, mapping, s, hq);
  const int64_t pair = (int64_t)s * heads + hq;
  const float ninf = -__builtin_inff();

  const float* __restrict__ lse = lse_part + pair * num_slots;
  const float* __restrict__ op = o_part + pair * (int64_t)num_slots * D;
  if (num_slots <= kSpec) {
    // Few slots: nothing here depends on the split count but which slots count, so the count, the
    // slot LSEs and every slot's row are requested together (one round trip instead of three);
    // rows of slots that turn out empty or beyond the count are dropped unread.
    int ns = num_split_per_seq[s];
    float l = (lane < num_slots) ? lse[lane] : ninf;
    float v[kSpec][CPL];
#pragma unroll
    for (int b = 0; b < kSpec; ++b) {
      if (b < num_slots) {
        const float* row = op + (int64_t)b * D + lane * CPL;
        if (CPL == 2) {
          const float2 t = *(const float2*)row;
          v[b][0] = t.x;
          v[b][CPL - 1] = t.y;
        } else {
          v[b][0] = row[0];
        }
      }
    }
    ns = ns < 0 ? 0 : (ns > max_split ? max_split : ns);
    const int nsl = ns * chunks_per_rank;
    if (lane >= nsl) l = ninf;
    float mx = l;
#pragma unroll
    for (int off = kSpec / 2; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    mx = __shfl(mx, 0);
    float e = (l != ninf) ? __expf(l - mx) : 0.f;
    float sum = e;
#pragma unroll
    for (int off = kSpec / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
    sum = __shfl(sum, 0);
    const float total = (sum != 0.f) ? mx + logf(sum) : ninf;
    const float w_mine = (l != ninf) ? __expf(l - total) : 0.f;
    float acc[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) acc[c] = 0.f;
#pragma unroll
    for (int b = 0; b < kSpec; ++b) {
      const float w = __shfl(w_mine, b);
      if (b < num_slots && w != 0.f) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) acc[c] += w * v[b][c];
      }
    }
    T* dst = (T*)p.out + (int64_t)s * p.o_stride_b + (int64_t)hq * p.o_stride_h + lane * CPL;
#pragma unroll
    for (int c = 0; c < CPL; ++c) dst[c] = (T)acc[c];
    if (p.lse_out != nullptr && lane == 0) p.lse_out[pair] = total;
    return;
  }
  int nsplit = num_split_per_seq[s];
  nsplit = nsplit < 0 ? 0 : (nsplit > max_split ? max_split : nsplit);
  const int nslots = nsplit * chunks_per_rank;  // slots are box-major

  // slot LSEs -> registers (slots past 256 are re-read below; no plan of the default buckets
  // gets there: 32 splits x 64 chunks would)
  float mine[kRegs];
  float mx = ninf;
#pragma unroll
  for (int r = 0; r < kRegs; ++r) {
    const int i = r * 64 + lane;
    mine[r] = (i < nslots) ? lse[i] : ninf;
    mx = fmaxf(mx, mine[r]);
  }
  for (int i = kRegs * 64 + lane; i < nslots; i += 64) mx = fmaxf(mx, lse[i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
  float sum = 0.f;
#pragma unroll
  for (int r = 0; r < kRegs; ++r) sum += (mine[r] != ninf) ? __expf(mine[r] - mx) : 0.f;
  for (int i = kRegs * 64 + lane; i < nslots; i += 64) { const float l = lse[i]; sum += (l != ninf) ? __expf(l - mx) : 0.f; }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  const float total = (sum != 0.f) ? mx + logf(sum) : ninf;

  float acc[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) acc[c] = 0.f;

  // weighted sum of the filled slots of one 64-slot group
  auto accumulate = [&](int base, float w_mine) {
    unsigned long long live = __ballot(w_mine != 0.f);
    while (live) {
      int js[kBatch];
      float v[kBatch][CPL];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        js[b] = live ? __builtin_ctzll(live) : -1;
        live &= live - 1;   // 0 stays 0
      }
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        if (js[b] >= 0) {
          const float* row = op + (int64_t)(base + js[b]) * D + lane * CPL;
          if (CPL == 2) {
            const float2 t = *(const float2*)row;
            v[b][0] = t.x;
            v[b][CPL - 1] = t.y;
          } else {
            v[b][0] = row[0];
          }
        }
      }
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        if (js[b] >= 0) {
          const float w = __shfl(w_mine, js[b]);
#pragma unroll
          for (int c = 0; c < CPL; ++c) acc[c] += w * v[b][c];
        }
      }
    }
  };
#pragma unroll
  for (int r = 0; r < kRegs; ++r) {
    if (r * 64 >= nslots) break;
    accumulate(r * 64, (mine[r] != ninf) ? __expf(mine[r] - total) : 0.f);
  }
  for (int base = kRegs * 64; base < nslots; base += 64) {
    const int i = base + lane;
    const float l = (i < nslots) ? lse[i] : ninf;
    accumulate(base, (l != ninf) ? __expf(l - total) : 0.f);
  }

  T* dst = (T*)p.out + (int64_t)s * p.o_stride_b + (int64_t)hq * p.o_stride_h + lane * CPL;
#pragma unroll
  for (int c = 0; c < CPL; ++c) dst[c] = (T)acc[c];
  if (p.lse_out != nullptr && lane == 0) p.lse_out[pair] = total;
}

// Launches with up to 8 slots per row and many rows (tens of thousands: hundreds of requests x
// 32-64 heads) are bound by the number of waves, each of which lives for one round trip: there a
// half-wave takes a (sequence, head), 16 bytes of a partial row per lane, which halves the waves and
// the load instructions per byte. Same arithmetic in the same order as the kernel above.
template <typename T, int D>
__global__ void __launch_bounds__(256) pat_merge_pairs_kernel(MERGE_ROWS, const MergeParams p) {
  constexpr int CPL = D / 32;   // columns per lane
  constexpr int kSpec = 8;
  const int lane = threadIdx.x & 63;
  const int half = lane >> 5, l32 = lane & 31;
  const int slot_in_wg = (int)(threadIdx.x >> 6) * 2 + half;   // 8 rows per workgroup
  unsigned u = (mapping & 256 ? blockIdx.x >> 3 : blockIdx.x) * 8 + slot_in_wg;
  const bool live = u < (unsigned)rows_per_list;
  if (!live) u = (unsigned)rows_per_list - 1;   // (an idle half repeats the last row's reads and stores nothing)
  int s, hq;
  row_of(u, blockIdx.x & 7, per_list, per_list_magic, mapping, s, hq);
  const int64_t pair = (int64_t)s * heads + hq;
  const float ninf = -__builtin_inff();
  const float* __restrict__ lse = lse_part + pair * num_slots;
  const float* __restrict__ op = o_part + pair * (int64_t)num_slots * D;
  int ns = num_split_per_seq[s];
  float l = (l32 < num_slots) ? lse[l32] : ninf;
  float v[kSpec][CPL];
#pragma unroll
  for (int b = 0; b < kSpec; ++b) {
    if (b < num_slots) {
      const float* row = op + (int64_t)b * D + l32 * CPL;
      if (CPL == 4) {
        const float4 t = *(const float4*)row;
        v[b][0] = t.x; v[b][1] = t.y; v[b][CPL - 2] = t.z; v[b][CPL - 1] = t.w;
      } else {
        const float2 t = *(const float2*)row;
        v[b][0] = t.x; v[b][CPL - 1] = t.y;
      }
    }
  }
  ns = ns < 0 ? 0 : (ns > max_split ? max_split : ns);
  const int nsl = ns * chunks_per_rank;
  if (l32 >= nsl) l = ninf;
  float mx = l;
#pragma unroll
  for (int off = kSpec / 2; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
  mx = __shfl(mx, half * 32);
  float e = (l != ninf) ? __expf(l - mx) : 0.f;
  float sum = e;
#pragma unroll
  for (int off = kSpec / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  sum = __shfl(sum, half * 32);
  const float total = (sum != 0.f) ? mx + logf(sum) : ninf;
  const float w_mine = (l != ninf) ? __expf(l - total) : 0.f;
  float acc[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) acc[c] = 0.f;
#pragma unroll
  for (int b = 0; b < kSpec; ++b) {
    const float w = __shfl(w_mine, half * 32 + b);
    if (b < num_slots && w != 0.f) {
#pragma unroll
      for (int c = 0; c < CPL; ++c) acc[c] += w * v[b][c];
    }
  }
  if (!live) return;
  T* dst = (T*)p.out + (int64_t)s * p.o_stride_b + (int64_t)hq * p.o_stride_h + l32 * CPL;
#pragma unroll
  for (int c = 0; c < CPL; ++c) dst[c] = (T)acc[c];
  if (p.lse_out != nullptr && l32 == 0) p.lse_out[pair] = total;
}

// Launches of 9 slots per row and more and few rows (a long request cut over the whole chip, a deep tree of a few dozen
// requests): a workgroup takes a (sequence, head), each of its WAVES waves every WAVES-th slot; the waves' sums are combined
// through LDS.
//  * SPEC: up to 8 slots per wave, whose LSEs and rows it requests at once like the kernels above: one round trip where the
//    general kernel's chain is split count -> LSEs -> rows by sixteens, and WAVES times the waves where rows are few. Empty
//    slots are requested too.
//  * otherwise the LSEs first, then the rows of the filled slots, eight at a time: two round trips, and nothing read for
//    empty slots, which most are where a launch reserves many (a slot per piece of the longest box for every box).
template <typename T, int D, int WAVES, bool SPEC>
__global__ void __launch_bounds__(WAVES * 64) pat_merge_wide_kernel(MERGE_ROWS, const MergeParams p) {
  constexpr int CPL = D / 64;
  constexpr int kBatch = kMergeWideBatch;   // rows a wave requests at once
  __shared__ float s_acc[WAVES][D];
  __shared__ float s_max[WAVES], s_sum[WAVES];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned u = mapping & 256 ? blockIdx.x >> 3 : blockIdx.x;
  if (u >= (unsigned)rows_per_list) return;
  int s, hq;
  row_of(u, blockIdx.x & 7, per_list, per_list_magic, mapping, s, hq);
  const int64_t pair = (int64_t)s * heads + hq;
  const float ninf = -__builtin_inff();
  const float* __restrict__ lse = lse_part + pair * num_slots;
  const float* __restrict__ op = o_part + pair * (int64_t)num_slots * D;
  int ns = num_split_per_seq[s];
  float mx = ninf, sum = 0.f, acc[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) acc[c] = 0.f;
  if (SPEC) {
    const int mine = wave + lane * WAVES;   // this lane's slot
    float l = (lane < kBatch && mine < num_slots) ? lse[mine] : ninf;
    float v[kBatch][CPL];
#pragma unroll
    for (int b = 0; b < kBatch; ++b)
      if (wave + b * WAVES < num_slots) {
        const float* row = op + (int64_t)(wave + b * WAVES) * D + lane * CPL;
#pragma unroll
        for (int c = 0; c < CPL; ++c) v[b][c] = row[c];
      }
    ns = ns < 0 ? 0 : (ns > max_split ? max_split : ns);
    if (mine >= ns * chunks_per_rank) l = ninf;
    mx = l;
#pragma unroll
    for (int off = kBatch / 2; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    mx = __shfl(mx, 0);
    const float w_mine = (l != ninf) ? __expf(l - mx) : 0.f;
    sum = w_mine;
#pragma unroll
    for (int off = kBatch / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      const float w = __shfl(w_mine, b);
      // (rows of slots that are empty or beyond the count hold anything: dropped, not multiplied)
      if (wave + b * WAVES < num_slots && w != 0.f) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) acc[c] += w * v[b][c];
      }
    }
  } else {
    // (WAVES x 64 slots at a time: one turn of the loop but for plans of caller's buckets)
    for (int base = 0; base < num_slots; base += WAVES * 64) {
      const int mine = base + wave + lane * WAVES;
      float l = mine < num_slots ? lse[mine] : ninf;
      int n = ns < 0 ? 0 : (ns > max_split ? max_split : ns);
      if (mine >= n * chunks_per_rank) l = ninf;
      float m_new = fmaxf(mx, l);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) m_new = fmaxf(m_new, __shfl_xor(m_new, off));
      const float w_mine = (l != ninf) ? __expf(l - m_new) : 0.f;
      const float scale = mx == m_new ? 1.f : __expf(mx - m_new);   // (equal: the first turn's -inf as well)
      mx = m_new;
      float part = w_mine;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off);
      sum = sum * scale + part;
#pragma unroll
      for (int c = 0; c < CPL; ++c) acc[c] *= scale;
      unsigned long long live = __ballot(w_mine != 0.f);
      while (live) {
        int js[kBatch];
        float v[kBatch][CPL];
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
          js[b] = live ? __builtin_ctzll(live) : -1;
          live &= live - 1;   // 0 stays 0
        }
#pragma unroll
        for (int b = 0; b < kBatch; ++b)
          if (js[b] >= 0) {
            const float* row = op + (int64_t)(base + wave + js[b] * WAVES) * D + lane * CPL;
#pragma unroll
            for (int c = 0; c < CPL; ++c) v[b][c] = row[c];
          }
#pragma unroll
        for (int b = 0; b < kBatch; ++b)
          if (js[b] >= 0) {
            const float w = __shfl(w_mine, js[b]);
#pragma unroll
            for (int c = 0; c < CPL; ++c) acc[c] += w * v[b][c];
          }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < CPL; ++c) s_acc[wave][lane * CPL + c] = acc[c];
  if (lane == 0) { s_max[wave] = mx; s_sum[wave] = sum; }
  __syncthreads();
  if (threadIdx.x >= D) return;
  float most = s_max[0];
#pragma unroll
  for (int w = 1; w < WAVES; ++w) most = fmaxf(most, s_max[w]);
  float all = 0.f, x = 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const float weight = s_sum[w] != 0.f ? __expf(s_max[w] - most) : 0.f;
    all += weight * s_sum[w];
    x += weight * s_acc[w][threadIdx.x];
  }
  T* dst = (T*)p.out + (int64_t)s * p.o_stride_b + (int64_t)hq * p.o_stride_h + threadIdx.x;
  *dst = (T)(all != 0.f ? x / all : 0.f);
  if (p.lse_out != nullptr && threadIdx.x == 0) p.lse_out[pair] = all != 0.f ? most + logf(all) : ninf;
}

typedef void (*MergeFn)(const int32_t*, const float*, const float*, int, int, int, int, int, int, unsigned, int, const MergeParams);
template <int WAVES, bool SPEC>
static MergeFn wide_instance(bool bf16, int head_dim) {
  if (bf16) return head_dim == 64 ? pat_merge_wide_kernel<__bf16, 64, WAVES, SPEC> : pat_merge_wide_kernel<__bf16, 128, WAVES, SPEC>;
  return head_dim == 64 ? pat_merge_wide_kernel<_Float16, 64, WAVES, SPEC> : pat_merge_wide_kernel<_Float16, 128, WAVES, SPEC>;
}

// Host launcher: one wave per (sequence, query head), four per workgroup; a half-wave each in large launches
// of few slots, a workgroup each where slots are many and rows few (the lines: merge_form, fwd_params.hpp).
hipError_t launch_merge(bool bf16, int head_dim, hipStream_t stream, const MergeParams& params) {
  const int64_t pairs = (int64_t)params.batch * params.heads;
  MergeFn fn;
  int per_wg = 4, threads = 256;
  switch (merge_form(pairs, params.num_slots, head_dim)) {
    case kMergeHalfWave:
      per_wg = 8;
      if (bf16) fn = head_dim == 64 ? pat_merge_pairs_kernel<__bf16, 64> : pat_merge_pairs_kernel<__bf16, 128>;
      else fn = head_dim == 64 ? pat_merge_pairs_kernel<_Float16, 64> : pat_merge_pairs_kernel<_Float16, 128>;
      break;
    case kMergeWide4All: per_wg = 1; fn = wide_instance<4, true>(bf16, head_dim); break;
    case kMergeWide8All: per_wg = 1; threads = 512; fn = wide_instance<8, true>(bf16, head_dim); break;
    case kMergeWide4: per_wg = 1; fn = wide_instance<4, false>(bf16, head_dim); break;
    case kMergeWide8: per_wg = 1; threads = 512; fn = wide_instance<8, false>(bf16, head_dim); break;
    default:
      if (bf16) fn = head_dim == 64 ? pat_merge_kernel<__bf16, 64> : pat_merge_kernel<__bf16, 128>;
      else fn = head_dim == 64 ? pat_merge_kernel<_Float16, 64> : pat_merge_kernel<_Float16, 128>;
  }
  // (a multiple of 8 kv heads: 8 interleaved lists of pairs, one per XCD, each rounded up to whole workgroups)
  const bool xcd_lists = params.kv_heads % 8 == 0;
  const int lists = xcd_lists ? 8 : 1, per_list = params.heads / lists, group = params.heads / params.kv_heads;
  const uint32_t magic = per_list > 1 ? (uint32_t)((((uint64_t)1 << 32) + per_list - 1) / per_list) : 0u;
  const int64_t rows_per_list = pairs / lists;   // (below 2^31: checked with the launch)
  const int64_t wgs = lists * ((rows_per_list + per_wg - 1) / per_wg);
  const dim3 grid((unsigned)wgs), block((unsigned)threads);
  hipLaunchKernelGGL(fn, grid, block, 0, stream, params.num_split_per_seq, params.lse_part, params.o_part, params.num_slots,
                     params.chunks_per_rank, params.max_split, params.heads, (int)rows_per_list, per_list, magic,
                     group + (xcd_lists ? 256 : 0), params);
  return hipGetLastError();
}

}  // namespace pat
