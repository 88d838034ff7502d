// Split-KV forward kernel for gfx950 (MI355X): one workgroup streams one chunk of a packed box's
// KV for one kv head (short boxes: of four) and all rows of the box, or of two boxes of one tree
// node, and writes a normalised partial output + LSE per row.
//
// Functional contract (what the reference's pat_fwd_splitkv_kernel computes,
// csrc/pat_fwd_kernel.h:25-299): rows r = g + G*j of a box are (sequence
// q_table[j], query head h*G + g); every row attends to the same kv tokens, found
// through the box's block table; the partial result is softmax(q.K^T*scale).V over
// those tokens plus LSE = max + ln(sum) (csrc/softmax.h:169-188).
//
// Mapping to the hardware (this kernel's own design):
//  * work item = (box, kv-head, KV chunk), one workgroup of 4 wave64 each, launched as a flat
//    list with the kv-head fastest: workgroups are dealt to the 8 XCDs round-robin, so with 8
//    kv-heads XCD x serves head x and boxes that share KV pages (the boxes of one prefix node)
//    find them in that XCD's L2. Inside a bucket the list is chunk-major. What a workgroup is to do
//    it reads from its launch record (fwd_params.hpp), written once per plan by the record kernel.
//  * buckets of very short boxes: one workgroup serves 4 kv heads, one per wave, each wave
//    walking its head's steps alone (no combine).
//  * boxes of up to 16 rows (one MFMA row tile): each wave owns every 4th 32-token step of
//    the chunk on wave-private tiles and runs an independent online softmax; the 4 states are
//    combined through LDS at the end. K rows are the MFMA A operand of S^T = K.Q^T, so a lane
//    loads 16 contiguous bytes of one token straight from HBM into operand layout (no LDS).
//  * boxes of 17..64 rows, and two boxes of one node together (up to 128 rows): 32-row tiles on
//    v_mfma_f32_32x32x16. All waves walk the chunk in super-steps of 64 tokens whose K and V tiles are
//    fetched once per workgroup, straight from memory into a two-stage LDS buffer. Per row and token that is
//    half the MFMA, operand-read and softmax instructions of 16-row tiles.
//  * S^T on v_mfma_f32_16x16x32 (32x32x16 for tall boxes); its accumulator layout is the B-operand
//    layout of O^T = V^T.P^T, so P never moves between lanes.
//  * V must be contracted along tokens but is contiguous along head_dim: V tiles sit row-major
//    in LDS (padded rows, or permuted ones where memory is loaded straight into LDS) and are read back
//    transposed with ds_read_b64_tr_b16.
//  * all softmax state of a row lives in the 4 lanes {n, n+16, n+32, n+48}.
//  * the chunk's page ids live in two VGPRs per wave (lane i holds page i) and are
//    broadcast with v_readlane; with the launch record the prologue is three dependent memory
//    round trips: {record: header, page ids} -> {sequence ids, slots: the record's lines again} -> {K, V, Q}.
#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>

#include "fwd_params.hpp"
#include "lane_ops.hpp"

namespace pat {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

#define PAT_LDS __attribute__((address_space(3)))

template <typename T> struct Elem;
template <> struct Elem<_Float16> {
  using vec8 = f16x8;
  static __device__ __forceinline__ f32x4 mfma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16 mfma32(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};
template <> struct Elem<__bf16> {
  using vec8 = bf16x8;
  static __device__ __forceinline__ f32x4 mfma(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x16 mfma32(vec8 a, vec8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float neg_inf() { return -__builtin_inff(); }

// Two forms of the tall path (boxes of 17..64 rows), one kernel instance each:
//  TALLK 32: 32-row tiles on 32x32x16 MFMAs, 64-token super-steps; the faster walk of a tall box
//            (a lone workgroup: 1.1-1.3 us per 64 tokens of one box, ~1.5 of two), at the price of 64
//            accumulator registers and 64 KB of LDS: 2 workgroups per CU at head_dim 128;
//  TALLK 16: a 16-row tile per wave on 16x16x32 MFMAs, 32-token steps, three steps ahead in registers
//            (1.7 us per 64 tokens), in the register and LDS budget of the <= 16-row path: 3 per CU.
// The host picks per launch: 32 where the tall boxes are what the launch waits for, 16 where the
// <= 16-row boxes are and the third resident workgroup per CU is worth more (pat_fwd_tuning.tall_rows).
__host__ __device__ constexpr int split_occupancy(int head_dim, int tallk) {
  return (head_dim == 128 && tallk == 32) ? 2 : 3;
}

// LDS bytes of one workgroup (dynamic: more than the 64 KB a static allocation may have).
__host__ __device__ constexpr int split_smem_bytes(int D, int tallk, int waves = kWaves) {
  const int wave_private = waves * kStepTokens * (D * 2 + 32);      // private V tiles
  const int combine = waves * 16 * (D + 4) * 4;                      // short boxes: the waves' states
  const int tall = tallk == 0 ? 0 : tallk == 32 ? 2 * (2 * kStepTokens) * 2 * (D * 2)                     // two stages of 64 K rows + 64 V rows
                               : 2 * kStepTokens * ((D * 2 + 16) + (D * 2 + 32));        // two stages of 32 K rows + 32 V rows
  int m = wave_private > combine ? wave_private : combine;
  return m > tall ? m : tall;
}

// 16 bytes per lane from memory into LDS: lane i's go to lds + 16 i (`lds` uniform: an offset in the workgroup's
// LDS). The compiler does not see the loads: the caller waits for them (vmcnt) ahead of the barrier that hands the tile over.
__device__ __forceinline__ void load_to_lds(const char* base, unsigned lane_offset, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_offset), "s"(base), "s"(lds) : "memory", "m0");
}

// DIRECT instances serve launches in which every row has one partial slot: they store `out`. STREAM instances serve launches
// whose records may ask for V past the caches (kRecordModeStreamV): a second loop over short boxes, whose mere presence cost
// the smallest launches 0.14 us of 5.5.
// WAVES: 4, or 8 in instances without a tall path (TALLK 0) for single launches of few workgroups whose boxes are more than eight steps
// long: a wave has half the steps, each a trip to memory behind the last (us per call: 8 requests of 288 tokens, 8 kv heads of 64, 64 workgroups, 5.5 / 4.7;
// 2 of 306..459 at 64/8, head_dim 64, 6.5 / 5.3; 17 of 188..282 at 8/8, head_dim 128, 6.8 / 6.3); and for launches of such boxes in pieces of
// double length, a workgroup per CU (8 of 2239 at 64/8, head_dim 128, 384 workgroups of four / 192 of eight, 18.1 / 16.9).
// TAILS instances (32-row form): tall workgroups also walk the tails of their rows' sequences.
// LISTS instances: workgroups of short buckets may serve several boxes of one sequence each (kRecordModeList).
template <typename T, int D, bool DIRECT, int TALLK, bool STREAM, bool TAILS, int WAVES, bool LISTS>
__global__ void __launch_bounds__(WAVES * 64, TALLK == 0 ? WAVES / 4 : split_occupancy(D, TALLK)) pat_split_kernel(const char* __restrict__ records, const int record_stride,
                                                                             const int record_max_seqs, const int record_max_pages, const SplitParams p) {
  using E = Elem<T>;
  using vec8 = typename E::vec8;
  constexpr int KK = D / 32;             // MFMA k-steps across head_dim in S^T = K.Q^T (16x16x32 tiles)
  constexpr int DB = D / 16;             // 16-wide head_dim blocks of O^T (16x16x32 tiles)
  constexpr int NV = D / 16;             // 16-byte V loads per lane per step (wave-private tiles)
  constexpr int CPR = D / 8;             // 16-byte pieces per token row
  constexpr int TPL = 64 / CPR;          // tokens covered by one wave-wide load instruction
  constexpr int RSV = D * 2 + 32;        // LDS row stride of a wave-private V tile (conflict-free transposed reads)
  constexpr int VSTAGE = kStepTokens * RSV;            // one wave's private V tile
  constexpr int OROW = D + 4;            // padded row of the combine buffer, floats
  constexpr int WSTAGE = VSTAGE;                       // one wave's private staging (V only)

  extern __shared__ __attribute__((aligned(256))) char smem[];
  __shared__ float s_m[WAVES * 16];
  __shared__ float s_l[WAVES * 16];

  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int g = lane >> 4;   // 16-row tiles: lane group 0..3
  const int n = lane & 15;   //               index inside the group
  const int h2 = lane >> 5;  // 32-row tiles: lane half
  const int n32 = lane & 31; //               index inside the half

  // ---- this workgroup's launch record: one round trip for everything the plan says about it ---
  // (header, sequence ids and partial-result slots of its rows, page ids of its piece: checked,
  // clamped and laid out by the record kernel once per plan). The launch is a flat list of
  // workgroups; consecutive ones serve consecutive kv heads of one piece (workgroups are dealt to
  // the 8 XCDs round-robin, so with 8 kv heads XCD x serves head x and the boxes that share KV
  // pages find them in that XCD's L2), and inside a bucket the list is chunk-major.
  // (the grid is padded to whole slices of kGridX only beyond 2^20 workgroups; the padding has
  // records too, empty ones, so nothing here waits for a bound from the kernel arguments)
  const unsigned wg_id = blockIdx.y * (unsigned)kGridX + blockIdx.x;
  const char* __restrict__ rec = records + (size_t)wg_id * (unsigned)record_stride;
  const int4 rh0 = *(const int4*)rec;
  const int4 rh1 = *(const int4*)(rec + 16);
  const int* __restrict__ rows_tab = (const int*)(rec + sizeof(RecordHead));
  const int* __restrict__ pages_tab = rows_tab + 2 * record_max_seqs;
  // Page ids of the piece: lane i of every wave holds pages i and 64 + i. The first 64 are requested with the header,
  // not behind it (the record kernel filled all record_max_pages entries with pages of the cache, so which of them the
  // piece has does not matter); the others, which few pieces have, wait for it. So do the rows' entries: requested with
  // the header as well, by all lanes and picked by shuffles, they made single launches of one long request 1 % faster
  // and launches that queue workgroups 1-2 % slower (369 boxes at head_dim 64 90.7 -> 92.5 us, 64 requests behind one
  // prefix 22.1 -> 22.5).
  const int pg0 = pages_tab[min(lane, record_max_pages - 1)];
  // the rest of the kernel's arguments, requested here as well (left alone, a round trip of their own ahead of K and V)
  asm volatile("" ::"s"(p.k), "s"(p.v), "s"(p.q), "s"(p.q_stride_b), "s"(p.k_stride_page), "s"(p.k_stride_slot), "s"(p.k_stride_h),
               "s"(p.v_stride_page), "s"(p.v_stride_slot), "s"(p.v_stride_h), "s"(p.page_size), "s"(p.scale_log2));
  // The piece's length, twice: as a scalar for the loops of the tall path, and laundered
  // into a vector register for the wave-private path. With loop bounds it can prove uniform the
  // compiler schedules the wave-private loops for 50 more registers; with vector bounds in the
  // tall path its per-step branches turn into masked execution of both sides.
  int ntok_v = rh0.x;
  asm volatile("" : "+v"(ntok_v));
  const int ntok = ntok_v;
  const int ntok_u = __builtin_amdgcn_readfirstlane(rh0.x);
  const int R = __builtin_amdgcn_readfirstlane(rh0.y);
  const int mode = __builtin_amdgcn_readfirstlane(rh0.z);
  const bool head_per_wave = (mode & kRecordModeHeadPerWave) != 0;
  // Boxes of up to 16 rows: the 4 waves split the piece's steps, each on wave-private tiles (or,
  // with a kv head per wave, each wave walks all steps of its own head).
  // Taller boxes: tiles shared through LDS; the 32-row form gives a wave rows 32w.. and every token, or, up to
  // 64 rows, rows 32(w&1).. and tokens 32(w>>1).. of every 64-token super-step.
  const bool tall = TALLK != 0 && (mode & 0xff) > 1;
  // (both uniform, and known to be: branches on them are scalar branches)
  const bool one_tile_per_wave = R > 64;   // tall boxes, 32-row tiles: four row tiles, a wave each
  const int rt = __builtin_amdgcn_readfirstlane(one_tile_per_wave ? wave : wave & 1);   // this wave's 32-row tile
  const int ph = __builtin_amdgcn_readfirstlane(one_tile_per_wave ? 0 : wave >> 1);     // and which half of a super-step it works on
  // (uniform over the wave: kept in a scalar register so that address arithmetic stays scalar)
  const int head = __builtin_amdgcn_readfirstlane(rh0.w + (head_per_wave ? (int)(threadIdx.x >> 6) : 0));
  const int fill_begin = __builtin_amdgcn_readfirstlane(rh1.x);
  const int fill_end = __builtin_amdgcn_readfirstlane(rh1.y);
  const int G = p.group;                       // 1, 2, 4 or 8 (checked on the host)
  const int gshift = 31 - __builtin_clz(G);
  const int page = p.page_size;
  const int pg1 = ntok_u > 64 * page ? pages_tab[min(64 + lane, record_max_pages - 1)] : 0;
  // this lane's row: sequence id and partial-result slot (-1: no such row)
  const int my_row = tall ? (TALLK == 32 ? rt * 32 + n32 : wave * 16 + n) : n;
  const int my_j = my_row >> gshift;
  const bool j_ok = (my_row < R) && my_j < record_max_seqs;
  const int my_seq = j_ok ? rows_tab[my_j] : -1;
  const int my_sl = j_ok ? rows_tab[record_max_seqs + my_j] : -1;

  const bool has_rows = !tall || (TALLK == 32 ? rt * 32 : wave * 16) < R;   // false: a wave that only helps loading shared tiles
  const bool row_ok = my_seq >= 0 && my_sl >= 0;
  const int my_hq = head * G + (my_row & (G - 1));
  // partial slot of (my row, this piece); -1: the row is not to be written
  const int my_slot0 = row_ok ? (my_seq * p.heads + my_hq) * p.num_slots + my_sl : -1;
  // the one lane per row that writes what exists once per row (LSE, empty-slot marks)
  const bool row_lead = tall ? (TALLK == 32 ? (ph == 0 && h2 == 0) : g == 0) : ((head_per_wave || wave == 0) && g == 0);

  // ---- where a finished row goes ---------------------------------------------------------
  // Normally into its partial slot (fp32, merged by the second kernel). A launch in which every
  // row has exactly one slot (no sequence in two boxes, no box in two chunks) has nothing to
  // merge: its rows go straight to `out` in the output type (the reference does the same when
  // max_split_per_seq is 1, csrc/api.h:230-238). A row's slot index is then its (sequence, head)
  // pair.
  constexpr bool direct = DIRECT;
  auto row_out = [&](int slot0) -> T* {
    const int s_ = slot0 / p.heads;
    return (T*)p.out + (int64_t)s_ * p.o_stride_b + (int64_t)(slot0 - s_ * p.heads) * p.o_stride_h;
  };
  auto put4 = [&](float* part, T* out, f32x4 v) {
    if (direct) {
      typedef T tx4 __attribute__((ext_vector_type(4)));
      *(tx4*)out = tx4{(T)v[0], (T)v[1], (T)v[2], (T)v[3]};
    } else {
      *(f32x4*)part = v;
    }
  };
  auto put_lse = [&](int64_t prow, float lse) {
    if (!direct) p.lse_part[prow] = lse;
    else if (p.lse_out != nullptr) p.lse_out[prow] = lse;
  };

  // ---- slots of these rows that no workgroup will fill are marked empty (-inf) -----------
  {
    const bool empty = ntok <= 0;
    const bool marker = row_lead && my_slot0 >= 0;
    if (direct) {
      // (one piece per box: only a box without tokens gets here; its rows are zero, LSE -inf)
      if (empty && marker) {
        T* o = row_out(my_slot0);
        for (int c = 0; c < D; c += 4) put4(nullptr, o + c, f32x4{0.f, 0.f, 0.f, 0.f});
        put_lse(my_slot0, neg_inf());
      }
    } else if (marker)
      for (int c = fill_begin; c < fill_end; ++c) p.lse_part[my_slot0 + c] = neg_inf();
    if (empty) return;
  }
  const int t_begin = 0, t_end = ntok;   // token positions are piece-relative from here on
  const int last_rel = ntok - 1;
  const int nsteps = (ntok + kStepTokens - 1) / kStepTokens;

  // ---- addressing ---------------------------------------------------------------------------
  // A 16-token half of a step never straddles a page, so its rows share one base address that is
  // uniform over the wave (page id broadcast with v_readlane, 64-bit arithmetic on the scalar
  // unit) and every lane adds a 32-bit byte offset that does not change from step to step.
  const int hpp = page >> 4;                                   // halves per page
  const int hshift = ((hpp & (hpp - 1)) == 0) ? 31 - __builtin_clz(hpp) : -1;
  const int64_t ksp = p.k_stride_page * (int64_t)sizeof(T), kss = p.k_stride_slot * (int64_t)sizeof(T);
  const int64_t vsp = p.v_stride_page * (int64_t)sizeof(T), vss = p.v_stride_slot * (int64_t)sizeof(T);
  const char* __restrict__ kbase = (const char*)p.k + (int64_t)head * p.k_stride_h * (int64_t)sizeof(T);
  const char* __restrict__ vbase = (const char*)p.v + (int64_t)head * p.v_stride_h * (int64_t)sizeof(T);

  // base address of half h (chunk-relative, uniform, h * 16 <= last_rel)
  auto half_base = [&](const char* base, int64_t sp, int64_t ss, int h) -> const char* {
    int pidx, s16;
    if (hshift >= 0) { pidx = h >> hshift; s16 = h & (hpp - 1); }
    else { pidx = (int)__umulhi((unsigned)h, p.hpp_magic); s16 = h - pidx * hpp; }
    const int pg = __builtin_amdgcn_readlane(pidx < 64 ? pg0 : pg1, pidx & 63);
    return base + (int64_t)pg * sp + (int64_t)(s16 * 16) * ss;
  };
  // per-lane address of token tok (chunk-relative; clamped to the last valid token, whose score
  // is masked and whose probability is 0 wherever it stands in for a token past the end). Only
  // the last, partial step of a chunk takes this slower route.
  auto lane_row = [&](const char* base, int64_t sp, int64_t ss, int tok) -> const char* {
    tok = tok > last_rel ? last_rel : tok;
    const int h = tok >> 4;
    int pidx, s16;
    if (hshift >= 0) { pidx = h >> hshift; s16 = h & (hpp - 1); }
    else { pidx = (int)__umulhi((unsigned)h, p.hpp_magic); s16 = h - pidx * hpp; }
    const int pg = __shfl(pidx < 64 ? pg0 : pg1, pidx & 63);
    return base + (int64_t)pg * sp + (int64_t)(s16 * 16 + (tok & 15)) * ss;
  };

  // Half h of the chunk as the loads see it (uniform over the wave): the half that holds its rows
  // and, in `lim`, the last row of that half that exists. Rows past the end of the chunk re-read
  // the chunk's last token (their scores are masked and their probabilities are 0); a half that
  // lies wholly past the end stands in for the half of that token.
  auto half_geom = [&](int h, int& lim) -> int {
    const int left = last_rel - h * 16;
    lim = left < 0 ? (last_rel & 15) : (left > 15 ? 15 : left);
    return left < 0 ? (last_rel >> 4) : h;
  };

  // Q rows as MFMA B operand of the 16x16x32 tiles (lane (g, n): row n, dims kk*32 + g*8 .. +7)
  vec8 qreg[KK];
  auto load_q = [&]() {
    const bool ok = my_seq >= 0;
    const T* qrow = (const T*)p.q + (ok ? ((int64_t)my_seq * p.q_stride_b + (int64_t)my_hq * p.q_stride_h) : 0);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      u32x4 raw = u32x4{0u, 0u, 0u, 0u};
      if (ok) raw = *(const u32x4*)(qrow + kk * 32 + g * 8);
      qreg[kk] = __builtin_bit_cast(vec8, raw);
    }
  };

  float m_run = neg_inf(), l_run = 0.f;
  f32x4 acc_o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc_o[db] = f32x4{0.f, 0.f, 0.f, 0.f};

  // One 32-token step of online-softmax attention for this wave's 16 rows. k_op(a, kk) yields the
  // K operand of half a / k-step kk; vtile is a row-major V tile in LDS with row stride RSV.
  // after_scores() runs once the K operands have been consumed: the caller refills their
  // registers there, so the next step's K is in flight during the softmax and the PV product.
  auto attend = [&](auto k_op, const PAT_LDS char* vtile, int t0, int t_end, float& m_run, float& l_run, auto after_scores) {
    f32x4 sc[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) acc = E::mfma(k_op(a, kk), qreg[kk], acc);
      sc[a] = acc * p.scale_log2;
    }
    after_scores();
    if (t0 + kStepTokens > t_end) {
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (t0 + a * 16 + g * 4 + i >= t_end) sc[a][i] = neg_inf();
    }
    // the row's running max is shared by its 4 lanes, the sum stays per lane until the end
    float mx = fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])),
                     fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
    mx = max_xor32(max_xor16(mx));
    const float m_new = fmaxf(m_run, mx);
    const float alpha = fast_exp2(m_run - m_new);
    // once the running maxima have settled no row of the wave needs its accumulator rescaled
    const bool rescale = __builtin_amdgcn_ballot_w64(m_new != m_run) != 0;
    m_run = m_new;
    float psum = 0.f;
    vec8 pv;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = fast_exp2(sc[a][i] - m_new);
        psum += e;
        pv[a * 4 + i] = (T)e;
      }
    l_run = l_run * alpha + psum;
    if (rescale) {
      asm volatile("" ::: "memory");   // a real branch: if-converted, the skipped multiplies come back as selects
#pragma unroll
      for (int db = 0; db < DB; ++db) acc_o[db] = acc_o[db] * alpha;
    }
    // O^T += V^T.P^T. V^T operand: lane (g, n) of d-block db gets 8 tokens of column db*16 + n:
    // tokens g*4..g*4+3 of each 16-token half, matching the accumulator layout of S^T.
    const PAT_LDS char* src = vtile + (g * 4 + (n >> 2)) * RSV + (n & 3) * 8;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PAT_LDS s16x4*)(src + db * 32));
      s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PAT_LDS s16x4*)(src + 16 * RSV + db * 32));
      s16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      acc_o[db] = E::mfma(__builtin_bit_cast(vec8, both), pv, acc_o[db]);
    }
  };

  // Short boxes of one sequence each, one after the other by one wave (`live`: which of up to 64): rows of a sequence on 16x16x32
  // tiles, K straight into operand registers, V through the wave's own LDS tile, the next step's tiles in flight. finish(j, max, sum)
  // takes box j's sums out of acc_o.
  auto walk_list = [&](uint64_t live, auto tokens_of, auto page_of, auto seq_of, PAT_LDS char* vtile, auto finish) {
    u32x4 kd[2][KK], vd[NV];
    // half of a step at token t of box j (`tok` tokens): base address; `lim`: its last row that exists (rows past the end
    // re-read the last token, as everywhere)
    auto half_at = [&](const char* base, int64_t sp, int64_t ss, int j, int tok, int t, int& lim) -> const char* {
      const int left = tok - 1 - t;
      lim = left < 0 ? (tok - 1) & 15 : (left > 15 ? 15 : left);
      const int h = left < 0 ? (tok - 1) >> 4 : t >> 4;
      int pidx, s16;
      if (hshift >= 0) { pidx = h >> hshift; s16 = h & (hpp - 1); }
      else { pidx = (int)__umulhi((unsigned)h, p.hpp_magic); s16 = h - pidx * hpp; }
      return base + (int64_t)page_of(j, pidx) * sp + (int64_t)(s16 * 16) * ss;
    };
    auto get_v = [&](int j, int tok, int t0) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        int lim;
        const char* vb = half_at(vbase, vsp, vss, j, tok, t0 + a * 16, lim);
#pragma unroll
        for (int i = 0; i < NV / 2; ++i) {
          const unsigned vo = (unsigned)min(i * TPL + lane / CPR, lim) * (unsigned)vss + (lane % CPR) * 16;
          vd[a * (NV / 2) + i] = *(const u32x4*)(vb + vo);
        }
      }
    };
    auto get_k = [&](int j, int tok, int t0) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        int lim;
        const char* kb = half_at(kbase, ksp, kss, j, tok, t0 + a * 16, lim);
        const unsigned ko = (unsigned)min(n, lim) * (unsigned)kss + g * 16;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) kd[a][kk] = *(const u32x4*)(kb + ko + kk * 64);
      }
    };
    auto get_q = [&](int j) {   // (columns past the sequence's rows hold one of them again: they go nowhere)
      const T* qrow = (const T*)p.q + ((int64_t)seq_of(j) * p.q_stride_b + (int64_t)(head * G + (n & (G - 1))) * p.q_stride_h);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) qreg[kk] = __builtin_bit_cast(vec8, *(const u32x4*)(qrow + kk * 32 + g * 8));
    };
    int j = (int)__builtin_ctzll(live), t0 = 0, tok = tokens_of(j);
    float m_t = neg_inf(), l_t = 0.f;
    get_v(j, tok, t0);
    get_k(j, tok, t0);
    get_q(j);
    // One step. Every request is made in every step but the last, which stands apart, so that a wait counts exactly the loads
    // behind the one it is for; with requests that may not be made each step waited for all of them, a full trip to memory
    // per box.
    auto step = [&](auto more_c) {
      constexpr bool more = decltype(more_c)::value;
      // the step behind this one: of this box, or the next one's first
      const bool ends = !more || t0 + kStepTokens >= tok;
      int next_j = j, next_t0 = t0 + kStepTokens, next_tok = tok;
      if (more && ends) {
        live &= live - 1;
        next_j = (int)__builtin_ctzll(live);
        next_t0 = 0;
        next_tok = tokens_of(next_j);
      }
#pragma unroll
      for (int i = 0; i < NV; ++i)
        *(PAT_LDS u32x4*)(vtile + (i * TPL + lane / CPR) * RSV + (lane % CPR) * 16) = vd[i];
      if (more) get_v(next_j, next_tok, next_t0);
      attend([&](int a, int kk) { return __builtin_bit_cast(vec8, kd[a][kk]); }, vtile, t0, tok, m_t, l_t, [&]() {
        if (more) {
          get_k(next_j, next_tok, next_t0);
          get_q(next_j);
        }
      });
      if (ends) {
        finish(j, m_t, sum_xor32(sum_xor16(l_t)));
        m_t = neg_inf();
        l_t = 0.f;
#pragma unroll
        for (int db = 0; db < DB; ++db) acc_o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      j = next_j;
      t0 = next_t0;
      tok = next_tok;
    };
    while ((live & (live - 1)) != 0 || t0 + kStepTokens < tok) step(std::true_type{});
    step(std::false_type{});
  };

  if (tall) {
    if constexpr (TALLK == 16) {
    constexpr int NP = D / 64;             // 16-byte K (and V) loads per thread per step
    constexpr int PF = 3;                  // steps kept in flight per workgroup (a 4th costs the registers that let the operand
                                           // reads of a step run ahead of its MFMAs: lone tall workgroups 6 % slower per step)
    constexpr int RSK = D * 2 + 16;        // LDS row stride of a K tile (conflict-free 16-byte row reads)
    constexpr int SHARED = kStepTokens * (RSK + RSV);    // one K + V stage
    static_assert(2 * SHARED <= split_smem_bytes(D, 16), "LDS size");
    const int nsteps_u = (ntok_u + kStepTokens - 1) / kStepTokens;
    // ============ tall box, 16-row tile per wave: 32-token tiles shared through LDS ============
    // Each step's K and V tile is fetched once per workgroup: thread t loads pieces t, t + 256 ..
    // of the tile (16 lanes cover one 256-byte row), PF steps ahead, and drops them into one of
    // two LDS stages; after a barrier every wave runs its own 16 rows against the stage.
    u32x4 kst[PF][NP], vst[PF][NP];
    int tok_in[NP];
    unsigned koff[NP], voff[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      tok_in[i] = (i * kThreads + tid) / CPR;                 // token of the step, 0..31
      const unsigned col = ((i * kThreads + tid) % CPR) * 16;
      koff[i] = (unsigned)((tok_in[i] & 15) * kss) + col;
      voff[i] = (unsigned)((tok_in[i] & 15) * vss) + col;
    }
    // Steps are fetched in order, so the half a wave reads next is tracked on the scalar unit
    // (page of the chunk, 16-token slot in the page, byte offset of the slot) instead of being
    // derived from the step number every time: a few scalar adds per half. Page strides are
    // below 4 GiB (checked on the host): page id x stride is one 32 x 32 -> 64 bit multiply.
    int f_page = 0, f_slot = 0;
    unsigned f_koff = 0, f_voff = 0;
    const unsigned ksp32 = (unsigned)ksp, vsp32 = (unsigned)vsp, k16 = (unsigned)(16 * kss), v16 = (unsigned)(16 * vss);
    auto next_half = [&]() {
      ++f_slot; f_koff += k16; f_voff += v16;
      if (f_slot == hpp) { f_slot = 0; f_koff = 0; f_voff = 0; ++f_page; }
    };
    // D = 64: one load per step and thread, waves 2 and 3 read the step's second half
    if (NP == 1 && __builtin_amdgcn_readfirstlane(wave >> 1)) next_half();
    auto fetch = [&](int st, u32x4 (&kd)[NP], u32x4 (&vd)[NP]) {
      if ((st + 1) * kStepTokens <= ntok_u) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          const unsigned pg = (unsigned)__builtin_amdgcn_readlane(f_page < 64 ? pg0 : pg1, f_page & 63);
          kd[i] = *(const u32x4*)(kbase + ((uint64_t)pg * ksp32 + f_koff) + koff[i]);
          vd[i] = *(const u32x4*)(vbase + ((uint64_t)pg * vsp32 + f_voff) + voff[i]);
          next_half();
        }
        if (NP == 1) next_half();
      } else {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          const unsigned col = ((i * kThreads + tid) % CPR) * 16;
          kd[i] = *(const u32x4*)(lane_row(kbase, ksp, kss, st * kStepTokens + tok_in[i]) + col);
          vd[i] = *(const u32x4*)(lane_row(vbase, vsp, vss, st * kStepTokens + tok_in[i]) + col);
        }
      }
    };
#pragma unroll
    for (int s = 0; s < PF; ++s)
      if (s < nsteps_u) fetch(s, kst[s], vst[s]);
    load_q();
    for (int st0 = 0; st0 < nsteps_u; st0 += PF) {
#pragma unroll
      for (int s = 0; s < PF; ++s) {
        const int st = st0 + s;
        if (st >= nsteps_u) break;
        PAT_LDS char* stage = (PAT_LDS char*)smem + (st & 1) * SHARED;
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          const int tok_in = (i * kThreads + tid) / CPR;
          const int col16 = ((i * kThreads + tid) % CPR) * 16;
          *(PAT_LDS u32x4*)(stage + tok_in * RSK + col16) = kst[s][i];
          *(PAT_LDS u32x4*)(stage + kStepTokens * RSK + tok_in * RSV + col16) = vst[s][i];
        }
        if (st + PF < nsteps_u) fetch(st + PF, kst[s], vst[s]);
        __syncthreads();
        if (has_rows)
          attend([&](int a, int kk) { return *(const PAT_LDS vec8*)(stage + (a * 16 + n) * RSK + (kk * 32 + g * 8) * 2); },
                 stage + kStepTokens * RSK, t_begin + st * kStepTokens, t_end, m_run, l_run, []() {});
      }
    }
    l_run = sum_xor32(sum_xor16(l_run));
    if (my_slot0 >= 0) {
      const int64_t prow = (int64_t)my_slot0;
      const float inv = 1.f / l_run;
      float* dst = p.o_part + prow * D + g * 4;
      T* o = direct ? row_out(my_slot0) + g * 4 : nullptr;
#pragma unroll
      for (int db = 0; db < DB; ++db) put4(dst + db * 16, o + db * 16, acc_o[db] * inv);
      if (g == 0) put_lse(prow, (m_run + __builtin_amdgcn_logf(l_run)) * 0.6931471805599453f);
    }
    } else if constexpr (TALLK == 32) {
    // ====================== tall box: 32-row tiles, K/V shared through LDS ======================
    // The piece is walked in super-steps of 64 tokens, whose K and V rows go from memory straight into one of
    // two LDS stages (global_load_lds, 16 bytes per lane): the next super-step is in flight while the waves work
    // on the current one, and no register holds a tile on its way. Wave w fetches the 16-token half w of every
    // super-step: one page id, one address.
    // What bounds it: the chain score - softmax - weighted sum of each wave. Two of these workgroups on a CU take ~2 us per
    // super-step of two boxes, ~1050 TFLOP/s in the steady state (65536 rows x 16384 tokens, 8 kv heads; a library matrix
    // product reaches 1200); over 65536 rows x 2048 tokens, prologue, stores and short boxes included, the MFMA pipe is
    // busy 29 % of the launch and LDS 16 %. With the tiles staged through registers and one box per workgroup (four workgroups
    // reading what one does now) that launch took 156 us, now 117.
    //  * more than 64 rows (two boxes of one node): wave w owns row tile w (rows 32w..) and all 64 tokens;
    //  * up to 64 rows: the wave pair ph = w >> 1 takes tokens 32ph.. of every super-step, wave w row tile
    //    w & 1; the pairs' states are combined through LDS at the end.
    //   S^T = K.Q^T on 32x32x16 tiles: A = K (lane: token n32, dims 16kk + 8h2 ..+7, a 16-byte
    //   LDS read), B = Q^T in registers; the accumulator holds, in lane (n32, h2), row n32's scores
    //   for tokens 8b + 4h2 + r (register 4b + r).
    //   O^T += V^T.P^T: B = P^T straight from those registers - k index 8h2 + j of MFMA t stands
    //   for token 16t + 8(j>>2) + 4h2 + (j&3), any order does as long as V^T uses the same - and
    //   A = V^T read transposed from LDS (two 4-token groups per lane and MFMA). The row's softmax
    //   state lives in the two lanes n32 and n32 + 32.
    // A load into LDS writes 64 consecutive 16-byte pieces, so rows cannot be padded: bank conflicts are kept
    // away by permuting the pieces inside a row instead (each lane fetches the piece that belongs where it
    // writes). K: piece p of row r stands at p ^ (r & 15) (head_dim 128; 64: p ^ ((r >> 1) & 7)), so the 16 rows
    // of a read step over all banks; V: 64-byte block b of row r at b ^ (r & 3) (64: b ^ ((r >> 1) & 1)), so the
    // four rows of a transposed read do.
    constexpr int KK2 = D / 16;            // MFMA k-steps across head_dim in S^T
    constexpr int DB2 = D / 32;            // 32-wide head_dim blocks of O^T
    constexpr int SST = 2 * kStepTokens;   // tokens per super-step
    constexpr int ROWB = D * 2;            // bytes of a K or V row
    constexpr int KTILE = SST * ROWB;      // one operand's tile of a super-step
    constexpr int STAGE2 = 2 * KTILE;      // K rows, then V rows
    constexpr int RPI = 64 / CPR;          // rows one load instruction covers
    constexpr int NI = 16 / RPI;           // load instructions per wave, operand and super-step
    static_assert(2 * STAGE2 <= split_smem_bytes(D, 32), "LDS size");
    static_assert(2 * (D / 8) * 64 * 16 <= 2 * STAGE2, "the exchange buffer of the epilogue fits the stages");
    const int nss_u = (ntok_u + SST - 1) / SST;
    const int last_rel_u = ntok_u - 1;
    // (a scale of 0 stands as the smallest normal number, which keeps masked scores at -inf; a NaN stays one)
    const float sc_abs = p.scale_log2 == 0.f ? 1.17549435e-38f : __builtin_fabsf(p.scale_log2);

    // Q^T operand (lane (n32, h2): row n32, dims 16kk + 8h2 ..+7). A negative softmax scale is
    // folded into Q's sign (exact), so that the row maximum can be taken over the raw scores.
    u32x4 q2[KK2];
    {
      const bool ok = my_seq >= 0;
      const T* qrow = (const T*)p.q + (ok ? ((int64_t)my_seq * p.q_stride_b + (int64_t)my_hq * p.q_stride_h) : 0);
      const unsigned flip = p.scale_log2 < 0.f ? 0x80008000u : 0u;
#pragma unroll
      for (int kk = 0; kk < KK2; ++kk) {
        u32x4 raw = u32x4{0u, 0u, 0u, 0u};
        if (ok) raw = *(const u32x4*)(qrow + kk * 16 + h2 * 8);
        q2[kk] = raw ^ u32x4{flip, flip, flip, flip};
      }
    }
    f32x16 acc2[DB2];
#pragma unroll
    for (int db = 0; db < DB2; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc2[db][i] = 0.f;

    // ---- tails: the few tokens that each sequence of the box has behind it, alone ----------------------
    // Behind the piece, whose registers are free again. A wave takes those of its own 32 rows one after the other (of two waves on the
    // same rows every second one): rows of one sequence on 16x16x32 tiles, as the boxes of <= 16 rows are walked, K straight into operand registers, V through a region of
    // LDS of this wave's own, the next step's tiles in flight. Each tail is a softmax of its own, added to its rows' state in fp32: a
    // tile that several sequences shared, masked, would carry one's infinite or NaN V into the others' sums.
    const int* __restrict__ tail_tab = pages_tab + record_max_pages;   // tokens by sequence, then pages
    const int per_tile = 32 >> gshift, tail_pages = TAILS ? p.tail_pages : 0;
    int tok_mine = 0, tp0 = 0, tp1 = 0;   // lane i: tokens of the tail of the tile's sequence i; pages i and 64 + i of the tile's tails
    uint64_t tails_mine = 0;              // bit i: this wave walks the tail of the tile's sequence i
    if constexpr (TAILS) {
      const int j0 = rt * per_tile, entries = record_max_seqs * (1 + tail_pages);
      if (lane < per_tile && j0 + lane < record_max_seqs) tok_mine = tail_tab[j0 + lane];
      const int first = record_max_seqs + j0 * tail_pages;
      tp0 = tail_tab[min(first + lane, entries - 1)];
      tp1 = tail_tab[min(first + 64 + lane, entries - 1)];
      tails_mine = __builtin_amdgcn_ballot_w64(tok_mine > 0);
      if (!one_tile_per_wave) {
        const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(tails_mine >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)tails_mine, 0u));
        tails_mine = __builtin_amdgcn_ballot_w64(tok_mine > 0 && (rank & 1) == ph);
      }
    }
    auto walk_tails = [&]() {
      constexpr int REGION = split_smem_bytes(D, 32) / kWaves;
      static_assert(VSTAGE + 8 * OROW * 4 <= REGION, "a wave's V tile and the result of a sequence's rows fit its part of LDS");
      uint64_t live = tails_mine;
      if (live == 0) return;
      PAT_LDS char* vtile = (PAT_LDS char*)smem + wave * REGION;
      PAT_LDS float* result = (PAT_LDS float*)(vtile + VSTAGE);   // [row of the sequence][OROW]
      walk_list(live, [&](int j) { return __builtin_amdgcn_readlane(tok_mine, j); },
                [&](int j, int page) {
                  const int e = j * tail_pages + page;
                  return __builtin_amdgcn_readlane(e < 64 ? tp0 : tp1, e & 63);
                },
                [&](int j) { return __builtin_amdgcn_readlane(my_seq, j << gshift); }, vtile, [&](int j, float m_t, float l_t) {
        // into the state of the sequence's rows: from lane (g, n), row n, columns 16 db + 4 g .. to lane (n32, h2)
        if (n < G) {
#pragma unroll
          for (int db = 0; db < DB; ++db) *(PAT_LDS f32x4*)(result + n * OROW + db * 16 + g * 4) = acc_o[db];
        }
        const int row = n32 & (G - 1);
        const float mt = __shfl(m_t, row), lt = __shfl(l_t, row);
        asm volatile("" ::: "memory");   // (the wave reads what its own lanes wrote: in order, no barrier)
        if ((n32 >> gshift) == j) {
          const float m_new = fmaxf(m_run, mt);
          const float wa = m_run == m_new ? 1.f : fast_exp2(m_run - m_new), wb = fast_exp2(mt - m_new);
          m_run = m_new;
          l_run = l_run * wa + (h2 == 0 ? lt * wb : 0.f);   // (the two lanes of a row hold parts of its sum)
#pragma unroll
          for (int db = 0; db < DB2; ++db)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
              const f32x4 x = *(const PAT_LDS f32x4*)(result + row * OROW + db * 32 + b * 8 + h2 * 4);
#pragma unroll
              for (int r = 0; r < 4; ++r) acc2[db][4 * b + r] = __builtin_fmaf(x[r], wb, acc2[db][4 * b + r] * wa);
            }
        }
      });
    };
    // this lane's place in its wave's half: row RPI*i + r_in of load i, and the piece it fetches there
    const int r_in = lane / CPR, c_in = lane % CPR;
    auto k_piece = [&](int i) { return (unsigned)(D == 128 ? c_in ^ ((RPI * i + r_in) & 15) : c_in ^ (((RPI * i + r_in) >> 1) & 7)) * 16u; };
    const unsigned v_piece = (unsigned)(D == 128 ? c_in ^ ((r_in & 3) << 2) : c_in ^ (((r_in >> 1) & 1) << 2)) * 16u;
    unsigned koff[NI], voff[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      koff[i] = (unsigned)((RPI * i + r_in) * kss) + k_piece(i);
      voff[i] = (unsigned)((RPI * i + r_in) * vss) + v_piece;
    }
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const unsigned lds_base = (unsigned)(size_t)(PAT_LDS char*)smem + (unsigned)wave_u * 16u * ROWB;
    // Addresses of this wave's halves, worked out once: lane i holds those of super-step i (the host plans no piece of
    // more than kMaxTall32Tokens = 64 super-steps for this form). Halves past the end stand in for the last one. Two
    // v_readlane per operand and super-step are all that is left of the addressing inside the loop.
    uint64_t k_at, v_at;
    {
      int h = lane * (SST / 16) + wave_u;
      h = h > (last_rel >> 4) ? last_rel >> 4 : h;
      int pidx, s16;
      if (hshift >= 0) { pidx = h >> hshift; s16 = h & (hpp - 1); }
      else { pidx = (int)__umulhi((unsigned)h, p.hpp_magic); s16 = h - pidx * hpp; }
      const int a0 = __shfl(pg0, pidx & 63), a1 = __shfl(pg1, pidx & 63);
      const int64_t pg = pidx < 64 ? a0 : a1;
      k_at = (uint64_t)(kbase + pg * ksp + (int64_t)(s16 * 16) * kss);
      v_at = (uint64_t)(vbase + pg * vsp + (int64_t)(s16 * 16) * vss);
    }
    auto at_step = [&](uint64_t v, int ss) -> const char* {
      const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, ss), hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), ss);
      uint64_t at = ((uint64_t)hi << 32) | lo;
      // A vector memory instruction may read a scalar register 5 wait states after a vector instruction wrote it. The
      // compiler keeps that distance for loads it sees; load_to_lds it does not see.
      asm volatile("s_nop 4" : "+s"(at));
      return (const char*)at;
    };
    auto fetch_k = [&](int ss) {
      const char* base = at_step(k_at, ss);
      const unsigned dst = lds_base + (unsigned)(ss & 1) * STAGE2;
      // (rows past the end of the piece re-read its last token: their scores are masked)
      const int left = last_rel_u - ss * SST - wave_u * 16;
      if (left >= 15) {
#pragma unroll
        for (int i = 0; i < NI; ++i) load_to_lds(base, koff[i], dst + i * 1024);
      } else {
        const int lim = left < 0 ? last_rel_u & 15 : left;
#pragma unroll
        for (int i = 0; i < NI; ++i) load_to_lds(base, RPI * i + r_in > lim ? (unsigned)(lim * kss) + k_piece(i) : koff[i], dst + i * 1024);
      }
    };
    auto fetch_v = [&](int ss) {
      const char* base = at_step(v_at, ss);
      const unsigned dst = lds_base + (unsigned)(ss & 1) * STAGE2 + KTILE;
      const int left = last_rel_u - ss * SST - wave_u * 16;
      if (left >= 15) {
#pragma unroll
        for (int i = 0; i < NI; ++i) load_to_lds(base, voff[i], dst + i * 1024);
      } else {
        const int lim = left < 0 ? last_rel_u & 15 : left;
#pragma unroll
        for (int i = 0; i < NI; ++i) load_to_lds(base, RPI * i + r_in > lim ? (unsigned)(lim * vss) + v_piece : voff[i], dst + i * 1024);
      }
    };

    // LDS offsets of this lane's operand reads inside a stage (token 0 of the stage; + 32 ROWB for tokens 32..). Those of kk and db differ from
    // those of 0 in the place inside the row alone, which is an exclusive or with 32 kk and 64 db (the stages start at multiples of a
    // row). Two offsets instead of twelve, 10 registers less, where those count: with tails or lists, and at head_dim 64, where 128 registers
    // are a fourth workgroup per CU (102 requests over 4848 tokens, 580..1160 of their own, at 32/8 heads 49.0 us, with twelve 54.3). Elsewhere
    // the sum ahead of the exclusive or is one more wait for each read (34 tall boxes in 170 workgroups 15.39 / 15.33, 64 requests behind one prefix
    // 21.81 / 21.71).
    constexpr bool TWO_OFFSETS = TAILS || LISTS || D == 64;
    constexpr int KRD = TWO_OFFSETS ? 1 : KK2, VRD = TWO_OFFSETS ? 1 : DB2;
    unsigned k_rd[KRD], v_rd[VRD];
#pragma unroll
    for (int kk = 0; kk < KRD; ++kk)
      k_rd[kk] = (unsigned)(n32 * ROWB + ((2 * kk + h2) ^ (D == 128 ? n32 & 15 : (n32 >> 1) & 7)) * 16);
#pragma unroll
    for (int db = 0; db < VRD; ++db)
      v_rd[db] = (unsigned)(KTILE + (h2 * 4 + (n >> 2)) * ROWB + (db ^ (D == 128 ? n >> 2 : (n >> 3) & 1)) * 64 + (g & 1) * 32 + (n & 3) * 8);
    auto k_row = [&](const PAT_LDS char* stage, int kk) -> const PAT_LDS char* {
      if constexpr (TWO_OFFSETS) return (const PAT_LDS char*)(size_t)(((unsigned)(size_t)stage + k_rd[0]) ^ (kk * 32u));
      else return stage + k_rd[kk];
    };
    auto v_row = [&](const PAT_LDS char* stage, int db) -> const PAT_LDS char* {
      if constexpr (TWO_OFFSETS) return (const PAT_LDS char*)(size_t)(((unsigned)(size_t)stage + v_rd[0]) ^ (db * 64u));
      else return stage + v_rd[db];
    };

    // HALVES x 32 tokens of online-softmax attention for this wave's 32 rows; `stage` points at the first of them
    // (its K rows; the V rows KTILE further), t0 is that token's place in the piece. First the scores and probabilities ...
    auto score32 = [&](auto halves_c, vec8 (&pv)[2 * decltype(halves_c)::value], const PAT_LDS char* stage, int t0) {
      constexpr int HALVES = decltype(halves_c)::value;
      f32x16 s[HALVES];
      // every K operand of a half is requested before the first MFMA waits for one (left alone, the
      // compiler reads each operand right ahead of its use and exposes the LDS latency KK2 times)
#pragma unroll
      for (int a = 0; a < HALVES; ++a) {
        vec8 kop[KK2];
#pragma unroll
        for (int kk = 0; kk < KK2; ++kk)
          kop[kk] = *(const PAT_LDS vec8*)(k_row(stage, kk) + a * 32 * ROWB);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 16; ++i) s[a][i] = 0.f;
#pragma unroll
        for (int kk = 0; kk < KK2; ++kk) s[a] = E::mfma32(kop[kk], __builtin_bit_cast(vec8, q2[kk]), s[a]);
      }
      // The rows' reference maxima move only when some row's maximum has left a window of kLazy
      // (base-2 exponent units) above its reference: probabilities then reach 2^kLazy at most, which
      // fp32 sums and 16-bit P hold as well as values below 1, and the accumulator is rescaled a few
      // times per piece instead of at nearly every step (with 32 rows per wave some row's maximum
      // moves at almost every step).
      constexpr float kLazy = 8.f;
      if (t0 + HALVES * kStepTokens > ntok_u) {
        // the piece's last step: tokens past its end are masked
#pragma unroll
        for (int a = 0; a < HALVES; ++a)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (t0 + a * kStepTokens + (i >> 2) * 8 + h2 * 4 + (i & 3) >= ntok_u) s[a][i] = neg_inf();
      }
      float mx = s[0][0];
#pragma unroll
      for (int a = 0; a < HALVES; ++a)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[a][i]);
      mx = max_xor32(mx) * sc_abs;
      if (__builtin_amdgcn_ballot_w64(mx > m_run + kLazy) != 0) {
        asm volatile("" ::: "memory");   // a real branch: if-converted, the skipped multiplies come back as selects
        const float m_new = fmaxf(m_run, mx);
        const float alpha = fast_exp2(m_run - m_new);   // (first step: m_run = -inf, alpha = 0)
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int db = 0; db < DB2; ++db) acc2[db] = acc2[db] * alpha;
      }
      float psum[2] = {0.f, 0.f};
#pragma unroll
      for (int a = 0; a < HALVES; ++a)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float e = fast_exp2(__builtin_fmaf(s[a][i], sc_abs, -m_run));
          psum[i & 1] += e;
          pv[2 * a + (i >> 3)][i & 7] = (T)e;
        }
      l_run += psum[0] + psum[1];
    };
    // ... then the weighted sum of the V rows.
    auto gather32 = [&](auto halves_c, const vec8 (&pv)[2 * decltype(halves_c)::value], const PAT_LDS char* stage) {
      constexpr int HALVES = decltype(halves_c)::value;
      auto read_v = [&](int t, s16x8 (&v)[DB2]) {
#pragma unroll
        for (int db = 0; db < DB2; ++db) {
          const PAT_LDS char* src = v_row(stage, db) + t * 16 * ROWB;
          s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PAT_LDS s16x4*)src);
          s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((PAT_LDS s16x4*)(src + 8 * ROWB));
          v[db] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
      };
      s16x8 vop[2][DB2];
      read_v(0, vop[0]);
      read_v(1, vop[1]);
#pragma unroll
      for (int t = 0; t < 2 * HALVES; ++t) {
#pragma unroll
        for (int db = 0; db < DB2; ++db) acc2[db] = E::mfma32(__builtin_bit_cast(vec8, vop[t & 1][db]), pv[t], acc2[db]);
        if (t + 2 < 2 * HALVES) read_v(t + 2, vop[t & 1]);
      }
    };

    // A stage's K and V tiles are handed over together or apart (p.tall_apart, the host's choice). Together: one barrier
    // per super-step, the next super-step's tiles are in flight for one step. Apart, half a step from each other: the K
    // tile of step ss + 2 is requested as soon as every wave has read its K operands of step ss, the V tile of step ss + 1
    // as soon as everybody has left step ss - 1; either is then in flight for a step and a half, at the price of a
    // second barrier per step.
    const bool apart = p.tall_apart != 0;
    fetch_k(0);
    fetch_v(0);
    // Q has to be there before the next load into LDS is issued (the first ones follow it right away): a wait for it
    // inside the loop would, loads returning in order, wait for the super-step in flight as well.
#pragma unroll
    for (int kk = 0; kk < KK2; ++kk) asm volatile("" : "+v"(q2[kk]));
    if (apart && nss_u > 1) fetch_k(1);
    // (loops of their own: in one loop the operands of both splits of the waves take 60 more registers, and a second
    // barrier that is only sometimes there keeps the V reads from being issued ahead of the softmax)
    auto walk = [&](auto halves_c, auto apart_c) {
      constexpr bool kApart = decltype(apart_c)::value;
      vec8 pv[2 * decltype(halves_c)::value];
      for (int ss = 0; ss < nss_u; ++ss) {
        const bool more = ss + 1 < nss_u;
        // this wave's part of the tiles has arrived (apart: of the K tile; the V tile and the next K tile were requested after it), ...
        if (!kApart) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NI) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NI) : "memory");
        __syncthreads();   // ... everybody's has, and nobody reads the other stage (apart: its V rows) any more
        if (more) {
          if (!kApart) fetch_k(ss + 1);
          fetch_v(ss + 1);
        }
        const int t0 = ss * SST + ph * kStepTokens;
        const PAT_LDS char* stage = (const PAT_LDS char*)smem + (ss & 1) * STAGE2 + ph * 32 * ROWB;
        const bool mine = has_rows && t0 < ntok_u;
        if constexpr (kApart) {
          if (mine) score32(halves_c, pv, stage, t0);
          if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NI) : "memory");
          else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          __syncthreads();   // the V tile is there, and nobody reads this stage's K rows any more
          if (ss + 2 < nss_u) fetch_k(ss + 2);
          if (mine) gather32(halves_c, pv, stage);
        } else if (mine) {
          score32(halves_c, pv, stage, t0);
          gather32(halves_c, pv, stage);
        }
      }
    };
    if (one_tile_per_wave) {
      if (apart) walk(std::integral_constant<int, 2>{}, std::true_type{});
      else walk(std::integral_constant<int, 2>{}, std::false_type{});
    } else {
      if (apart) walk(std::integral_constant<int, 1>{}, std::true_type{});
      else walk(std::integral_constant<int, 1>{}, std::false_type{});
    }
    if constexpr (TAILS) {
      __syncthreads();   // (every wave is done with the stages)
      walk_tails();
    }
    l_run = sum_xor32(l_run);
    if (one_tile_per_wave) {
      if (my_slot0 >= 0) {
        const int64_t prow = (int64_t)my_slot0;
        const float inv = 1.f / l_run;
        float* dst = p.o_part + prow * D + h2 * 4;
        T* o = direct ? row_out(my_slot0) + h2 * 4 : nullptr;
#pragma unroll
        for (int db = 0; db < DB2; ++db)
#pragma unroll
          for (int b = 0; b < 4; ++b)
            put4(dst + db * 32 + b * 8, o + db * 32 + b * 8,
                 f32x4{acc2[db][4 * b], acc2[db][4 * b + 1], acc2[db][4 * b + 2], acc2[db][4 * b + 3]} * inv);
        if (h2 == 0) put_lse(prow, (m_run + __builtin_amdgcn_logf(l_run)) * 0.6931471805599453f);
      }
      return;
    }
    // ---- the two wave pairs' states of the same rows are combined through LDS ----------------
    float* xbuf = (float*)smem;                 // [rt][DB2 * 4 pieces][64 lanes] x 16 bytes
    __syncthreads();                            // every wave is done with the stages
    if (ph == 1 && has_rows) {
#pragma unroll
      for (int db = 0; db < DB2; ++db)
#pragma unroll
        for (int b = 0; b < 4; ++b)
          *(f32x4*)(xbuf + (((rt * DB2 + db) * 4 + b) * 64 + lane) * 4) =
              f32x4{acc2[db][4 * b], acc2[db][4 * b + 1], acc2[db][4 * b + 2], acc2[db][4 * b + 3]};
      if (h2 == 0) { s_m[rt * 32 + n32] = m_run; s_l[rt * 32 + n32] = l_run; }
    }
    __syncthreads();
    if (ph == 0 && has_rows && my_slot0 >= 0) {
      const float m1 = s_m[rt * 32 + n32], l1 = s_l[rt * 32 + n32];   // (a pair without steps: -inf, 0)
      const float mm = fmaxf(m_run, m1);
      const float w0 = fast_exp2(m_run - mm), w1 = fast_exp2(m1 - mm);
      const float lsum = l_run * w0 + l1 * w1;
      const float a0 = w0 / lsum, a1 = w1 / lsum;
      const int64_t prow = (int64_t)my_slot0;
      float* dst = p.o_part + prow * D + h2 * 4;
      T* o = direct ? row_out(my_slot0) + h2 * 4 : nullptr;
#pragma unroll
      for (int db = 0; db < DB2; ++db)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const f32x4 x = *(const f32x4*)(xbuf + (((rt * DB2 + db) * 4 + b) * 64 + lane) * 4);
          const f32x4 mine = f32x4{acc2[db][4 * b], acc2[db][4 * b + 1], acc2[db][4 * b + 2], acc2[db][4 * b + 3]};
          put4(dst + db * 32 + b * 8, o + db * 32 + b * 8, mine * a0 + x * a1);
        }
      if (h2 == 0) put_lse(prow, (mm + __builtin_amdgcn_logf(lsum)) * 0.6931471805599453f);
    }
    }   // TALLK
  } else if (LISTS && (mode & kRecordModeList)) {
    // ====================== several short boxes: each wave walks them all for its kv head ======================
    // Launches of more short private boxes than places (a step of K and V each, the requests' own ends): a workgroup of one of
    // them is 4-5 us of launch, record, page ids and first tiles for 0.5 us of work, and the boxes beyond the places wait for as
    // long again. Here that is paid once per list, and a further box costs 2-2.5 us, a trip to memory of which its neighbour's
    // arithmetic covers part (512 requests of 1408 + 32 tokens at 16/8 heads: 30.6 us per call, 27.3 in lists of four).
    const int count = ntok_u, pages = p.list_pages, most = p.list_boxes;
    const int seq_l = lane < count ? rows_tab[min(lane, record_max_seqs - 1)] : -1;
    const int slot_l = lane < count ? rows_tab[record_max_seqs + min(lane, record_max_seqs - 1)] : -1;
    // (the record's page entries: the boxes' tokens, then their pages)
    const uint64_t live = __builtin_amdgcn_ballot_w64(lane < count && pg0 > 0 && seq_l >= 0);
    auto slot_of = [&](int j) {   // the first partial slot of box j's row n
      const int seq = __builtin_amdgcn_readlane(seq_l, j), sl = __builtin_amdgcn_readlane(slot_l, j);
      return seq >= 0 && sl >= 0 && n < G ? (int64_t)(seq * p.heads + head * G + n) * p.num_slots + sl : (int64_t)-1;
    };
    for (int j = 0; j < count; ++j) {   // slots that stay empty
      const int64_t at = slot_of(j);
      if (g == 0 && at >= 0)
        for (int c = __builtin_amdgcn_readlane(pg0, j) > 0 ? 1 : 0; c < fill_end; ++c) p.lse_part[at + c] = neg_inf();
    }
    if (live != 0)
      walk_list(live, [&](int j) { return __builtin_amdgcn_readlane(pg0, j); },
                [&](int j, int page) { return __builtin_amdgcn_readlane(pg0, most + j * pages + page); },
                [&](int j) { return __builtin_amdgcn_readlane(seq_l, j); }, (PAT_LDS char*)smem + wave * WSTAGE, [&](int j, float m_t, float l_t) {
        const int64_t at = slot_of(j);
        if (at >= 0) {
          const float inv = 1.f / l_t;
          float* dst = p.o_part + at * D + g * 4;
#pragma unroll
          for (int db = 0; db < DB; ++db) *(f32x4*)(dst + db * 16) = acc_o[db] * inv;
          if (g == 0) p.lse_part[at] = (m_t + __builtin_amdgcn_logf(l_t)) * 0.6931471805599453f;
        }
      });
  } else {
    // ====================== short box: KV steps split over the 4 waves ========================
    // Each wave holds one step's K and V in registers and refills either as soon as it has been consumed: V when it has gone to
    // LDS, K behind the score MFMAs. (Two steps in registers, 243 VGPRs: no faster where the memory system is full.)
    load_q();
    // K rows go straight into MFMA operand layout (16 rows x 64 bytes per load instruction); V rows
    // are fetched TPL whole rows per instruction and staged in this wave's LDS region. (Staging K
    // the same way and reading operands back from LDS was measured: no faster, twice the LDS.)
    PAT_LDS char* vstage = (PAT_LDS char*)smem + wave * WSTAGE;
    const unsigned koff = (unsigned)(n * kss) + g * 16;                          // K: row n of a half, dims g*8..
    const unsigned voff = (unsigned)((lane / CPR) * vss) + (lane % CPR) * 16;    // V: TPL rows per instruction
    auto fetch_v = [&](int st, u32x4 (&vd)[NV], auto stream_c) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        int lim;
        const int h = half_geom(__builtin_amdgcn_readfirstlane(st * 2 + a), lim);
        const char* vb = half_base(vbase, vsp, vss, h);
#pragma unroll
        for (int j = 0; j < NV / 2; ++j) {
          unsigned vo = voff + (unsigned)(j * TPL) * (unsigned)vss;
          if (lim < 15 && j * TPL + lane / CPR > lim) vo = (unsigned)(lim * vss) + (lane % CPR) * 16;
          const u32x4* at = (const u32x4*)(vb + vo);
          vd[a * (NV / 2) + j] = decltype(stream_c)::value ? __builtin_nontemporal_load(at) : *at;
        }
      }
    };
    auto fetch_k = [&](int st, u32x4 (&kd)[2][KK]) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        int lim;
        const int h = half_geom(__builtin_amdgcn_readfirstlane(st * 2 + a), lim);
        const char* kb = half_base(kbase, ksp, kss, h);
        unsigned ko = koff;
        if (lim < 15 && n > lim) ko = (unsigned)(lim * kss) + g * 16;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) kd[a][kk] = *(const u32x4*)(kb + ko + kk * 64);
      }
    };
    // steps of this wave: every kWaves-th one of the chunk, or, with a kv head per wave, all of them
    const int step0 = head_per_wave ? 0 : wave;
    const int stride = head_per_wave ? 1 : WAVES;
    auto walk = [&](auto stream_c) {
      u32x4 kd[2][KK], vd[NV];
      fetch_v(step0, vd, stream_c);
      fetch_k(step0, kd);
      // Q is here before the loop starts, and the last step, which requests nothing, stands apart from it: every wait inside
      // then counts exactly the loads behind the one it is for. In one loop with Q on its way and requests that may not be made,
      // the score MFMAs of every step waited for the V tile requested just ahead of them (fp16, 8 kv heads: 123 requests over
      // 240 + 224 tokens 17.0 us, now 15.6; head_dim 64, 48 over 768 11.7 / 10.2; 32 x 4096 at 64/8 heads 96.0 / 94.6).
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) asm volatile("" : "+v"(qreg[kk]));
      auto step = [&](int st, auto more_c) {
        constexpr bool more = decltype(more_c)::value;
        // V tile -> this wave's LDS region, row-major with padded rows; its registers are free again at once and take the
        // next V tile
#pragma unroll
        for (int j = 0; j < NV; ++j)
          *(PAT_LDS u32x4*)(vstage + (j * TPL + lane / CPR) * RSV + (lane % CPR) * 16) = vd[j];
        if (more) fetch_v(st + stride, vd, stream_c);
        // Few tall workgroups with long chains (p.tall_apart): the launch ends on those, and these waves' requests, of two
        // steps at once, hold theirs up (us per call without / with this wait: 64 requests over 2048 tokens, 32/8 heads, 22.8 /
        // 22.0, 32 over 16384 at 64/8 57.6 / 56.3). Of 125 launches of this form measured both ways the 35 such are 1.4 %
        // slower without it, the other 90 1.6 % faster, 37 x (848 + 239..478) at 32/8 heads 19 %.
        if constexpr (more && TALLK == 32) {
          if (p.tall_apart) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        // the K registers are refilled as soon as the score MFMAs have read them
        attend([&](int a, int kk) { return __builtin_bit_cast(vec8, kd[a][kk]); }, vstage,
               t_begin + st * kStepTokens, t_end, m_run, l_run, [&]() { if (more) fetch_k(st + stride, kd); });
      };
      int st = step0;
      for (; st + stride < nsteps; st += stride) step(st, std::true_type{});
      step(st, std::false_type{});
    };
    // (V past the caches: for launches of 92 MB and more, the records say which pieces; 1-15 % faster there. A loop of its own: inside one
    // loop the two kinds of load are either merged, without the hint, or cost 3 % as a branch; and a branch known to be uniform
    // costs 28 spilled registers, like uniform loop bounds above)
    if (step0 < nsteps) {
      if constexpr (STREAM) {
        int past = mode & kRecordModeStreamV;
        asm volatile("" : "+v"(past));
        if (past) walk(std::true_type{});
        else walk(std::false_type{});
      } else {
        walk(std::false_type{});
      }
    }
    l_run = sum_xor32(sum_xor16(l_run));

    if (head_per_wave) {
      // the wave has seen the whole chunk of its head: its rows go out as they are
      if (my_slot0 >= 0) {
        const int64_t prow = (int64_t)my_slot0;
        const float inv = 1.f / l_run;
        float* dst = p.o_part + prow * D + g * 4;
        T* o = direct ? row_out(my_slot0) + g * 4 : nullptr;
#pragma unroll
        for (int db = 0; db < DB; ++db) put4(dst + db * 16, o + db * 16, acc_o[db] * inv);
        if (g == 0) put_lse(prow, (m_run + __builtin_amdgcn_logf(l_run)) * 0.6931471805599453f);
      }
    } else {
    // combine the 4 waves' states through LDS and write the partial
    float* cbuf = (float*)smem;
    constexpr int COLS = 16 * D / (WAVES * 64) > 4 ? 16 * D / (WAVES * 64) : 4;   // columns a thread finalises
    constexpr int TPR = D / COLS;               // threads a row
    const int crow = (int)((unsigned)tid / TPR);          // row this thread finalises (past 16: none)
    const int ccol = (int)((unsigned)tid % TPR) * COLS;   // its first column
    __syncthreads();  // every wave is done with its staging region
    if (g == 0) { s_m[wave * 16 + n] = m_run; s_l[wave * 16 + n] = l_run; }
#pragma unroll
    for (int db = 0; db < DB; ++db)
      *(f32x4*)(cbuf + (wave * 16 + n) * OROW + db * 16 + g * 4) = acc_o[db];
    __syncthreads();

    // the slot of row crow sits in lane crow of every wave
    const int cslot0 = __shfl(my_slot0, WAVES * 64 > 16 * TPR ? crow & 15 : crow);
    if (cslot0 >= 0 && (WAVES * 64 == 16 * TPR || crow < 16)) {
      float mw[WAVES], mmax = neg_inf();
#pragma unroll
      for (int w = 0; w < WAVES; ++w) { mw[w] = s_m[w * 16 + crow]; mmax = fmaxf(mmax, mw[w]); }
      float wsum = 0.f, wgt[WAVES];
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        wgt[w] = fast_exp2(mw[w] - mmax);   // a wave without steps has m = -inf -> weight 0
        wsum += wgt[w] * s_l[w * 16 + crow];
      }
      const float inv = 1.f / wsum;
      const int64_t prow = (int64_t)cslot0;
      float* dst = p.o_part + prow * D + ccol;
      T* od = direct ? row_out(cslot0) + ccol : nullptr;
#pragma unroll
      for (int c = 0; c < COLS; c += 4) {
        f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WAVES; ++w)
          o += *(const f32x4*)(cbuf + (w * 16 + crow) * OROW + ccol + c) * wgt[w];
        put4(dst + c, od + c, o * inv);
      }
      if (ccol == 0)
        put_lse(prow, (mmax + __builtin_amdgcn_logf(wsum)) * 0.6931471805599453f);
    }
    }   // combine
  }
}

// Host launcher: picks the instance for (element type, head_dim, single-slot launch, form of the tall path, V past the caches, tails).
typedef void (*SplitFn)(const char*, int, int, int, const SplitParams);
template <bool DIRECT, int TALLK, bool STREAM, bool TAILS = false, int WAVES = kWaves>
static SplitFn split_instance(bool bf16, int head_dim) {
  if (bf16) return head_dim == 64 ? pat_split_kernel<__bf16, 64, DIRECT, TALLK, STREAM, TAILS, WAVES, false> : pat_split_kernel<__bf16, 128, DIRECT, TALLK, STREAM, TAILS, WAVES, false>;
  return head_dim == 64 ? pat_split_kernel<_Float16, 64, DIRECT, TALLK, STREAM, TAILS, WAVES, false> : pat_split_kernel<_Float16, 128, DIRECT, TALLK, STREAM, TAILS, WAVES, false>;
}
template <bool STREAM>
static SplitFn split_instance(bool bf16, int head_dim, bool direct, bool t32) {
  if (direct) return t32 ? split_instance<true, 32, STREAM>(bf16, head_dim) : split_instance<true, 16, STREAM>(bf16, head_dim);
  return t32 ? split_instance<false, 32, STREAM>(bf16, head_dim) : split_instance<false, 16, STREAM>(bf16, head_dim);
}

hipError_t launch_split(bool bf16, int head_dim, hipStream_t stream, const SplitParams& params) {
  const bool t32 = params.tall_rows != 16, direct = params.direct != 0;
  const bool past = params.stream_v != 0, tails = params.tail_pages > 0, lists = params.list_boxes > 0;
  const int waves = params.waves;
  // Eight waves: launches without tall boxes, at head_dim 64 those that write `out`. Lists: the 32-row form at head_dim 128, partial rows.
  // Tails: the 32-row form. None of them with another or with V past the caches: there is no such instance.
  if ((waves != kWaves && waves != 8) || (waves == 8 && (past || tails || lists || (!direct && head_dim != 128))) ||
      (lists && (past || tails || direct || !t32 || head_dim != 128)) || (tails && (past || !t32)))
    return hipErrorInvalidValue;
  SplitFn fn = waves == 8 ? (direct ? split_instance<true, 0, false, false, 8>(bf16, head_dim)
                           : bf16 ? pat_split_kernel<__bf16, 128, false, 0, false, false, 8, false> : pat_split_kernel<_Float16, 128, false, 0, false, false, 8, false>)
             : lists ? (bf16 ? pat_split_kernel<__bf16, 128, false, 32, false, false, kWaves, true> : pat_split_kernel<_Float16, 128, false, 32, false, false, kWaves, true>)
             : tails ? (direct ? split_instance<true, 32, false, true>(bf16, head_dim) : split_instance<false, 32, false, true>(bf16, head_dim))
             : past ? split_instance<true>(bf16, head_dim, direct, t32) : split_instance<false>(bf16, head_dim, direct, t32);
  const unsigned lds = (unsigned)split_smem_bytes(head_dim, waves != kWaves ? 0 : t32 ? 32 : 16, waves);
  // more dynamic LDS than the default limit of a kernel: raised once per instance and device
  {
    static std::mutex mutex;
    static bool raised[64][256] = {{false}};
    int dev = 0;
    if (const hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
    const int inst = (lists ? 128 : 0) + (waves == 8 ? 64 : 0) + (tails ? 32 : 0) + (past ? 16 : 0) + (t32 ? 8 : 0) + (bf16 ? 4 : 0) + (head_dim == 128 ? 2 : 0) + (direct ? 1 : 0);
    std::lock_guard<std::mutex> lock(mutex);
    if (dev >= 0 && dev < 64 && !raised[dev][inst]) {
      if (const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
          e != hipSuccess)
        return e;
      raised[dev][inst] = true;
    }
  }
  const unsigned wgs = (unsigned)params.total_items;
  const dim3 grid(wgs < (unsigned)kGridX ? wgs : (unsigned)kGridX, (wgs + kGridX - 1) / kGridX);
  hipLaunchKernelGGL(fn, grid, dim3((unsigned)waves * 64u), lds, stream, params.records, params.record_stride, params.record_max_seqs,
                     params.record_max_pages, params);
  return hipGetLastError();
}

}  // namespace pat
