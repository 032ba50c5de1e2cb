// Paged prefill attention for gfx950 (MI355X), wave64 + MFMA.
//
// Math (AttentionBackendGPU.prefill_attention,
// mini_vllm/attention/paged_attention_gpu.py:577-661): for every prefill
// sequence with `cached` tokens already in the pool and a chunk of
// `q_len` new tokens,
//   keys 0 .. cached-1     from the pool (table row `seq_indices[i]`),
//   keys cached .. +q_len  from the chunk's own key / value rows,
//   out[t, hq] = softmax_j<=cached+t(scale * q[t, hq] . k_j) v_j,
// kv head hk = hq / n_rep, scale = head_dim^-1/2 -- the reference's
// gather + cat + repeat_interleave + masked SDPA, in one pass over the
// keys with no gathered copy.
//
// Work decomposition: one work group per (sequence, kv head, block of query
// tokens); its MFMA rows are the GQA group's query heads of its tokens, so
// one K/V pass serves them all. The waves share one stream of keys, staged
// from HBM straight to LDS (global_load_lds, XOR piece swizzle as in the
// decode kernel), one barrier per stage, two stages in flight:
//   * prefix keys are addressed through the sequence's block ids, staged
//     in LDS per window of kPfIdCap blocks; chunk keys through the chunk's
//     row strides (q / k / v may be views of one fused QKV output).
// The 16-bit types run on 32x32x16 MFMAs (mv_prefill16.h); fp32 on the
// kernel below: a wave owns 16 MFMA rows (floor(16 / n_rep) tokens), a stage
// is one 16-key sub-tile per wave, every wave computes S^T = K Q^T, the
// per-row causal mask, the online softmax (once per stage) and O += P V.
//
// Key split (mv_paged_prefill_parts): when a launch has fewer (sequence, kv
// head, token block) units than the device has CUs, the host cuts a unit's
// keys into parts at stage boundaries, one work group each. A part leaves
// its rows' normalised O and (max, sum) in a workspace with device-coherent
// stores and counts itself on the unit's counter; the work group that
// completes the count folds the parts in part order (log-sum-exp) and
// writes the rows, so the result does not depend on which part finishes
// last.
#include <algorithm>
#include <climits>
#include <cstring>
#include <memory>
#include <new>

#include "mv_prefill.h"
#include "mv_prefill16.h"

namespace mv {
namespace {

// fp32: 8 waves per work group where two stages of 8 sub-tiles fit the LDS,
// else 4 (head_dim 128).
template <int D>
struct Prefill32Traits : TileGeom<MV_DTYPE_F32, D> {
  using G = TileGeom<MV_DTYPE_F32, D>;
  static constexpr int kSubBytes = 2 * G::kTileBytes;  // K and V sub-tile of one wave
  static constexpr int kWaves = 2 * 8 * kSubBytes + kPfIdCap * 4 <= 160 * 1024 ? 8 : 4;
  static constexpr int kStageTokens = kWaves * kTile;
  static constexpr int kStageBytes = kWaves * kSubBytes;
  static constexpr int kIdsOffset = 2 * kStageBytes;
  static constexpr int kLdsBytes = kIdsOffset + kPfIdCap * 4;
  static_assert(kLdsBytes <= 160 * 1024 - 64, "LDS of one work group");
};

template <int D, typename BT>
__device__ __forceinline__ void prefill32(const PrefillArgs& a) {
  using Tr = Prefill32Traits<D>;
  constexpr int DTYPE = MV_DTYPE_F32;
  constexpr int L = Tr::kLoads;
  constexpr int RP = Tr::kRowPieces;
  constexpr int QP = Tr::kLanePieces;
  constexpr int W = Tr::kWaves;

  __shared__ __attribute__((aligned(16))) char s_lds[Tr::kLdsBytes];
  int32_t* s_ids = reinterpret_cast<int32_t*>(s_lds + Tr::kIdsOffset);
  const uint32_t lds0 = lds_address(s_lds);

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int t = lane & 15;  // MFMA: key row (K operand) / query row (results)
  const int g = lane >> 4;  // MFMA: dim quarter (K operand) / key quad (results)

  const PrefillItem it = load_item(a);
  if (!it.ok) return;
  const int h = it.h, tok0 = it.tok0, ntok = it.ntok;
  const int64_t row = a.seqs[4 * it.seq];
  const int cached = static_cast<int>(a.seqs[4 * it.seq + 1]);
  const int64_t chunk_row0 = a.seqs[4 * it.seq + 2];
  const int64_t qbase = chunk_row0 + tok0;  // chunk row of token tok0
  // keys of this work group: [kb0, key_end); the rows see keys below
  // cached + tok0 + ntok, and a part ends at a stage boundary below that
  const int key_end = min(cached + tok0 + ntok, it.kb1);

  // ---- rows of this wave: limits and Q (registers, straight from HBM)
  const int tpw = 16 / a.n_rep;
  const int wtok0 = wave * tpw;
  const int wtok_end = min(ntok, wtok0 + tpw);
  // the last key any row of the wave sees (-1: the wave has no rows)
  const int wave_limit = wtok0 < ntok ? cached + tok0 + wtok_end - 1 : -1;
  int limit;
  uint4 qr[QP];
  {
    const int rtok = wtok0 + t / a.n_rep;
    const bool ok = t < tpw * a.n_rep && rtok < ntok;
    limit = ok ? cached + tok0 + rtok : -1;  // -1: a padding row, never written
    const char* qrow = reinterpret_cast<const char*>(static_cast<const float*>(a.q) +
                                                     (qbase + (ok ? rtok : 0)) * a.q_st +
                                                     (h * a.n_rep + (ok ? t % a.n_rep : 0)) * a.q_sh);
#pragma unroll
    for (int c = 0; c < QP; ++c) {
      qr[c] = *reinterpret_cast<const uint4*>(qrow + (g * QP + c) * 16);
      // a padding row's Q is zero: finite scores, never written
      if (!ok) qr[c] = uint4{0, 0, 0, 0};
    }
  }
  // Q must have landed before the tile copies are counted by vmcnt.
#pragma unroll
  for (int c = 0; c < QP; ++c) asm volatile("" ::"v"(qr[c].x), "v"(qr[c].y), "v"(qr[c].z), "v"(qr[c].w));

  float m_run = kNegInf, l_run = 0.f;
  f32x4 o[1][D / 16];
#pragma unroll
  for (int c = 0; c < D / 16; ++c) o[0][c] = f32x4{0.f, 0.f, 0.f, 0.f};

  SubTileCopy<DTYPE, D> copy{a, s_ids, h, cached, key_end, chunk_row0, lane, {}, {}, {}};
  copy.init();
  int win_blk0 = 0;
  auto issue = [&](int k, int st) __attribute__((always_inline)) -> unsigned {
    const int kb = k * Tr::kStageTokens + wave * kTile;
    return copy.copy(kb, win_blk0, lds0 + st * Tr::kStageBytes + wave * Tr::kSubBytes, copy.block_id_of(kb, win_blk0));
  };
  // V slots of keys that were not loaded read pool row 0 instead: zero
  // them (P is 0 there, but 0 * NaN would not be).
  auto zero_invalid_v = [&](int st, unsigned valid) __attribute__((always_inline)) {
    char* vdst = s_lds + st * Tr::kStageBytes + wave * Tr::kSubBytes + Tr::kTileBytes;
#pragma unroll
    for (int c = 0; c < L; ++c)
      if (!((valid >> c) & 1u)) *reinterpret_cast<uint4*>(vdst + c * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
  };

  // One stage for this wave's rows, over its W sub-tiles of 16 keys: S^T for
  // every sub-tile some row sees, one mask + max + rescale for the whole
  // stage, then the P V updates. Key limits are increasing in the row, so
  // sub-tiles past the last row's limit are skipped.
  auto compute_stage = [&](int k, int st) __attribute__((always_inline)) {
    const int k_first = k * Tr::kStageTokens;
    if (k_first > wave_limit) return;
    const int nu = min(W, (wave_limit - k_first) / kTile + 1);
    const char* stage = s_lds + st * Tr::kStageBytes;
    const int ksw = piece_swizzle<RP>(t);
    f32x4 acc[W];
    // Head_dim 64: a stage all of whose sub-tiles are seen branches on none of
    // them, so their K reads and MFMAs overlap (16 x (2000 + 1) at 8 / 8 heads
    // 56.4 -> 52.8 us, 16 x (500 + 300) 101 -> 97); at 128, with 4 waves, it
    // gave 1 % either way.
    if (D == 64 && nu == W) {
#pragma unroll
      for (int u = 0; u < W; ++u) {
        acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        const char* k_tile = stage + u * Tr::kSubBytes;
#pragma unroll
        for (int c = 0; c < QP; ++c)
          acc[u] = mfma_qk<DTYPE>(
              *reinterpret_cast<const uint4*>(k_tile + (t * RP + ((g * QP + c) ^ ksw)) * 16), qr[c], acc[u]);
      }
    } else {
#pragma unroll
      for (int u = 0; u < W; ++u) {
        acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (u < nu) {
          const char* k_tile = stage + u * Tr::kSubBytes;
#pragma unroll
          for (int c = 0; c < QP; ++c)
            acc[u] = mfma_qk<DTYPE>(
                *reinterpret_cast<const uint4*>(k_tile + (t * RP + ((g * QP + c) ^ ksw)) * 16), qr[c], acc[u]);
        }
      }
    }
    float pr[W][1][4];
    float mc = kNegInf;
#pragma unroll
    for (int u = 0; u < W; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = k_first + u * kTile + 4 * g + e;
        const float sv = u < nu && key <= limit ? acc[u][e] * a.scale_log2 : kNegInf;
        acc[u][e] = sv;
        mc = fmaxf(mc, sv);
      }
    mc = fmaxf(mc, __shfl_xor(mc, 16));
    mc = fmaxf(mc, __shfl_xor(mc, 32));
    const float m_new = fmaxf(m_run, mc);
    const float m_ref = m_new == kNegInf ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_ref);
    float lc = 0.f;
#pragma unroll
    for (int u = 0; u < W; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        pr[u][0][e] = __builtin_amdgcn_exp2f(acc[u][e] - m_ref);
        lc += pr[u][0][e];
      }
    lc += __shfl_xor(lc, 16);
    lc += __shfl_xor(lc, 32);
    l_run = l_run * alpha + lc;
    m_run = m_new;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float ar = __shfl(alpha, 4 * g + e);
#pragma unroll
      for (int c = 0; c < D / 16; ++c) o[0][c][e] *= ar;
    }
#pragma unroll
    for (int u = 0; u < W; ++u)
      if (u < nu) mfma_pv_rows<DTYPE, D, 1>(pr[u], stage + u * Tr::kSubBytes + Tr::kTileBytes, g, t, o);
  };

  // ---- windows of kPfIdCap prefix blocks (one window below 2048 blocks)
  // (first: the first key of the window's stages, a stage boundary)
  const BT* btp = static_cast<const BT*>(a.block_table);
  const int win_tokens = kPfIdCap << a.bs_log2;  // a multiple of the stage size
  for (int first = it.kb0; first < key_end;) {
    const int win0 = first / win_tokens * win_tokens;
    win_blk0 = win0 >> a.bs_log2;
    if (win0 < cached) {
      const int pref_end = min(cached, win0 + win_tokens);
      const int nb = ((pref_end - 1) >> a.bs_log2) - win_blk0 + 1;
      for (int i = threadIdx.x; i < nb; i += W * 64)
        s_ids[i] = static_cast<int32_t>(btp[row * a.bt_stride + win_blk0 + i]);
    }
    __syncthreads();  // block ids of the window visible; previous window's stages released
    const int k0 = first / Tr::kStageTokens;
    const int n = (min(key_end, win0 + win_tokens) - first + Tr::kStageTokens - 1) / Tr::kStageTokens;
    unsigned valid = issue(k0, 0);
    // Stage i: wait for this wave's copies of it, clear its invalid V slots,
    // one barrier (every wave's part landed; stage i-1 consumed by all),
    // then refill stage i-1's buffer with stage i+1 and compute stage i.
    auto step = [&](int i, auto st_c) __attribute__((always_inline)) {
      constexpr int ST = decltype(st_c)::value;
      wait_vmcnt<0>();
      asm volatile("" ::: "memory");
      if (__builtin_amdgcn_ballot_w64(valid != copy.kAllValid) != 0) zero_invalid_v(ST, valid);
      __syncthreads();
      if (i + 1 < n) valid = issue(k0 + i + 1, ST ^ 1);
      asm volatile("" ::: "memory");
      compute_stage(k0 + i, ST);
    };
    for (int i = 0; i < n; i += 2) {
      step(i, IntC<0>{});
      if (i + 1 >= n) break;
      step(i + 1, IntC<1>{});
    }
    __syncthreads();  // every wave is done with this window's stages and ids
    first = win0 + win_tokens;
  }

  // Lane coordinates and n_rep's division constants are recomputed for the
  // epilogue rather than kept live through the key loop.
  const int lane_e = __lane_id();
  const int te = lane_e & 15, ge = lane_e >> 4;
  int n_rep_e = a.n_rep;
  asm volatile("" : "+s"(n_rep_e));

  // ---- normalise and store this wave's rows: to the output, or as this
  // part's partial rows (row index within the unit: token * n_rep + head)
  const PrefillPart part = load_part<D>(a, n_rep_e);
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  float* recs = part.recs + (static_cast<int64_t>(part.part) * part.rows_cap + wtok0 * n_rep_e) * (D + 2);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int r = 4 * ge + e;  // row of o[0][.][e]
    const float ir = __shfl(inv, r);
    const int rtok = wtok0 + r / n_rep_e;
    if (r < tpw * n_rep_e && rtok < ntok) {
      if (part.nparts == 1) {
        float* op = static_cast<float*>(a.out) + (qbase + rtok) * a.o_st + (h * n_rep_e + r % n_rep_e) * a.o_sh;
#pragma unroll
        for (int c = 0; c < D / 16; ++c) op[16 * c + te] = o[0][c][e] * ir;
      } else {
        uint32_t* pp = reinterpret_cast<uint32_t*>(recs + r * (D + 2));
#pragma unroll
        for (int c = 0; c < D / 16; ++c) store_coherent_u32(pp + 16 * c + te, __float_as_uint(o[0][c][e] * ir));
      }
    }
  }
  if (part.nparts == 1) return;
  // the (max, sum) of row te, from the lanes ge == 0
  if (ge == 0 && te < tpw * n_rep_e && wtok0 + te / n_rep_e < ntok)
    store_coherent_u64(reinterpret_cast<uint64_t*>(recs + te * (D + 2) + D), pack_f32x2(m_run, l_run));
  fold_parts<DTYPE, D, W * 64>(a, part, ntok * n_rep_e, n_rep_e, qbase, h);
}

// Work groups of 128 query rows in 4 waves x 2 key sets (the 16-bit types), or
// of floor(16 / n_rep) tokens per wave (fp32).
template <int DTYPE, int D>
struct PrefillCfg : Prefill16Traits<DTYPE, D, 4, 2> {};
template <int D>
struct PrefillCfg<MV_DTYPE_F32, D> : Prefill32Traits<D> {
  static constexpr int kThreads = Prefill32Traits<D>::kWaves * 64;
};

template <int DTYPE, int D, typename BT>
__global__ __launch_bounds__((PrefillCfg<DTYPE, D>::kThreads)) void paged_prefill_kernel(PrefillArgs a) {
  if constexpr (DTYPE == MV_DTYPE_F32) prefill32<D, BT>(a);
  else prefill16<PrefillCfg<DTYPE, D>, BT>(a);
}

// Query tokens an item of mv_paged_prefill may hold: floor(32 / n_rep) per 32
// rows (16-bit types at head_dim 64) or floor(16 / n_rep) per 16 rows.
int prefill_tokens_per_group(int n_rep, int head_dim, int dtype) {
  if (n_rep > 16) return 0;
  if (dtype == MV_DTYPE_F32)
    return (head_dim == 64 ? Prefill32Traits<64>::kWaves : Prefill32Traits<128>::kWaves) * (16 / n_rep);
  return head_dim == 64 ? 4 * (32 / n_rep) : 8 * (16 / n_rep);
}

// Query tokens an item of mv_paged_prefill_blocks may hold: as many as 128
// (`wide`: 256) packed rows hold, for the 16-bit types.
int prefill_block_tokens(int n_rep, int head_dim, int dtype, bool wide) {
  if (n_rep > 16) return 0;
  return dtype == MV_DTYPE_F32 ? prefill_tokens_per_group(n_rep, head_dim, dtype) : (wide ? 256 : 128) / n_rep;
}

template <int DTYPE, int D>
int launch_prefill(const PrefillArgs& a, int groups, bool bt_i64, hipStream_t s) {
  constexpr int kThreads = PrefillCfg<DTYPE, D>::kThreads;
  if (bt_i64) paged_prefill_kernel<DTYPE, D, int64_t><<<groups, kThreads, 0, s>>>(a);
  else paged_prefill_kernel<DTYPE, D, int32_t><<<groups, kThreads, 0, s>>>(a);
  return check_launch("mv_paged_prefill");
}

template <int DTYPE>
int launch_prefill_d(const PrefillArgs& a, int d, int groups, bool bt_i64, hipStream_t s) {
  return d == 64 ? launch_prefill<DTYPE, 64>(a, groups, bt_i64, s) : launch_prefill<DTYPE, 128>(a, groups, bt_i64, s);
}

}  // namespace
}  // namespace mv

namespace mv {
namespace {

// Device-side prefill plan for a launch of fixed size (graph capture, where
// the lengths cannot be read back): one work group validates each
// sequence's prefix entries, scans the chunk lengths into chunk rows, and
// writes the work list in sequence order, every slot past the last work
// group marked unused. status[0] = sequences with a bad row, length or
// prefix table entry; status[1] = work groups (or -1 when they exceed the
// capacity, or the chunk lengths the query rows: then every slot is unused).
constexpr int kPfPlanThreads = 256;
template <typename BT>
__global__ __launch_bounds__(kPfPlanThreads) void prefill_plan_kernel(
    const int64_t* rows, const int64_t* cached, const int64_t* qlen, int32_t num_seqs,
    int64_t total_rows, const BT* bt, int64_t bt_stride, int32_t bt_rows, int32_t max_blocks,
    int32_t bs_log2, int64_t num_blocks, int32_t tpg, int32_t num_kv_heads, int64_t* seqs,
    int32_t* work, int32_t work_cap, int32_t* status) {
  __shared__ int s_bad;
  __shared__ int64_t s_rows_total, s_groups;
  const int tid = threadIdx.x;
  if (tid == 0) {
    s_bad = 0;
    s_rows_total = 0;
    s_groups = 0;
  }
  __syncthreads();
  // 1. validate, sequence by sequence (prefill batches hold few sequences)
  for (int i = 0; i < num_seqs; ++i) {
    const int64_t r = rows[i], c = cached[i], q = qlen[i];
    const int64_t need = (c + (int64_t(1) << bs_log2) - 1) >> bs_log2;
    const bool shape_ok = r >= 0 && r < bt_rows && c >= 0 && q >= 0 && c <= INT_MAX / 2 &&
                          q <= INT_MAX / 2 && need <= max_blocks;
    int bad = 0;
    if (shape_ok) {
      for (int64_t j = tid; j < need; j += kPfPlanThreads) {
        const int64_t blk = static_cast<int64_t>(bt[r * bt_stride + j]);
        bad |= blk < 0 || blk >= num_blocks;
      }
    }
    bad = __syncthreads_or(bad);
    if (tid == 0) {
      if (!shape_ok || bad) ++s_bad;
      s_rows_total += q >= 0 ? q : 0;
      s_groups += q > 0 ? ((q + tpg - 1) / tpg) * num_kv_heads : 0;
    }
    __syncthreads();
  }
  const bool ok = s_bad == 0 && s_rows_total <= total_rows && s_groups <= work_cap;
  // 2. per-sequence rows and work groups (thread 0: a short sequential scan)
  if (tid == 0 && ok) {
    int64_t start = 0, slot = 0;
    for (int i = 0; i < num_seqs; ++i) {
      const int64_t q = qlen[i];
      seqs[4 * i] = rows[i];
      seqs[4 * i + 1] = cached[i];
      seqs[4 * i + 2] = start;
      seqs[4 * i + 3] = q;
      for (int64_t t0 = 0; t0 < q; t0 += tpg) {
        const int nt = static_cast<int>(q - t0 < tpg ? q - t0 : tpg);
        for (int h = 0; h < num_kv_heads; ++h, ++slot)
          reinterpret_cast<int4*>(work)[slot] = make_int4(i, h, static_cast<int>(t0), nt);
      }
      start += q;
    }
  }
  // 3. the unused slots (all of them for an unusable plan)
  const int64_t used = ok ? s_groups : 0;
  for (int64_t slot = used + tid; slot < work_cap; slot += kPfPlanThreads)
    reinterpret_cast<int4*>(work)[slot] = make_int4(-1, 0, 0, 0);
  if (tid == 0) {
    status[0] = s_bad;
    status[1] = ok ? static_cast<int32_t>(s_groups) : -1;
  }
}

}  // namespace
}  // namespace mv

namespace mv {
namespace {

// Prefix entries of the eager plan's sequences: one work group per sequence
// reads the table entries its cached prefix needs (status[i] = some entry is
// not a pool block). Bound by latency (a launch and one read-back per step);
// on the host the same check took a copy of the whole table and three tensor
// operations per sequence, 130 us of a step of 16 sequences.
constexpr int kPrefixCheckThreads = 256;
template <typename BT>
__global__ __launch_bounds__(kPrefixCheckThreads) void prefix_entries_kernel(
    const int64_t* seqs, const BT* bt, int64_t bt_stride, int32_t bt_rows, int32_t max_blocks,
    int32_t bs_log2, int64_t num_blocks, int32_t* status) {
  const int64_t row = seqs[4 * blockIdx.x], cached = seqs[4 * blockIdx.x + 1];
  const int64_t need = (cached + (int64_t(1) << bs_log2) - 1) >> bs_log2;
  const bool shape_ok = row >= 0 && row < bt_rows && cached >= 0 && need <= max_blocks;
  int bad = !shape_ok;
  if (shape_ok) {
    for (int64_t j = threadIdx.x; j < need; j += kPrefixCheckThreads) {
      const int64_t blk = static_cast<int64_t>(bt[row * bt_stride + j]);
      bad |= blk < 0 || blk >= num_blocks;
    }
  }
  bad = __syncthreads_or(bad);
  if (threadIdx.x == 0) status[blockIdx.x] = bad;
}

}  // namespace
}  // namespace mv

// Host code: a step's first prefill layer waits for this list. Built here it takes
// 2-10 us; in Python one step of one sequence took 15 us with numpy, and 0.5 us
// per work group in a loop.
extern "C" int mv_prefill_work_items(const int64_t* rows, const int64_t* cached, const int64_t* query_len,
                                     int32_t num_seqs, int32_t num_kv_heads, int32_t tokens_per_item,
                                     int32_t cu_count, int32_t max_parts, int64_t* seqs,
                                     int32_t* work_items, int64_t capacity_ints, int32_t* info) {
  using namespace mv;
  constexpr int64_t kPartKeys = 256;  // parts start at stage boundaries
  if (num_seqs < 0 || num_kv_heads <= 0 || tokens_per_item <= 0 || cu_count <= 0 || capacity_ints < 0)
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_work_items: bad sizes");
  if (max_parts > 255) return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_work_items: %d parts", max_parts);
  if (!info || (num_seqs > 0 && (!rows || !cached || !query_len || !seqs || !work_items)))
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_work_items: null pointer");
  int64_t start = 0, units = 0, most_keys = 0;
  for (int i = 0; i < num_seqs; ++i) {
    const int64_t c = cached[i], q = query_len[i];
    if (c < 0 || q < 0 || c > INT_MAX / 2 || q > INT_MAX / 2)
      return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_work_items: sequence %d: lengths %lld + %lld", i,
                  static_cast<long long>(c), static_cast<long long>(q));
    seqs[4 * i] = rows[i];
    seqs[4 * i + 1] = c;
    seqs[4 * i + 2] = start;
    seqs[4 * i + 3] = q;
    start += q;
    units += (q + tokens_per_item - 1) / tokens_per_item * num_kv_heads;
    if (q > 0) most_keys = std::max(most_keys, c + q);
  }
  // parts of a unit of this many keys
  const int64_t split = units > 0 && units < cu_count
                            ? std::max<int64_t>(1, std::min<int64_t>(max_parts, cu_count / units)) : 1;
  auto parts_of = [&](int64_t keys) {
    return std::max<int64_t>(1, std::min(split, (keys + kPartKeys - 1) / kPartKeys / 2));
  };
  const int64_t most = parts_of(most_keys);  // grows with the keys
  const int ints = most > 1 ? 8 : 4;
  const int64_t bound = most > 1 ? cu_count : units;  // units * split at most
  if (bound * ints > capacity_ints || bound > INT_MAX / 8)
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_work_items: %lld items may exceed the capacity",
                static_cast<long long>(bound));
  struct Item {
    int32_t keys, w[8];
  };
  const std::unique_ptr<Item[]> items(new (std::nothrow) Item[bound + 1]);  // (no exception leaves a C entry)
  if (!items) return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_work_items: out of host memory");
  int64_t count = 0;
  int32_t unit = 0;
  for (int i = 0; i < num_seqs; ++i) {
    const int64_t blocks = (query_len[i] + tokens_per_item - 1) / tokens_per_item;
    for (int64_t b = blocks - 1; b >= 0; --b) {  // the last block has the most keys
      const int64_t t0 = b * tokens_per_item;
      const int64_t nt = std::min<int64_t>(tokens_per_item, query_len[i] - t0);
      const int64_t keys = cached[i] + t0 + nt, nb = (keys + kPartKeys - 1) / kPartKeys;
      const int64_t parts = parts_of(keys);
      for (int h = 0; h < num_kv_heads; ++h, ++unit)
        for (int64_t p = 0; p < parts; ++p) {
          const int64_t k0 = p * nb / parts * kPartKeys;
          const int64_t k1 = p + 1 == parts ? keys : (p + 1) * nb / parts * kPartKeys;
          items[count++] = {static_cast<int32_t>(k1 - k0),
                            {i, h, static_cast<int32_t>(t0), static_cast<int32_t>(nt), static_cast<int32_t>(k0),
                             static_cast<int32_t>(k1), unit, static_cast<int32_t>(p | parts << 8 | most << 16)}};
        }
    }
  }
  std::stable_sort(items.get(), items.get() + count, [](const Item& a, const Item& b) { return a.keys > b.keys; });
  for (int64_t k = 0; k < count; ++k) std::memcpy(work_items + k * ints, items[k].w, ints * 4);
  info[0] = static_cast<int32_t>(count);
  info[1] = static_cast<int32_t>(units);
  info[2] = static_cast<int32_t>(most);
  return MV_OK;
}

extern "C" int mv_prefill_prefix_check(const int64_t* seqs, int32_t num_seqs, const void* block_table,
                                       int32_t bt_is_i64, int64_t bt_stride, int32_t bt_rows,
                                       int32_t max_blocks, int32_t block_size, int64_t num_blocks,
                                       int32_t* status, void* stream) {
  using namespace mv;
  if (num_seqs < 0 || bt_rows < 0 || max_blocks < 0)
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_prefix_check: bad sizes");
  if (!is_pow2(block_size))
    return fail(MV_ERR_UNSUPPORTED, "mv_prefill_prefix_check: block_size %d is not a power of 2", block_size);
  if (num_seqs == 0) return MV_OK;
  if (!seqs || !status || (bt_rows > 0 && max_blocks > 0 && !block_table))
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_prefix_check: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int rows_ok = block_table ? bt_rows : 0;
  if (bt_is_i64)
    prefix_entries_kernel<int64_t><<<num_seqs, kPrefixCheckThreads, 0, s>>>(
        seqs, static_cast<const int64_t*>(block_table), bt_stride, rows_ok, max_blocks,
        ilog2_exact(block_size), num_blocks, status);
  else
    prefix_entries_kernel<int32_t><<<num_seqs, kPrefixCheckThreads, 0, s>>>(
        seqs, static_cast<const int32_t*>(block_table), bt_stride, rows_ok, max_blocks,
        ilog2_exact(block_size), num_blocks, status);
  return check_launch("mv_prefill_prefix_check");
}

extern "C" int mv_prefill_plan(const int64_t* seq_rows, const int64_t* cached_len,
                               const int64_t* query_len, int32_t num_seqs, int64_t total_query_rows,
                               const void* block_table, int32_t bt_is_i64, int64_t bt_stride,
                               int32_t bt_rows, int32_t max_blocks, int32_t block_size,
                               int64_t num_blocks, int32_t tokens_per_group, int32_t num_kv_heads,
                               int64_t* seqs, int32_t* work_items, int32_t work_capacity,
                               int32_t* status, void* stream) {
  using namespace mv;
  if (!status || !work_items || (num_seqs > 0 && (!seq_rows || !cached_len || !query_len || !seqs)))
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_plan: null pointer");
  if (num_seqs < 0 || work_capacity < 0 || tokens_per_group <= 0 || num_kv_heads <= 0 ||
      total_query_rows < 0 || bt_rows < 0 || max_blocks < 0)
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_plan: bad sizes");
  if (!is_pow2(block_size))
    return fail(MV_ERR_UNSUPPORTED, "mv_prefill_plan: block_size %d is not a power of 2", block_size);
  if (bt_rows > 0 && max_blocks > 0 && !block_table)
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_plan: null block table");
  if (reinterpret_cast<uintptr_t>(work_items) % 16)
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_prefill_plan: work_items not 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int bl = ilog2_exact(block_size);
  const int rows_ok = block_table ? bt_rows : 0;
  if (bt_is_i64)
    prefill_plan_kernel<int64_t><<<1, kPfPlanThreads, 0, s>>>(
        seq_rows, cached_len, query_len, num_seqs, total_query_rows,
        static_cast<const int64_t*>(block_table), bt_stride, rows_ok, max_blocks, bl, num_blocks,
        tokens_per_group, num_kv_heads, seqs, work_items, work_capacity, status);
  else
    prefill_plan_kernel<int32_t><<<1, kPfPlanThreads, 0, s>>>(
        seq_rows, cached_len, query_len, num_seqs, total_query_rows,
        static_cast<const int32_t*>(block_table), bt_stride, rows_ok, max_blocks, bl, num_blocks,
        tokens_per_group, num_kv_heads, seqs, work_items, work_capacity, status);
  return check_launch("mv_prefill_plan");
}

extern "C" int mv_prefill_tokens_per_group(int32_t num_q_heads, int32_t num_kv_heads,
                                           int32_t head_dim, int32_t dtype) {
  if (num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads) return 0;
  if ((head_dim != 64 && head_dim != 128) || mv::dtype_bytes(dtype) == 0) return 0;
  return mv::prefill_tokens_per_group(num_q_heads / num_kv_heads, head_dim, dtype);
}

extern "C" int mv_prefill_block_tokens(int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                       int32_t dtype, int32_t wide) {
  if (mv_prefill_tokens_per_group(num_q_heads, num_kv_heads, head_dim, dtype) == 0) return 0;
  return mv::prefill_block_tokens(num_q_heads / num_kv_heads, head_dim, dtype, wide != 0);
}

extern "C" size_t mv_paged_prefill_blocks_workspace_bytes(int32_t num_units, int32_t max_parts,
                                                          int32_t tokens_per_item,
                                                          int32_t num_q_heads, int32_t num_kv_heads,
                                                          int32_t head_dim, int32_t dtype) {
  const int most = mv_prefill_block_tokens(num_q_heads, num_kv_heads, head_dim, dtype, 1);
  if (tokens_per_item <= 0 || tokens_per_item > most || num_units <= 0 || max_parts <= 1) return 0;
  const size_t rows = static_cast<size_t>(num_units) * max_parts * tokens_per_item * (num_q_heads / num_kv_heads);
  return mv::kPfCountersBytes + rows * (head_dim + 2) * 4;
}

extern "C" size_t mv_paged_prefill_workspace_bytes(int32_t num_units, int32_t max_parts,
                                                   int32_t num_q_heads, int32_t num_kv_heads,
                                                   int32_t head_dim, int32_t dtype) {
  return mv_paged_prefill_blocks_workspace_bytes(
      num_units, max_parts, mv_prefill_tokens_per_group(num_q_heads, num_kv_heads, head_dim, dtype),
      num_q_heads, num_kv_heads, head_dim, dtype);
}

namespace mv {
namespace {

// Key split of mv_paged_prefill_parts (null for mv_paged_prefill).
struct PrefillParts {
  int32_t num_units;
  int32_t max_parts;
  void* workspace;
  size_t workspace_bytes;
};

int paged_prefill(const void* query, int64_t q_stride_tok, int64_t q_stride_head,
                  const void* key, int64_t k_stride_tok, int64_t k_stride_head,
                  const void* value, int64_t v_stride_tok, int64_t v_stride_head,
                  const void* key_cache, const void* value_cache, const void* block_table,
                  int32_t bt_is_i64, int64_t bt_stride, const int64_t* seqs, int32_t num_seqs,
                  const int32_t* work_items, int32_t num_work_groups, int32_t tokens_per_item,
                  void* out, int64_t out_stride_tok, int64_t out_stride_head, float scale,
                  int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                  int32_t block_size, int64_t num_blocks, int32_t dtype,
                  const PrefillParts* parts, void* stream) {
  const int eb = dtype_bytes(dtype);
  if (eb == 0) return fail(MV_ERR_UNSUPPORTED, "mv_paged_prefill: unknown dtype %d", dtype);
  if (head_dim != 64 && head_dim != 128)
    return fail(MV_ERR_UNSUPPORTED, "mv_paged_prefill: head_dim %d not supported (64, 128)", head_dim);
  if (!is_pow2(block_size))
    return fail(MV_ERR_UNSUPPORTED, "mv_paged_prefill: block_size %d is not a power of 2", block_size);
  const int tpg = mv_prefill_tokens_per_group(num_q_heads, num_kv_heads, head_dim, dtype);
  if (tpg == 0)
    return fail(MV_ERR_UNSUPPORTED, "mv_paged_prefill: %d query heads over %d kv heads not supported",
                num_q_heads, num_kv_heads);
  const int n_rep = num_q_heads / num_kv_heads;
  if (tokens_per_item <= 0) tokens_per_item = tpg;  // mv_paged_prefill, _parts
  if (tokens_per_item > prefill_block_tokens(n_rep, head_dim, dtype, true))
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_paged_prefill: %d tokens per item (at most %d)", tokens_per_item,
                prefill_block_tokens(n_rep, head_dim, dtype, true));
  if (num_seqs < 0 || num_work_groups < 0 || num_blocks <= 0)
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_paged_prefill: bad sizes");
  if (num_work_groups == 0) return MV_OK;
  if (!query || !key || !value || !key_cache || !value_cache || !seqs || !work_items || !out ||
      (!block_table && bt_stride != 0))
    return fail(MV_ERR_INVALID_ARGUMENT, "mv_paged_prefill: null pointer");
  if ((reinterpret_cast<uintptr_t>(query) | reinterpret_cast<uintptr_t>(key) |
       reinterpret_cast<uintptr_t>(value) | reinterpret_cast<uintptr_t>(key_cache) |
       reinterpret_cast<uintptr_t>(value_cache) | reinterpret_cast<uintptr_t>(work_items)) % 16 ||
      ((q_stride_tok | q_stride_head | k_stride_tok | k_stride_head | v_stride_tok |
        v_stride_head) * eb) % 16)
    return fail(MV_ERR_INVALID_ARGUMENT,
                "mv_paged_prefill: query/key/value rows and caches must be 16-byte aligned");
  PrefillArgs a;
  a.work = work_items;
  a.seqs = seqs;
  a.q = query;
  a.k_new = static_cast<const char*>(key);
  a.v_new = static_cast<const char*>(value);
  a.k_cache = static_cast<const char*>(key_cache);
  a.v_cache = static_cast<const char*>(value_cache);
  a.block_table = block_table;
  a.out = out;
  a.q_st = q_stride_tok;
  a.q_sh = q_stride_head;
  a.k_st = k_stride_tok * eb;
  a.k_sh = k_stride_head * eb;
  a.v_st = v_stride_tok * eb;
  a.v_sh = v_stride_head * eb;
  a.o_st = out_stride_tok;
  a.o_sh = out_stride_head;
  a.bt_stride = bt_stride;
  a.scale_log2 = scale * 1.4426950408889634f;
  a.num_kv_heads = num_kv_heads;
  a.n_rep = num_q_heads / num_kv_heads;
  a.max_tokens = tokens_per_item;
  a.bs_log2 = ilog2_exact(block_size);
  a.num_blocks_u32 = static_cast<uint32_t>(std::min<int64_t>(num_blocks, int64_t(1) << 31));
  {
    const int64_t span = 16 * std::max(std::abs(a.k_st), std::abs(a.v_st)) + 16 * head_dim * eb;
    a.lane_offsets_32 = a.k_st >= 0 && a.v_st >= 0 && span < (int64_t(1) << 31);
  }
  a.out_vec = reinterpret_cast<uintptr_t>(out) % 16 == 0 && (out_stride_tok * eb) % 16 == 0 &&
              (out_stride_head * eb) % 16 == 0;
  a.item_ints = 4;
  a.ws = nullptr;
  a.num_units = 0;
  a.max_parts = 1;
  if (parts) {
    a.item_ints = 8;
    if (parts->num_units < 0 || parts->num_units > kPfMaxUnits || parts->max_parts < 1 ||
        parts->max_parts > kPfMaxParts)
      return fail(MV_ERR_INVALID_ARGUMENT,
                  "mv_paged_prefill_parts: %d units of %d parts (at most %d units, %d parts)",
                  parts->num_units, parts->max_parts, kPfMaxUnits, kPfMaxParts);
    if (parts->max_parts > 1) {
      const size_t need = mv_paged_prefill_blocks_workspace_bytes(
          parts->num_units, parts->max_parts, tokens_per_item, num_q_heads, num_kv_heads, head_dim, dtype);
      if (!parts->workspace || parts->workspace_bytes < need)
        return fail(MV_ERR_INVALID_ARGUMENT, "mv_paged_prefill_parts: workspace %zu bytes, need %zu",
                    parts->workspace_bytes, need);
      if (reinterpret_cast<uintptr_t>(parts->workspace) % 256)
        return fail(MV_ERR_INVALID_ARGUMENT, "mv_paged_prefill_parts: workspace not 256-byte aligned");
      a.ws = static_cast<char*>(parts->workspace);
      a.num_units = parts->num_units;
      a.max_parts = parts->max_parts;
    }
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool i64 = bt_is_i64 != 0;
  if (dtype != MV_DTYPE_F32 && tokens_per_item * n_rep > 128)
    return launch_prefill_wide(a, head_dim, dtype, num_work_groups, i64, s);
  switch (dtype) {
    case MV_DTYPE_F32: return launch_prefill_d<MV_DTYPE_F32>(a, head_dim, num_work_groups, i64, s);
    case MV_DTYPE_F16: return launch_prefill_d<MV_DTYPE_F16>(a, head_dim, num_work_groups, i64, s);
    default: return launch_prefill_d<MV_DTYPE_BF16>(a, head_dim, num_work_groups, i64, s);
  }
}

}  // namespace
}  // namespace mv

extern "C" int mv_paged_prefill(const void* query, int64_t q_stride_tok, int64_t q_stride_head,
                                const void* key, int64_t k_stride_tok, int64_t k_stride_head,
                                const void* value, int64_t v_stride_tok, int64_t v_stride_head,
                                const void* key_cache, const void* value_cache,
                                const void* block_table, int32_t bt_is_i64, int64_t bt_stride,
                                const int64_t* seqs, int32_t num_seqs, const int32_t* work_items,
                                int32_t num_work_groups, void* out, int64_t out_stride_tok,
                                int64_t out_stride_head, float scale, int32_t num_q_heads,
                                int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                                int64_t num_blocks, int32_t dtype, void* stream) {
  return mv::paged_prefill(query, q_stride_tok, q_stride_head, key, k_stride_tok, k_stride_head,
                           value, v_stride_tok, v_stride_head, key_cache, value_cache, block_table,
                           bt_is_i64, bt_stride, seqs, num_seqs, work_items, num_work_groups, 0, out,
                           out_stride_tok, out_stride_head, scale, num_q_heads, num_kv_heads,
                           head_dim, block_size, num_blocks, dtype, nullptr, stream);
}

extern "C" int mv_paged_prefill_parts(const void* query, int64_t q_stride_tok, int64_t q_stride_head,
                                      const void* key, int64_t k_stride_tok, int64_t k_stride_head,
                                      const void* value, int64_t v_stride_tok, int64_t v_stride_head,
                                      const void* key_cache, const void* value_cache,
                                      const void* block_table, int32_t bt_is_i64, int64_t bt_stride,
                                      const int64_t* seqs, int32_t num_seqs,
                                      const int32_t* work_items, int32_t num_work_groups,
                                      int32_t num_units, int32_t max_parts, void* out, int64_t out_stride_tok, int64_t out_stride_head,
                                      float scale, int32_t num_q_heads, int32_t num_kv_heads,
                                      int32_t head_dim, int32_t block_size, int64_t num_blocks,
                                      int32_t dtype, void* workspace, size_t workspace_bytes,
                                      void* stream) {
  const mv::PrefillParts parts{num_units, max_parts, workspace, workspace_bytes};
  return mv::paged_prefill(query, q_stride_tok, q_stride_head, key, k_stride_tok, k_stride_head,
                           value, v_stride_tok, v_stride_head, key_cache, value_cache, block_table,
                           bt_is_i64, bt_stride, seqs, num_seqs, work_items, num_work_groups, 0, out,
                           out_stride_tok, out_stride_head, scale, num_q_heads, num_kv_heads,
                           head_dim, block_size, num_blocks, dtype, &parts, stream);
}

extern "C" int mv_paged_prefill_blocks(
    const void* query, int64_t q_stride_tok, int64_t q_stride_head, const void* key,
    int64_t k_stride_tok, int64_t k_stride_head, const void* value, int64_t v_stride_tok,
    int64_t v_stride_head, const void* key_cache, const void* value_cache, const void* block_table,
    int32_t bt_is_i64, int64_t bt_stride, const int64_t* seqs, int32_t num_seqs,
    const int32_t* work_items, int32_t num_work_groups, int32_t tokens_per_item, int32_t num_units,
    int32_t max_parts, void* out, int64_t out_stride_tok, int64_t out_stride_head, float scale,
    int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
    int64_t num_blocks, int32_t dtype, void* workspace, size_t workspace_bytes, void* stream) {
  if (tokens_per_item <= 0)
    return mv::fail(MV_ERR_INVALID_ARGUMENT, "mv_paged_prefill_blocks: %d tokens per item", tokens_per_item);
  const mv::PrefillParts parts{num_units, max_parts, workspace, workspace_bytes};
  return mv::paged_prefill(query, q_stride_tok, q_stride_head, key, k_stride_tok, k_stride_head,
                           value, v_stride_tok, v_stride_head, key_cache, value_cache, block_table,
                           bt_is_i64, bt_stride, seqs, num_seqs, work_items, num_work_groups,
                           tokens_per_item, out, out_stride_tok, out_stride_head, scale, num_q_heads,
                           num_kv_heads, head_dim, block_size, num_blocks, dtype,
                           max_parts > 1 ? &parts : nullptr, stream);
}
