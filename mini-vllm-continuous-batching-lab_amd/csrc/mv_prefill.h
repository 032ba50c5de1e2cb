// Shared by the prefill kernels: the launch's arguments, a work group's work
// item, the copy of one 16-key K/V sub-tile into LDS, and the key split's
// hand-off and fold.
#pragma once

#include <climits>

#include "mv_coherent.h"
#include "mv_common.h"
#include "mv_tile.h"

namespace mv {

struct PrefillArgs {
  const int32_t* work;   // per work group: (sequence, kv head, first token, tokens)
  const int64_t* seqs;   // per sequence: (table row, cached tokens, first chunk row, chunk tokens)
  const void* q;
  const char* k_new;
  const char* v_new;
  const char* k_cache;
  const char* v_cache;
  const void* block_table;
  void* out;
  int64_t q_st, q_sh;     // elements
  int64_t k_st, k_sh;     // bytes
  int64_t v_st, v_sh;     // bytes
  int64_t o_st, o_sh;     // elements
  int64_t bt_stride;      // elements
  float scale_log2;
  int32_t num_kv_heads, n_rep, bs_log2;
  int32_t max_tokens;     // tokens an item may hold (kernel rows / n_rep at most)
  uint32_t num_blocks_u32;
  int32_t lane_offsets_32;  // 16 chunk rows of K and of V span < 2 GiB: 32-bit lane offsets
  int32_t out_vec;        // 16-byte aligned output rows: 16-byte stores
  // Key split: work items of 8 ints whose second half is (first key, end
  // key, unit, part | parts << 8 | max parts << 16); 4 ints: whole key
  // ranges, no split.
  int32_t item_ints;
  // The split's workspace: kPfMaxUnits int32 counters (parts done per
  // unit, zero at rest), then per unit max_parts blocks of max_tokens *
  // n_rep records (D normalised fp32 values, the fp32 (max, sum) pair):
  // record after record (fp32), or, for the 16-bit types, whose lanes hold
  // one row each, pair of values after pair of values over all records.
  // num_units / max_parts are the host-checked sizes it was allocated for;
  // an item outside them is skipped, never addressed.
  char* ws;
  int32_t num_units, max_parts;
};

// paged_prefill_wide.hip: the 16-bit types with 256 query rows per work group.
int launch_prefill_wide(const PrefillArgs& a, int head_dim, int dtype, int groups, bool bt_i64, hipStream_t s);

namespace {

constexpr int kPfIdCap = 2048;  // prefix block ids staged in LDS per window
// Key split: at most kPfMaxParts parts per unit, kPfMaxUnits units per launch
// (the workspace's counters come first, kPfCountersBytes of them).
constexpr int kPfMaxParts = 8;
constexpr int kPfMaxUnits = 16384;
constexpr int kPfCountersBytes = kPfMaxUnits * 4;

// One work group's item. `ok` is false for an unused slot and for a part
// that would not address a record block of the workspace.
struct PrefillItem {
  bool ok;
  int seq, h, tok0, ntok;
  int kb0, kb1;  // key range of a split unit ([0, INT_MAX): whole)
};

__device__ __forceinline__ PrefillItem load_item(const PrefillArgs& a) {
  PrefillItem it{true, 0, 0, 0, 0, 0, INT_MAX};
  const int4 w = reinterpret_cast<const int4*>(a.work)[blockIdx.x * (a.item_ints >> 2)];
  it.seq = w.x;
  it.h = w.y;
  it.tok0 = w.z;
  it.ntok = min(w.w, a.max_tokens);
  if (w.x < 0) it.ok = false;  // an unused slot of a launch of fixed size
  if (a.item_ints == 8) {
    const int4 w2 = reinterpret_cast<const int4*>(a.work)[blockIdx.x * 2 + 1];
    it.kb0 = w2.x;
    it.kb1 = w2.y;
    const int unit = w2.z, part = w2.w & 0xff, nparts = (w2.w >> 8) & 0xff;
    if (nparts < 1 || part >= nparts ||
        (nparts > 1 && (a.ws == nullptr || unit < 0 || unit >= a.num_units || nparts > a.max_parts)))
      it.ok = false;
  }
  return it;
}

// Where a work group's rows go: its unit, part and parts (1: straight to the
// output). Read after the key loop rather than kept in registers through it.
struct PrefillPart {
  int part, nparts, rows_cap;
  float* recs;  // the unit's records
  int32_t* counter;
};

template <int D>
__device__ __forceinline__ PrefillPart load_part(const PrefillArgs& a, int n_rep) {
  int unit = 0;
  PrefillPart p{0, 1, a.max_tokens * n_rep, nullptr, nullptr};
  if (a.item_ints == 8) {
    const int4 w2 = reinterpret_cast<const int4*>(a.work)[blockIdx.x * 2 + 1];
    unit = w2.z;
    p.part = w2.w & 0xff;
    p.nparts = (w2.w >> 8) & 0xff;
  }
  p.recs = reinterpret_cast<float*>(a.ws + kPfCountersBytes) +
           static_cast<int64_t>(unit) * a.max_parts * p.rows_cap * (D + 2);
  p.counter = reinterpret_cast<int32_t*>(a.ws) + unit;
  return p;
}

// The K/V copies of one work group: 16-key sub-tiles, HBM -> LDS in 1 KiB
// loads. Prefix keys go through the block ids staged in LDS, chunk keys
// through the chunk's row strides. The layout of a sub-tile in LDS:
//   fp32     16 rows of D elements under the tiles' piece swizzle (mv_tile.h);
//   16-bit   for every 64 dims a block of 16 rows of 128 bytes under the
//            swizzle of 8 pieces: a lane's read addresses are a few bases
//            plus constants, and a load still covers whole 128-byte lines.
template <int DTYPE, int D>
struct SubTileCopy {
  using G = TileGeom<DTYPE, D>;
  static constexpr int L = G::kLoads;
  static constexpr int RP = DTYPE == MV_DTYPE_F32 ? G::kRowPieces : 8;  // pieces per LDS row
  static constexpr int kBlockLoads = 16 * RP / 64;                     // loads per block of 16 rows
  static constexpr unsigned kAllValid = (1u << L) - 1;

  const PrefillArgs& a;
  const int32_t* s_ids;
  int h, cached, key_end;
  int64_t chunk_row0;  // chunk row of the sequence's first chunk token
  int lane;
  // byte offsets of this lane's piece in each load of a block, from key row 0
  uint32_t off_pool[kBlockLoads], off_k[kBlockLoads], off_v[kBlockLoads];

  // load c holds key row row_of(c) of the lane, 16 bytes at piece_of(c) of
  // block c / kBlockLoads
  static __device__ __forceinline__ int row_of(int lane, int c) {
    return (64 * (c % kBlockLoads) + lane) / RP;
  }
  static __device__ __forceinline__ int piece_of(int lane, int c) {
    return ((lane % RP) ^ piece_swizzle<RP>(row_of(lane, c))) * 16;
  }
  static constexpr int block_of(int c) { return c / kBlockLoads * RP * 16; }
  __device__ __forceinline__ void init() {
#pragma unroll
    for (int c = 0; c < kBlockLoads; ++c) {
      off_pool[c] = row_of(lane, c) * G::kRowBytes + piece_of(lane, c);
      off_k[c] = static_cast<uint32_t>(row_of(lane, c) * a.k_st + piece_of(lane, c));
      off_v[c] = static_cast<uint32_t>(row_of(lane, c) * a.v_st + piece_of(lane, c));
    }
  }

  // The id of the block that holds key kb, read ahead of the copy.
  __device__ __forceinline__ int block_id_of(int kb, int win_blk0) const {
    return s_ids[min(max((kb >> a.bs_log2) - win_blk0, 0), kPfIdCap - 1)];
  }

  // Copies keys kb .. kb + 15 to LDS address dst (K tile, then V tile; only
  // one of them with K or V false); returns the loads whose key row is one
  // of the work group's. Always L loads per tensor. Two wave-uniform cases
  // take one base address in SGPRs and a 32-bit offset per lane: 16 prefix
  // keys in one pool block (block size >= 16), and 16 chunk keys all below
  // key_end; the rest (a sub-tile that straddles the prefix end or key_end,
  // or smaller blocks) computes each lane's address.
  template <bool K = true, bool V = true>
  __device__ __forceinline__ unsigned copy(int kb, int win_blk0, uint32_t dst, int block_id) const {
    const int bs_mask = (1 << a.bs_log2) - 1;
    const uint32_t dst_v = dst + G::kTileBytes;
    if (kb + kTile <= cached && a.bs_log2 >= 4) {
      const int id = __builtin_amdgcn_readfirstlane(block_id);
      const bool ok = static_cast<uint32_t>(id) < a.num_blocks_u32;
      const int64_t row0 = ok ? ((static_cast<int64_t>(id) * a.num_kv_heads + h) << a.bs_log2) + (kb & bs_mask) : 0;
      const char* bk = a.k_cache + row0 * G::kRowBytes;
      const char* bv = a.v_cache + row0 * G::kRowBytes;
#pragma unroll
      for (int c = 0; c < L; ++c) {
        if (K) copy_to_lds_16B_sv(bk + block_of(c), off_pool[c % kBlockLoads], __builtin_amdgcn_readfirstlane(dst + c * 1024));
        if (V) copy_to_lds_16B_sv(bv + block_of(c), off_pool[c % kBlockLoads], __builtin_amdgcn_readfirstlane(dst_v + c * 1024));
      }
      return ok ? kAllValid : 0u;
    }
    if (kb >= cached && kb + kTile <= key_end && a.lane_offsets_32) {
      const int64_t cr0 = chunk_row0 + (kb - cached);  // chunk row of key kb
      const char* bk = a.k_new + cr0 * a.k_st + h * a.k_sh;
      const char* bv = a.v_new + cr0 * a.v_st + h * a.v_sh;
#pragma unroll
      for (int c = 0; c < L; ++c) {
        if (K) copy_to_lds_16B_sv(bk + block_of(c), off_k[c % kBlockLoads], __builtin_amdgcn_readfirstlane(dst + c * 1024));
        if (V) copy_to_lds_16B_sv(bv + block_of(c), off_v[c % kBlockLoads], __builtin_amdgcn_readfirstlane(dst_v + c * 1024));
      }
      return kAllValid;
    }
    // (opaque to hoisting: these addresses are not kept through the key loop)
    int lane_l = lane;
    asm volatile("" : "+v"(lane_l));
    unsigned valid = 0;
#pragma unroll
    for (int c = 0; c < L; ++c) {
      const int j = kb + row_of(lane_l, c);
      bool ok = j < key_end;
      int64_t offk = block_of(c) + piece_of(lane_l, c), offv = offk;
      const char* bk = a.k_cache;
      const char* bv = a.v_cache;
      if (j < cached) {
        const int id = block_id_of(j, win_blk0);
        ok = ok && static_cast<uint32_t>(id) < a.num_blocks_u32;
        const int64_t rowoff = (((static_cast<int64_t>(id) * a.num_kv_heads + h) << a.bs_log2) +
                                (j & bs_mask)) * G::kRowBytes;
        offk += ok ? rowoff : 0;
        offv = offk;
      } else if (ok) {
        const int64_t cr = chunk_row0 + (j - cached);  // chunk row of key j
        offk += cr * a.k_st + h * a.k_sh;
        offv += cr * a.v_st + h * a.v_sh;
        bk = a.k_new;
        bv = a.v_new;
      }
      valid |= ok ? (1u << c) : 0u;
      if (K) copy_to_lds_16B(bk + offk, __builtin_amdgcn_readfirstlane(dst + c * 1024));
      if (V) copy_to_lds_16B(bv + offv, __builtin_amdgcn_readfirstlane(dst_v + c * 1024));
    }
    return valid;
  }
};

// Counts a finished part on its unit; the work group that completes the
// count folds the unit's parts in part order (log-sum-exp), so the result
// does not depend on which part finishes last, and writes the rows. The
// partial rows are device-coherent stores; once every wave has seen them
// acknowledged, the counter increment publishes them. A thread folds 16 dims
// of a row; consecutive threads take what lies together in the records.
template <int DTYPE, int D, int THREADS>
__device__ __forceinline__ void fold_parts(const PrefillArgs& a, const PrefillPart& p, int nrows, int n_rep,
                                           int64_t qbase, int h) {
  using raw_t = typename Elem<DTYPE>::raw;
  constexpr bool kByPair = DTYPE != MV_DTYPE_F32;
  constexpr int kPairs = D / 2 + 1;  // 8-byte pairs per record: the row, then (max, sum)
  constexpr int kRowThreads = D / 16;
  __shared__ int s_last;
  __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
  __syncthreads();
  if (threadIdx.x == 0) {
    const int prev = __hip_atomic_fetch_add(p.counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = prev == p.nparts - 1;
  }
  __syncthreads();
  if (!s_last) return;
  for (int i = threadIdx.x; i < nrows * kRowThreads; i += THREADS) {
    const int gr = kByPair ? i % nrows : i / kRowThreads;
    const int pr0 = (kByPair ? i / nrows : i % kRowThreads) * 8;
    const int64_t step = kByPair ? p.rows_cap : 1;  // from pair to pair
    const uint64_t* rec0 = reinterpret_cast<const uint64_t*>(p.recs) + (kByPair ? gr : static_cast<int64_t>(gr) * kPairs);
    float m_all = kNegInf, l_all = 0.f;
    float acc[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.f;
    // rounds of 4 parts, every load of a round in flight before the first use
    for (int p0 = 0; p0 < p.nparts; p0 += 4) {
      uint64_t ml[4], ov[4][8];
#pragma unroll
      for (int pp = 0; pp < 4; ++pp) {
        const uint64_t* rec = rec0 + static_cast<int64_t>(min(p0 + pp, p.nparts - 1)) * p.rows_cap * kPairs;
        ml[pp] = load_coherent_u64(rec + (D / 2) * step);
#pragma unroll
        for (int j = 0; j < 8; ++j) ov[pp][j] = load_coherent_u64(rec + (pr0 + j) * step);
      }
      float m_round = m_all;
#pragma unroll
      for (int pp = 0; pp < 4; ++pp)
        if (p0 + pp < p.nparts) m_round = fmaxf(m_round, unpack_lo(ml[pp]));
      // every row sees key 0, which part 0 holds: m_round is finite
      const float rescale = m_all == kNegInf ? 0.f : __builtin_amdgcn_exp2f(m_all - m_round);
      l_all *= rescale;
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[j] *= rescale;
#pragma unroll
      for (int pp = 0; pp < 4; ++pp) {
        const float mp = unpack_lo(ml[pp]);
        const float wgt = p0 + pp < p.nparts && mp != kNegInf
                              ? unpack_hi(ml[pp]) * __builtin_amdgcn_exp2f(mp - m_round) : 0.f;
        l_all += wgt;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          acc[2 * j] += wgt * unpack_lo(ov[pp][j]);
          acc[2 * j + 1] += wgt * unpack_hi(ov[pp][j]);
        }
      }
      m_all = m_round;
    }
    const float inv = 1.f / l_all;
    raw_t* op = static_cast<raw_t*>(a.out) + (qbase + gr / n_rep) * a.o_st + (h * n_rep + gr % n_rep) * a.o_sh + 2 * pr0;
#pragma unroll
    for (int j = 0; j < 16; ++j) op[j] = from_f32<DTYPE>(acc[j] * inv);
  }
  if (threadIdx.x == 0)  // ready for the next call
    __hip_atomic_store(p.counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace
}  // namespace mv
