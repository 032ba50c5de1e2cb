// Prefill attention of the 16-bit types on 32x32x16 MFMAs: the body of
// paged_prefill_kernel (128 query rows per work group) and of
// paged_prefill_wide_kernel (256).
//
// A wave owns 32 query rows, one per MFMA column, and keeps S^T = K Q^T and
// O^T += V^T P^T transposed: a lane holds half of one row's scores, so the
// softmax needs no exchange between lanes beyond lane ^ 32, the reference and
// the rescale of O are one value per lane, and the scores' registers are, once
// packed, the B operand of the P V product as they stand (the keys' order in
// it is the one the transposed V reads return).
//
// Bound: at head_dim 64 a 32 x 32 tile costs 8 MFMAs (120 ns of its SIMD's
// matrix core, measured) and 16 exponentials, multiply-adds, 8 packs and 8 row
// sums per lane (116-129 ns of VALU); the two overlap only where both are in
// flight, 188 ns together. So each tile's softmax runs while the next tile's
// Q K^T is in the matrix core (across the stage boundary too, for which the
// next stage has to land one tile early), and V's operands are read a tile
// ahead. The copies into LDS (64 bytes per clock and CU) stall the waves that
// issue them: 256 rows per pass over the keys halve them per row, and lane
// offsets are kept in registers. Measured (bf16, against the 16x16x32 kernel
// of 112 rows per work group that this replaces): 4 x (1536 cached + 512) at
// 14 / 2 heads x 64 30.5 -> 27.3 us, 16 of them 102 -> 76 us (690 TFLOP/s), one
// 8192-token prompt at 28 / 4 x 128 866 -> 451 us (1067 TFLOP/s).
// Slower and not kept: two 32-row tiles per wave (135 against 97 us on the 16
// sequences), the softmax and the MFMAs pinned in alternation (5-10 %), copies
// spread over a stage's tiles, four tiles per stage.
#pragma once

#include "mv_prefill.h"

namespace mv {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// A tile of 32 keys keeps p = exp2(s - m) with the row's reference m
// unchanged while every lane's sum of its keys' p is at most this (every p
// then lies in fp16's range too, and l, at least 1 since the row's first
// exact tile, far above it).
constexpr float kPfFastMax = 4096.f;
// The reference before a row's first key: finite, so that a masked score
// gives p = 0, and so low that any other score leaves the range.
constexpr float kPfStart = -3e38f;

// RW row waves of 32 query rows x SETS key sets that split every stage's
// tiles; a stage holds T tiles of 32 keys for each set, two stages in LDS.
template <int DTYPE_, int D_, int RW_, int SETS_>
struct Prefill16Traits : TileGeom<DTYPE_, D_> {
  using G = TileGeom<DTYPE_, D_>;
  static constexpr int DTYPE = DTYPE_, D = D_, RW = RW_, SETS = SETS_, T = 2;
  static constexpr int kWaves = RW * SETS;
  static constexpr int kThreads = kWaves * 64;
  static constexpr int kRows = RW * 32;
  static constexpr int kSubBytes = 2 * G::kTileBytes;  // K and V of 16 keys
  static constexpr int kSubs = 2 * SETS * T;           // 16-key sub-tiles per stage
  // one sub-tile copied by each wave; with twice as many waves as sub-tiles
  // its K or its V half
  static constexpr bool kHalfSubs = 2 * kSubs == kWaves;
  static constexpr int kWaveLoads = (kHalfSubs ? 1 : 2) * G::kLoads;
  static constexpr int kStageTokens = kSubs * kTile;
  static constexpr int kStageBytes = kSubs * kSubBytes;
  // the set merge reuses the stage buffers: m, l and O of the waves of sets 1..
  static constexpr int kMergeFloats = 32 * 2 + (D / 32) * 16 * 64;
  static constexpr int kMergeBytes = (SETS - 1) * RW * kMergeFloats * 4;
  static constexpr int kIdsOffset = 2 * kStageBytes > kMergeBytes ? 2 * kStageBytes : kMergeBytes;
  static constexpr int kLdsBytes = kIdsOffset + kPfIdCap * 4;
  static_assert(kHalfSubs || kSubs == kWaves, "every wave copies the same amount");
  static_assert(256 % kStageTokens == 0, "parts start at stage boundaries");
  static_assert(kLdsBytes <= 160 * 1024 - 64, "LDS of one work group");
};

template <int DTYPE>
__device__ __forceinline__ f32x16 mfma32(u32x4 x, u32x4 y, f32x16 c) {
  if constexpr (DTYPE == MV_DTYPE_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, x), __builtin_bit_cast(f16x8, y), c, 0, 0, 0);
}

// This lane's value combined with the other half of the wave's (lane ^ 32).
__device__ __forceinline__ float halves_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float halves_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <class Tr, typename BT>
__device__ __forceinline__ void prefill16(const PrefillArgs& a) {
  constexpr int DTYPE = Tr::DTYPE, D = Tr::D, RW = Tr::RW, SETS = Tr::SETS, T = Tr::T;
  constexpr int KB = D / 16;  // 16-dim steps of K Q^T
  constexpr int C = D / 32;   // 32-dim tiles of O^T
  constexpr int L = Tr::kLoads;
  using raw_t = typename Elem<DTYPE>::raw;

  __shared__ __attribute__((aligned(16))) char s_lds[Tr::kLdsBytes];
  int32_t* s_ids = reinterpret_cast<int32_t*>(s_lds + Tr::kIdsOffset);
  const uint32_t lds0 = lds_address(s_lds);

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int n = lane & 31;  // query row of the wave (MFMA column)
  const int half = lane >> 5;
  const int rwave = wave % RW;
  const int set = wave / RW;

  const PrefillItem it = load_item(a);
  if (!it.ok) return;
  const int h = it.h, tok0 = it.tok0, ntok = it.ntok;
  const int64_t row = a.seqs[4 * it.seq];
  const int cached = static_cast<int>(a.seqs[4 * it.seq + 1]);
  const int64_t chunk_row0 = a.seqs[4 * it.seq + 2];
  const int64_t qbase = chunk_row0 + tok0;
  const int key_end = min(cached + tok0 + ntok, it.kb1);

  // ---- rows: row r of the work group is query head h * n_rep + r % n_rep of
  // token tok0 + r / n_rep, packed without gaps
  const int nrows = ntok * a.n_rep;
  const int row0 = rwave * 32;
  // keys up to first_limit are seen by every row of the wave, keys past
  // last_limit by none (-1: the wave has no rows)
  const int first_limit = __builtin_amdgcn_readfirstlane(cached + tok0 + row0 / a.n_rep);
  const int last_limit = __builtin_amdgcn_readfirstlane(
      row0 < nrows ? cached + tok0 + (min(nrows, row0 + 32) - 1) / a.n_rep : -1);
  int lim;  // the row's last key (-1: a padding row, never written)
  u32x4 q[KB];
  {
    const int r = row0 + n;
    const bool ok = r < nrows;
    const int tok = ok ? r / a.n_rep : 0;
    lim = ok ? cached + tok0 + tok : -1;
    const char* qrow = reinterpret_cast<const char*>(
        static_cast<const raw_t*>(a.q) + (qbase + tok) * a.q_st +
        (h * a.n_rep + (ok ? r - tok * a.n_rep : 0)) * a.q_sh);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      q[kb] = *reinterpret_cast<const u32x4*>(qrow + (2 * kb + half) * 16);
      if (!ok) q[kb] = u32x4{0, 0, 0, 0};  // finite scores
    }
  }

  // ---- lane bases of the LDS reads within a 32-key tile (two sub-tiles)
  // K operand: lane (n, half) reads key row n, dims 16 kb + 8 half .. + 7: a
  // base per kb & 3. V operand (transposed): the 16 lanes (half, n >> 4) read
  // 4 keys, 8 j + 4 half .. + 3, of 16 dims, 64 (c >> 1) + 16 (c & 1) + 32 (n
  // >> 4) .. of O^T tile c (the 32 lanes served together then fall into
  // different banks): a base per (c & 1, j).
  const int t16 = lane & 15;
  constexpr int kBases = 2 * Tr::kStageBytes > 65536 ? 2 : 1;  // read offsets hold 16 bits
  uint32_t k_base[kBases][4], v_base[kBases][2][2];
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int v_row = 8 * (x & 1) + 4 * half + (t16 >> 2);
    const uint32_t tile = lds0 + 2 * set * Tr::kSubBytes;
    k_base[0][x] = tile + (n >> 4) * Tr::kSubBytes + t16 * 128 + (((2 * x + half) ^ piece_swizzle<8>(t16)) << 4);
    v_base[0][x >> 1][x & 1] =
        tile + Tr::kTileBytes + v_row * 128 +
        (((4 * (n >> 4) + 2 * (x >> 1) + ((t16 & 3) >> 1)) ^ piece_swizzle<8>(v_row)) << 4) + (t16 & 1) * 8;
    // (opaque: the rest of every address is a constant offset)
    asm volatile("" : "+v"(k_base[0][x]), "+v"(v_base[0][x >> 1][x & 1]));
    if constexpr (kBases == 2) {
      k_base[1][x] = k_base[0][x] + Tr::kStageBytes;
      v_base[1][x >> 1][x & 1] = v_base[0][x >> 1][x & 1] + Tr::kStageBytes;
      asm volatile("" : "+v"(k_base[1][x]), "+v"(v_base[1][x >> 1][x & 1]));
    }
  }
  typedef __attribute__((address_space(3))) char* lds_ptr;
  auto lds_b128 = [&](uint32_t base, uint32_t off) __attribute__((always_inline)) {
    return *reinterpret_cast<__attribute__((address_space(3))) u32x4*>(reinterpret_cast<lds_ptr>(base) + off);
  };
  auto lds_tr = [&](uint32_t base, uint32_t off) __attribute__((always_inline)) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        reinterpret_cast<__attribute__((address_space(3))) s16x4*>(reinterpret_cast<lds_ptr>(base) + off));
  };

  float m = kPfStart, l = 0.f;  // reference; this half's share of the sum
  f32x16 o[C];                  // O^T: 32 dims x 32 rows, relative to m
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[c][e] = 0.f;
  u32x4 kp[KB];    // K operands of the next tile
  u32x4 v[2][C];   // V operands of the tile at hand

  // (buffer st, tile at byte offset `tile` of it)
  auto read_k = [&](int st, uint32_t tile) __attribute__((always_inline)) {
    const uint32_t off = tile + (kBases == 1 ? st * Tr::kStageBytes : 0);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) kp[kb] = lds_b128(k_base[kBases == 1 ? 0 : st][kb & 3], off + (kb >> 2) * 2048);
  };
  auto read_v = [&](int st, uint32_t tile) __attribute__((always_inline)) {
    const uint32_t off = tile + (kBases == 1 ? st * Tr::kStageBytes : 0);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const uint32_t (&b)[2] = v_base[kBases == 1 ? 0 : st][c & 1];
        const s16x4 lo = lds_tr(b[0], off + u * Tr::kSubBytes + (c >> 1) * 2048);
        const s16x4 hi = lds_tr(b[1], off + u * Tr::kSubBytes + (c >> 1) * 2048);
        v[u][c] = __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
  };
  // steps [j0, j1) of the next tile's S^T = K Q^T
  auto qk = [&](int j0, int j1, f32x16& s) __attribute__((always_inline)) {
#pragma unroll
    for (int kb = j0; kb < j1; ++kb) {
      f32x16 z;
#pragma unroll
      for (int e = 0; e < 16; ++e) z[e] = 0.f;
      s = mfma32<DTYPE>(kp[kb], q[kb], kb == 0 ? z : s);
    }
  };
  // p = exp2(s scale - m) of scores 4 j .. 4 j + 3, packed: half a register
  // quad of the P operand; the rounded values' sum added to `sum`
  auto exp4 = [&](const f32x16& s, int j, u32x4 (&p)[2], float& sum) __attribute__((always_inline)) {
    auto ex = [&](float x) __attribute__((always_inline)) {
      return __builtin_amdgcn_exp2f(__builtin_fmaf(x, a.scale_log2, -m));
    };
    const uint2 w = __builtin_bit_cast(uint2, pack_p<DTYPE>(ex(s[4 * j]), ex(s[4 * j + 1]), ex(s[4 * j + 2]),
                                                            ex(s[4 * j + 3]), sum));
    p[j >> 1][2 * (j & 1)] = w.x;
    p[j >> 1][2 * (j & 1) + 1] = w.y;
  };

  // ---- the key stream: this wave's share of stage k's copies into buffer st
  SubTileCopy<DTYPE, D> copy{a, s_ids, h, cached, key_end, chunk_row0, lane, {}, {}, {}};
  copy.init();
  int win_blk0 = 0;
  const int su = Tr::kHalfSubs ? wave >> 1 : wave;  // the wave's sub-tile
  auto stage_id = [&](int k) __attribute__((always_inline)) {
    return copy.block_id_of(k * Tr::kStageTokens + su * kTile, win_blk0);
  };
  auto issue = [&](int k, int st, int id) __attribute__((always_inline)) -> unsigned {
    const int kb = k * Tr::kStageTokens + su * kTile;
    const uint32_t dst = lds0 + st * Tr::kStageBytes + su * Tr::kSubBytes;
    if constexpr (Tr::kHalfSubs) {
      if (wave & 1) return copy.template copy<false, true>(kb, win_blk0, dst, id);
      copy.template copy<true, false>(kb, win_blk0, dst, id);
      return copy.kAllValid;  // (only V slots are cleared)
    } else {
      return copy.copy(kb, win_blk0, dst, id);
    }
  };
  // Waits for this wave's copies of a stage (the next stage's may stay in
  // flight) and meets the other waves: the stage is whole, and every wave has
  // read what it needs of the one before. V slots of keys that were not
  // loaded read pool row 0 instead: they are cleared first (P is 0 there, but
  // 0 * NaN would not be).
  auto land = [&](int st, unsigned ok, bool more) __attribute__((always_inline)) {
    wait_vmcnt_groups<Tr::kWaveLoads, 1>(more);
    asm volatile("" ::: "memory");
    if (__builtin_amdgcn_ballot_w64(ok != copy.kAllValid) != 0) {
      char* vdst = s_lds + st * Tr::kStageBytes + su * Tr::kSubBytes + Tr::kTileBytes;
#pragma unroll
      for (int c = 0; c < L; ++c)
        if (!((ok >> c) & 1u)) *reinterpret_cast<uint4*>(vdst + c * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
    }
    __syncthreads();
  };

  // One tile of 32 keys: masks its scores where a row does not see a key,
  // turns them into P while the next tile's Q K^T runs (NEXT; `next_k` reads
  // its K operands), and adds P V.
  auto do_tile = [&](int key0, f32x16& sc, auto next_c, f32x16& sn, auto next_k) __attribute__((always_inline)) {
    constexpr bool NEXT = decltype(next_c)::value != 0;
    if (key0 + 31 > first_limit) {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        sc[e] = key0 + 8 * (e >> 2) + 4 * half + (e & 3) <= lim ? sc[e] : kNegInf;
    }
    // p against the reference as it stands; where a lane's sum leaves the
    // range (or is NaN) the reference moves to the maximum so far, O and l are
    // rescaled and p is computed again, once
    u32x4 p[2];
    float sum;
    int again = 1;
    asm volatile("" : "+s"(again));  // a loop, not two copies of it
    while (true) {
      float part[2] = {0.f, 0.f};
      next_k();
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        exp4(sc, j, p, part[j & 1]);
        if constexpr (NEXT) qk(j * KB / 4, (j + 1) * KB / 4, sn);
      }
      sum = part[0] + part[1];
      if (__builtin_amdgcn_ballot_w64(!(sum <= kPfFastMax)) == 0 || again == 0) break;
      again = 0;
      float mc = kNegInf;
#pragma unroll
      for (int e = 0; e < 16; ++e) mc = fmaxf(mc, sc[e]);
      const float mn = fmaxf(m, halves_max(mc) * a.scale_log2);
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[c][e] *= alpha;
    }
    l += sum;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int c = 0; c < C; ++c) o[c] = mfma32<DTYPE>(v[u][c], p[u], o[c]);
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
      for (int i = threadIdx.x; i < nb; i += Tr::kThreads)
        s_ids[i] = static_cast<int32_t>(btp[row * a.bt_stride + win_blk0 + i]);
    }
    // Q must have landed before the tile copies are counted by vmcnt (its
    // loads and the ids' are in flight together).
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) asm volatile("" ::"v"(q[kb]));
    __syncthreads();  // block ids of the window visible; previous window's stages released
    const int k0 = first / Tr::kStageTokens;
    const int ns = (min(key_end, win0 + win_tokens) - first + Tr::kStageTokens - 1) / Tr::kStageTokens;
    const unsigned ok = issue(k0, 0, stage_id(k0));
    unsigned ok_next = 0;
    if (ns > 1) ok_next = issue(k0 + 1, 1, stage_id(k0 + 1));
    land(0, ok, ns > 1);

    // this wave's tiles that some row of it sees, and the stages full of them
    const int set_key = first + set * 32;
    const int na = max(0, min(ns * T, (last_limit - set_key + SETS * 32) / (SETS * 32)));
    const int nf = na / T;
    constexpr uint32_t kTileStep = SETS * 2 * Tr::kSubBytes;
    int i = 0;
    // Stage i + 1 has to land before stage i's last tile is turned into P
    // (stage i + 1's first Q K^T runs then); with that tile's V read, stage
    // i's buffer is free for stage i + 2.
    if (nf > 0) {
      f32x16 s[2];
      read_k(0, 0);
      read_v(0, 0);
      qk(0, KB, s[0]);
      auto step = [&](auto st_c) __attribute__((always_inline)) {
        constexpr int ST = decltype(st_c)::value;
        do_tile(set_key + i * T * SETS * 32, s[0], IntC<1>{}, s[1], [&] { read_k(ST, kTileStep); });
        read_v(ST, kTileStep);
        if (i + 1 < ns) land(ST ^ 1, ok_next, false);
        const int id = stage_id(k0 + i + 2);
        do_tile(set_key + (i * T + 1) * SETS * 32, s[1], IntC<1>{}, s[0], [&] { read_k(ST ^ 1, 0); });
        read_v(ST ^ 1, 0);
        if (i + 2 < ns) ok_next = issue(k0 + i + 2, ST, id);
        asm volatile("" ::: "memory");
        ++i;
      };
      while (true) {
        step(IntC<0>{});
        if (i >= nf) break;
        step(IntC<1>{});
        if (i >= nf) break;
      }
    }
    // the stage some of whose tiles the wave's rows see, and those after it
    for (; i < ns; ++i) {
      const int st = i & 1;
      for (int t = 0; t < T && i * T + t < na; ++t) {
        f32x16 s;
        read_k(0, st * Tr::kStageBytes + t * kTileStep);
        read_v(0, st * Tr::kStageBytes + t * kTileStep);
        qk(0, KB, s);
        do_tile(set_key + (i * T + t) * SETS * 32, s, IntC<0>{}, s, [] {});
      }
      if (i + 1 < ns) land(st ^ 1, ok_next, false);
      if (i + 2 < ns) ok_next = issue(k0 + i + 2, st, stage_id(k0 + i + 2));
      asm volatile("" ::: "memory");
    }
    __syncthreads();  // every wave is done with this window's stages and ids
    first = win0 + win_tokens;
  }

  l = halves_sum(l);
  if (!(l > 0.f)) m = kNegInf;  // saw no key: no weight in the merges

  // ---- merge the sets' softmax states (same rows): sets 1.. leave m, l and
  // O in LDS (the stage buffers, free after the last barrier), set 0 folds
  // them in and stores. At head_dim 128 this moves 16 KiB per row wave, 0.45
  // us of a prompt of a few tokens with all four: waves without rows have no
  // part in it, and up to 32 keys set 0 holds them all.
  if constexpr (SETS > 1) {
    if (key_end - it.kb0 > 32) {
      if (set > 0 && row0 < nrows) {
        float* x = reinterpret_cast<float*>(s_lds) + ((set - 1) * RW + rwave) * Tr::kMergeFloats;
        if (half == 0) {
          x[n] = m;
          x[32 + n] = l;
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
          for (int e = 0; e < 16; ++e) x[64 + (c * 16 + e) * 64 + lane] = o[c][e];
      }
      __syncthreads();
      if (set == 0 && row0 < nrows) {
#pragma unroll
        for (int s = 1; s < SETS; ++s) {
          const float* x = reinterpret_cast<const float*>(s_lds) + ((s - 1) * RW + rwave) * Tr::kMergeFloats;
          const float m1 = x[n], l1 = x[32 + n];
          const float mm = fmaxf(m, m1);
          const float mr = mm == kNegInf ? 0.f : mm;
          const float a0 = __builtin_amdgcn_exp2f(m - mr), a1 = __builtin_amdgcn_exp2f(m1 - mr);
          l = l * a0 + l1 * a1;
          m = mm;
#pragma unroll
          for (int c = 0; c < C; ++c)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[c][e] = o[c][e] * a0 + x[64 + (c * 16 + e) * 64 + lane] * a1;
        }
      }
    }
  }

  // ---- normalise and store: to the output, or as this part's partial rows.
  // Register 8 b + 4 d + e of o[c] is dim 64 (c >> 1) + 16 (c & 1) + 32 b + 8 d + 4 half + e.
  int n_rep_e = a.n_rep;
  asm volatile("" : "+s"(n_rep_e));  // its division constants are not kept through the key loop
  const PrefillPart part = load_part<D>(a, n_rep_e);
  if (set == 0) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const int r = row0 + n;
    if (part.nparts == 1) {
      const int tok = r / n_rep_e;
      raw_t* op = static_cast<raw_t*>(a.out) + (qbase + tok) * a.o_st + (h * n_rep_e + r - tok * n_rep_e) * a.o_sh;
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          uint32_t w[4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            w[i] = static_cast<uint32_t>(from_f32<DTYPE>(o[c][8 * b + 2 * i] * inv)) |
                   static_cast<uint32_t>(from_f32<DTYPE>(o[c][8 * b + 2 * i + 1] * inv)) << 16;
          // half 0 / 1 hold dims (0-3, 8-11) / (4-7, 12-15) of 16: swapped to 8 in a row each
          const auto x = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
          const auto y = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
          if (r < nrows) {
            raw_t* dst = op + 64 * (c >> 1) + 16 * (c & 1) + 32 * b + 8 * half;
            if (a.out_vec) {
              *reinterpret_cast<uint4*>(dst) = make_uint4(x[0], y[0], x[1], y[1]);
            } else {
              const uint32_t e[4] = {x[0], y[0], x[1], y[1]};
#pragma unroll
              for (int i = 0; i < 8; ++i) dst[i] = static_cast<raw_t>(e[i >> 1] >> (16 * (i & 1)));
            }
          }
        }
    } else if (r < nrows) {
      // (32 rows' pairs lie together: 256 bytes a store)
      uint64_t* rec = reinterpret_cast<uint64_t*>(part.recs) +
                      static_cast<int64_t>(part.part) * part.rows_cap * (D / 2 + 1) + r;
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
          const int pair = 32 * (c >> 1) + 8 * (c & 1) + 16 * (e >> 3) + 4 * ((e >> 2) & 1) + 2 * half + ((e >> 1) & 1);
          store_coherent_u64(rec + pair * part.rows_cap, pack_f32x2(o[c][e] * inv, o[c][e + 1] * inv));
        }
      if (half == 0) store_coherent_u64(rec + D / 2 * part.rows_cap, pack_f32x2(m, l));
    }
  }
  if (part.nparts == 1) return;
  fold_parts<DTYPE, D, Tr::kThreads>(a, part, nrows, n_rep_e, qbase, h);
}

}  // namespace
}  // namespace mv
