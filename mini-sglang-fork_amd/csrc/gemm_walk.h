// Grouped (fused-MoE prefill) GEMM: a persistent walk over tall items of an
// expert's rows, gfx950 only.
//
// One block per CU (8 waves, 2 x 4 of 96 x 64) walks (expert, column tile,
// row chunk) items of up to 192 sorted rows x 256 weight rows.  What bounds
// it (profiled at E 128, top-8, H 2048, I 768): at few rows per expert the
// weight stream from HBM (300 tokens: GEMM1 reads 407 MB past L2, 403 of them
// weights, in 69.9 us = 5.8 TB/s); at 256 rows a round of one item per CU, of
// about 1.05 us per stage (its MFMAs 0.64 at the nominal rate) and 7.5 us
// besides, in which the epilogue leaves the matrix cores idle (4096 tokens:
// MFMA busy 0.32, a third of the wave cycles in waits).
//
//  * 128-byte row segments: 1.33 GB of operands move through L2 in 146 us
//    (GEMM1, 4096 tokens, 9.2 TB/s), where the 128 x 256 tiles on 64-byte
//    stages that this walk replaces took 186 us.
//  * The two operands have rings and loading waves of their own: waves 0-3
//    load A (2 slots of 24 KB: the gathered rows mostly hit in L2), waves
//    4-7 W (3 slots of 32 KB: the weights come from HBM, about 1.5 us away).
//    vmcnt retires in order, so a wave that loaded both could not wait for
//    an A stage without the W stages issued before it (one ring of two
//    stages of 320 x 256: 2.1 us per stage at 4096 tokens).  A refills go out
//    right behind the barrier, W refills behind the MFMAs, so that they do
//    not queue in front of the A loads (4096 tokens: 173 -> 159 us).
//  * Weights stream with the non-temporal policy, also where two chunks
//    share them (side by side on one XCD): they would evict the rows that
//    the expert's other column tiles re-read.
//  * The rings run on across items: the next item's first stages are issued
//    during the current item's last ones and land while it writes its
//    output.
//  * The weight rows are the MFMA's "A" operand and the token rows its "B"
//    operand, so a lane holds four consecutive output columns of one token:
//    the epilogue scales and packs them in registers, one
//    v_permlane16_swap per packed word makes them 16-byte row segments, and
//    each wave stores its own columns.  No LDS staging, no barrier, and the
//    ring keeps its slots.
//  * 16-row fragments past a chunk's last pair skip their MFMAs (one instance
//    of the stage loop per count, no branch inside); the fragments of a
//    chunk are dealt to the two wave rows in turn, so a short chunk stays
//    balanced; rows past them read zeros without traffic.
//  * Every wait counts exactly what was issued behind the stage it needs,
//    loads and stores; past the last item the loads go on through an empty
//    buffer view, so the counts stay the same.
//  * The item metadata (pair ids, row and weight scales, routed weights)
//    goes into double-buffered LDS tables by buffer_load ... lds during the
//    previous item.
//
// MI355X, weights from HBM, us per launch, 128 x 256 walk on 64-byte stages
// (300 tokens: 64 x 128 tiles) -> this walk, E 128, top-8, H 2048, I 768 at
// 300 / 1024 / 2048 / 4096 / 8192 tokens: GEMM1 with silu 79 / 85 / 118 /
// 186 / 300 -> 67 / 72 / 80 / 146 / 236; GEMM2 with the routed weight 45 /
// 59 / 86 / 129 / 218 -> 43 / 52 / 65 / 114 / 193.
#pragma once

#include "gemm_kernels.h"

namespace mw8 {

constexpr int kWalkBM = 192, kWalkBN = 256, kWalkBK = 128;
constexpr int kWalkASlots = 2, kWalkWSlots = 3;
constexpr int kWalkMinStages = 5;  // the metadata of item i + 1 lands during item i
constexpr int kWalkLds = (kWalkASlots * kWalkBM + kWalkWSlots * kWalkBN) * kWalkBK;

struct WalkItem {
  int m0, n0;      // first sorted row; first output (kAct: activation) column
  int e;           // expert
  int rows;        // sorted rows of the chunk
  int ok;          // 0: no item
};

// kAct >= 0: gate|up weights [2I, K]; the tile's 256 weight rows are 128 gate
// rows and the matching 128 up rows (32 + 32 per wave column), the output
// bf16(act_fn(g) * u) of 128 activation columns, as the separate activation
// kernel computes it from the bf16-rounded g and u.
template <int kAct>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void walk_gemm_kernel(GemmArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int BM = kWalkBM, BN = kWalkBN, BK = kWalkBK, kWaves = 8, MF = 16;
  using Mf = MfmaI8<MF>;
  using Acc = typename Mf::Acc;
  constexpr int kWM = 2, kWN = 4;                            // wave rows x wave columns
  constexpr int kFM = BM / (MF * kWM), kFN = BN / (MF * kWN);  // token x weight fragments of a wave
  constexpr int kWaveN = BN / kWN;
  constexpr int kStageA = BM * BK, kStageB = BN * BK, kRingB = kWalkASlots * kStageA;
  constexpr int kRoleWaves = kWaves / 2;                       // waves 0-3 load A, waves 4-7 load W
  constexpr int kLA = BM / (8 * kRoleWaves), kLB = BN / (8 * kRoleWaves);
  constexpr int kPairs = kAct >= 0 ? kFN / 4 : kFN / 2;        // 16-byte stores per token fragment
  constexpr int kStores = kFM * kPairs;
  constexpr int kMeta = 2;                   // metadata loads of an A wave per event
  static_assert(kFM * MF * kWM == BM && kFN * MF * kWN == BN && kFN == 4, "shape");
  static_assert(kLA * 8 * kRoleWaves == BM && kLB * 8 * kRoleWaves == BN, "DMA split");
  constexpr int kWS = kWalkWSlots;
  static_assert(kWalkASlots == 2 && kLA + kStores < 64 && (kWS - 1) * kLB + kStores < 64, "vmcnt range");
  constexpr int kTileCols = kAct >= 0 ? BN / 2 : BN;

  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ int32_t t_p[2][BM];
  __shared__ float t_sa[2][BM], t_rt[2][BM];
  __shared__ __align__(16) float t_sw[2][BN];
  __shared__ int32_t t_none[64];  // target of the metadata loads that have no table entry
  __shared__ int run_start[kPersistMaxSlots + 1], act_base[kPersistMaxSlots + 1], wave_tot[kWaves];
  static_assert(kWalkLds + 2 * 4 * (3 * BM + BN) + 256 + 4 * (2 * kPersistMaxSlots + 2 + kWaves) <= 163840,
                "LDS budget");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / kWN, wn = wave % kWN;
  const int frow = lane & 15, fgrp = lane >> 4;
  // The lane id through an empty asm: per-lane values derived from it are
  // recomputed where they are used instead of held through the K loop.
  auto opaque_lane = [] {
    int l = static_cast<int>(threadIdx.x) & 63;
    asm volatile("" : "+v"(l));
    return l;
  };

  // ---------------------------------------------------------------- walk
  const int per_tile = BM / g.align_bsz;
  bool runs = true;
  const int carry = build_run_tables<512>(g, per_tile, run_start, act_base, wave_tot, runs);
  const int N32 = static_cast<int>(g.N), half32 = N32 / 2, K32 = static_cast<int>(g.K);
  const int lda32 = static_cast<int>(g.lda), ldo32 = static_cast<int>(g.ldo);
  const int nval32 = static_cast<int>(g.num_valid);
  const int out_cols = kAct >= 0 ? half32 : N32;
  const int tn = out_cols / kTileCols, total = carry * tn;
  const int G = gridDim.x, xcd = blockIdx.x % kXcds, local = blockIdx.x / kXcds;
  const int per_xcd = G / kXcds + (xcd < G % kXcds ? 1 : 0);  // blocks on this XCD
  const int base = total / kXcds, rem = total % kXcds;
  const int begin = xcd * base + (xcd < rem ? xcd : rem), count = base + (xcd < rem ? 1 : 0);
  // item j of this block (expert-major, column tile, chunk fastest: the
  // column tiles of an expert and the chunks of a weight tile run side by
  // side on one XCD)
  auto item_of = [&](int j) -> WalkItem {
    WalkItem it{0, 0, 0, 0, 0};
    const int pos = local + j * per_xcd;
    if (pos >= count) return it;
    const int item = begin + pos;
    it.ok = 1;
    if (!runs) {  // a list that is not sorted by expert: (alignment block, column tile)
      const int b = item / tn, e = g.expert_ids[b];
      const bool real = static_cast<unsigned>(e) < static_cast<unsigned>(g.num_experts);
      it.m0 = __builtin_amdgcn_readfirstlane(b * g.align_bsz);
      it.n0 = __builtin_amdgcn_readfirstlane((item - b * tn) * kTileCols);
      it.e = __builtin_amdgcn_readfirstlane(real ? e : 0);
      it.rows = __builtin_amdgcn_readfirstlane(real ? g.align_bsz : 0);  // 0: nothing is written
      return it;
    }
    int lo = 0, hi = g.num_experts - 1;  // the expert: last e with act_base[e] * tn <= item
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (act_base[mid] * tn <= item) lo = mid; else hi = mid - 1;
    }
    const int b_first = run_start[lo], nblocks = run_start[lo + 1] - b_first;
    const int nch = (nblocks + per_tile - 1) / per_tile;
    const int off = item - act_base[lo] * tn, n_tile = off / nch, c = off % nch;
    const int c0 = b_first + c * nblocks / nch, c1 = b_first + (c + 1) * nblocks / nch;
    it.m0 = __builtin_amdgcn_readfirstlane(c0 * g.align_bsz);
    it.n0 = __builtin_amdgcn_readfirstlane(n_tile * kTileCols);
    it.e = __builtin_amdgcn_readfirstlane(lo);
    it.rows = __builtin_amdgcn_readfirstlane((c1 - c0) * g.align_bsz);
    return it;
  };
  // pair id of tile row r of an item whose sorted ids sit in t_p[par] (-1: padding or past the chunk)
  auto pair_of = [&](int par, int r, int rows) -> int32_t {
    const int32_t p = t_p[par][r];
    return r < rows && p >= 0 && p < nval32 ? p : -1;
  };
  // weight row, relative to the item's first column, of tile row r
  auto w_rel = [&](int r) -> int {
    if constexpr (kAct >= 0) {
      const int rr = r % kWaveN, a = r / kWaveN * (kWaveN / 2) + rr % (kWaveN / 2);
      return rr < kWaveN / 2 ? a : half32 + a;
    } else {
      return r;
    }
  };

  // ----------------------------------------------------------------- DMA
  // Waves 0-3 load the A stages, waves 4-7 the W stages, so that each ring
  // has its own depth: vmcnt retires in order, and a wave that loaded both
  // could not wait for an A stage without waiting for every W stage issued
  // before it.  Instruction j of a wave fills tile rows j * 32 + 8 (wave %
  // 4) .. + 7; lane -> (row, 16-byte chunk under the swizzle).  doff: the
  // lane's offsets, set per item for A (a row without a pair gets one past
  // the buffer: zeros, no traffic), once for W (the host takes whole column
  // tiles only).
  const bool role_a = wave < kRoleWaves;
  const int drow = (wave % kRoleWaves) * 8 + (lane >> 3);
  const int dchunk = 16 * ((lane & 7) ^ swz_f<BK>(drow));
  uint32_t doff[kLA > kLB ? kLA : kLB];
  auto set_rows = [&](int par, int rows) {
#pragma unroll
    for (int j = 0; j < kLA; ++j) {
      const int32_t p = pair_of(par, j * 32 + drow, rows);
      doff[j] = p >= 0 ? static_cast<uint32_t>((p / g.top_k) * lda32 + dchunk) : 0x80000000u;
    }
  };
  if (!role_a) {
#pragma unroll
    for (int j = 0; j < kLB; ++j) doff[j] = static_cast<uint32_t>(w_rel(j * 32 + drow) * K32 + dchunk);
  }
  // A stage at byte k0 of the K axis into the slot at aoff: 32 rows per
  // instruction, 4 of the 6 for chunks of up to 128 rows; ok = 0 (no item):
  // an empty buffer view, so the loads keep their count without traffic
  auto issue_a = [&](int rows, int ok, int aoff, int k0) {
    unsigned char* dst = lds + aoff + (wave % kRoleWaves) * 1024;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        scalar_ptr(const_cast<int8_t*>(g.A)), 0, ok ? 0x7fffffff : 0, kBufferFlags);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(dst + j * 4096), 16, doff[j], k0, 0, 0);
    if (rows > 128) {
#pragma unroll
      for (int j = 4; j < kLA; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(dst + j * 4096), 16, doff[j], k0, 0, 0);
    }
  };
  // W cursor: the item and byte of the K axis that the next W issue loads
  const int8_t* w_src = nullptr;
  int w_ok = 1, w_k = 0;
  auto w_base = [&](const WalkItem& it) { return g.W + (static_cast<int64_t>(it.e) * N32 + it.n0) * K32; };
  auto issue_w = [&](const WalkItem& nxt, int woff) {
    unsigned char* dst = lds + kRingB + woff + (wave % kRoleWaves) * 1024;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(scalar_ptr(const_cast<int8_t*>(w_src)), 0,
                                                                         w_ok ? 0x7fffffff : 0, kBufferFlags);
#pragma unroll
    for (int j = 0; j < kLB; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)(dst + j * 4096), 16, doff[j], w_k, 0, kStreamAux);
    w_k += BK;
    if (w_k == K32) {
      w_k = 0;
      w_src = w_base(nxt);
      w_ok = nxt.ok;
    }
  };

  // ------------------------------------------------------------ metadata
  // Two events per item, issued by the A waves (a fixed count each; a load
  // without table entries goes past its source's end into t_none): the next
  // item's pair ids and weight scales, then, from the pair ids, its row
  // scales and routed weights.
  auto rsrc_of = [](const void* p, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(scalar_ptr(const_cast<void*>(p)), 0,
                                             static_cast<int>(bytes < 0x7fffffff ? bytes : 0x7fffffff), kBufferFlags);
  };
  static_assert(BM % 64 == 0 && BM <= 256 && BN == 256 && kRoleWaves == 4, "64 table entries per A wave");
  auto meta_ids = [&](const WalkItem& it, int par) {
    const int r = 64 * wave + opaque_lane();
    const bool rw = wave < BM / 64;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rsrc_of(g.sorted_ids, 0x7fffffff), (lds_ptr_t)(rw ? &t_p[par][64 * wave] : t_none), 4,
        rw && r < it.rows ? static_cast<uint32_t>((it.m0 + r) * 4) : 0x80000000u, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_of(g.sw, 0x7fffffff), (lds_ptr_t)(&t_sw[par][64 * wave]), 4,
                                             static_cast<uint32_t>((it.e * N32 + it.n0 + w_rel(r)) * 4), 0, 0, 0);
  };
  auto meta_rows = [&](const WalkItem& it, int par) {
    const int r = 64 * wave + opaque_lane();
    const bool rw = wave < BM / 64;
    const int32_t p = rw ? pair_of(par, r, it.rows) : -1;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rsrc_of(g.sa, 0x7fffffff), (lds_ptr_t)(rw ? reinterpret_cast<int32_t*>(&t_sa[par][64 * wave]) : t_none), 4,
        p >= 0 ? static_cast<uint32_t>((p / g.top_k) * 4) : 0x80000000u, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rsrc_of(g.topk_w ? g.topk_w : g.sa, 0x7fffffff),
        (lds_ptr_t)(rw ? reinterpret_cast<int32_t*>(&t_rt[par][64 * wave]) : t_none), 4,
        p >= 0 && g.topk_w ? static_cast<uint32_t>(p * 4) : 0x80000000u, 0, 0, 0);
  };

  using kYes = std::integral_constant<bool, true>;
  using kNo = std::integral_constant<bool, false>;
  // ----------------------------------------------------------- fragments
  // Token fragment i: tile rows 16 (2 i + wm) + frow; weight fragment j:
  // tile rows kWaveN wn + 16 j + frow.  16-row steps keep the chunk swizzle.
  // Two register sets, one per 64-byte substep.
  const int a_lane[2] = {swz_lds<BK>(MF * wm + frow, 2 * fgrp), swz_lds<BK>(MF * wm + frow, 2 * fgrp + 1)};
  const int b_lane[2] = {kRingB + swz_lds<BK>(kWaveN * wn + frow, 2 * fgrp),
                         kRingB + swz_lds<BK>(kWaveN * wn + frow, 2 * fgrp + 1)};
  v4i fa[2][kFM], fb[2][kFN];
  Acc acc[kFM][kFN];
  auto read_frags = [&](auto live_tag, int aoff, int woff, int ks) {
    constexpr int kLive = decltype(live_tag)::value;
    const unsigned char* pa = lds + aoff + a_lane[ks];
    const unsigned char* pb = lds + woff + b_lane[ks];
#pragma unroll
    for (int j = 0; j < kFN; ++j) fb[ks][j] = *reinterpret_cast<const v4i*>(pb + MF * BK * j);
#pragma unroll
    for (int i = 0; i < kLive; ++i) fa[ks][i] = *reinterpret_cast<const v4i*>(pa + kWM * MF * BK * i);
  };
  auto mfmas = [&](auto live_tag, int ks) {
    constexpr int kLive = decltype(live_tag)::value;
#pragma unroll
    for (int i = 0; i < kLive; ++i)
#pragma unroll
      for (int j = 0; j < kFN; ++j) acc[i][j] = Mf::mma(fb[ks][j], fa[ks][i], acc[i][j]);
  };

  // -------------------------------------------------------------- output
  const __amdgpu_buffer_rsrc_t o_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      scalar_ptr(g.out), 0, static_cast<int>(g.num_valid * g.ldo * 2), kBufferFlags);
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float v4f __attribute__((ext_vector_type(4)));
  auto pack = [](float a, float b) {
    return __builtin_bit_cast(uint32_t, bf16x2{(__bf16)a, (__bf16)b});
  };
  auto epilogue = [&](const WalkItem& it, int par, int live, auto routed_tag) {
    constexpr bool kRouted = decltype(routed_tag)::value;
    const int lane = opaque_lane(), frow = lane & 15, fgrp = lane >> 4;
    // lane group g holds columns 4 g .. 4 g + 3 of a fragment; after the
    // swap of fragments (j, j + 1) it holds 8 columns of fragment j + (g & 1)
    // from 8 (g >> 1)
    const int col0 = it.n0 + (kAct >= 0 ? kWaveN / 2 : kWaveN) * wn + 16 * (fgrp & 1) + 8 * (fgrp >> 1);
#pragma unroll
    for (int i = 0; i < kFM; ++i) {
      if (i >= live) break;  // wave-uniform
      const int r = MF * (kWM * i + wm) + frow;
      const int32_t p = pair_of(par, r, it.rows);
      const float sa = t_sa[par][r];
      float rt = 1.0f;
      if constexpr (kRouted) rt = t_rt[par][r];
      const uint32_t row_off = static_cast<uint32_t>(p) * static_cast<uint32_t>(ldo32 * 2);
      // packed bf16 columns of fragment j (gate or plain)
      auto val = [&](int j, int v, const v4f& sw) {
        float t = epi_scale(acc[i][j][v], sa, sw[v]);
        if constexpr (kRouted) t = t * rt;
        return t;
      };
      auto frag = [&](int j) -> uint2 {
        const v4f sw = *reinterpret_cast<const v4f*>(&t_sw[par][kWaveN * wn + 16 * j + 4 * fgrp]);
        if constexpr (kAct >= 0) {
          const v4f su = *reinterpret_cast<const v4f*>(&t_sw[par][kWaveN * wn + kWaveN / 2 + 16 * j + 4 * fgrp]);
          float a[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float gv = static_cast<float>((__bf16)val(j, v, sw));
            const float uv = static_cast<float>((__bf16)val(j + kFN / 2, v, su));
            a[v] = act_fn<kAct>(gv) * uv;
          }
          return make_uint2(pack(a[0], a[1]), pack(a[2], a[3]));
        } else {
          return make_uint2(pack(val(j, 0, sw), val(j, 1, sw)), pack(val(j, 2, sw), val(j, 3, sw)));
        }
      };
#pragma unroll
      for (int q = 0; q < kPairs; ++q) {
        const uint2 x = frag(2 * q), y = frag(2 * q + 1);
        const auto s0 = __builtin_amdgcn_permlane16_swap(x.x, y.x, false, false);
        const auto s1 = __builtin_amdgcn_permlane16_swap(x.y, y.y, false, false);
        const v4i d = {static_cast<int>(s0[0]), static_cast<int>(s1[0]), static_cast<int>(s0[1]),
                       static_cast<int>(s1[1])};
        const int c = col0 + 32 * q;
        const uint32_t voff = p >= 0 ? row_off + static_cast<uint32_t>(c * 2) : 0x80000000u;
        __builtin_amdgcn_raw_buffer_store_b128(d, o_rsrc, voff, 0, kStreamAux);
      }
    }
  };

  // ---------------------------------------------------------------- main
  WalkItem cur = item_of(0);
  if (!cur.ok) return;  // block-uniform
  const int nk = K32 / BK;
  int par = 0, jn = 1;
  int aoff = 0, woff = 0;  // ring slots (byte offsets) of the stage being consumed
  // first item: the W waves start its weights at once; the A waves fetch its
  // pair ids (and weight scales), then start its rows and the metadata that
  // the ids lead to
  if (!role_a) {
    w_src = w_base(cur);
#pragma unroll
    for (int st = 0; st < kWS; ++st) issue_w(cur, st * kStageB);
  } else {
    const int32_t p = tid < cur.rows ? g.sorted_ids[cur.m0 + tid] : -1;
    t_sw[0][tid] = g.sw[static_cast<int64_t>(cur.e) * N32 + cur.n0 + w_rel(tid)];
    if (tid < BM) t_p[0][tid] = p;
  }
  wait_vmcnt_lgkm0<63>();
  raw_barrier();
  if (role_a) {
    set_rows(0, cur.rows);
    issue_a(cur.rows, 1, 0, 0);
    issue_a(cur.rows, 1, kStageA, BK);
    meta_rows(cur, 0);
  }
  int stored = 0;  // the previous item's token fragments that this wave stored
  // wait until at most n loads and that item's stores are outstanding
  auto wait_past = [&](auto n_tag) {
    constexpr int n = decltype(n_tag)::value;
    switch (stored) {
      case 0: wait_vmcnt_lgkm0<n>(); break;
      case 1: wait_vmcnt_lgkm0<n + kPairs>(); break;
      case 2: wait_vmcnt_lgkm0<n + 2 * kPairs>(); break;
      case 3: wait_vmcnt_lgkm0<n + 3 * kPairs>(); break;
      case 4: wait_vmcnt_lgkm0<n + 4 * kPairs>(); break;
      case 5: wait_vmcnt_lgkm0<n + 5 * kPairs>(); break;
      default: wait_vmcnt_lgkm0<n + 6 * kPairs>(); break;
    }
  };
  static_assert(kFM == 6, "wait_past");
  for (;;) {
    const WalkItem nxt = item_of(jn++);
    int live;
    {  // this wave's token fragments up to the chunk's last pair
      int end = 0;
#pragma unroll
      for (int h = 0; h < BM; h += 64) {
        const uint64_t pairs = __ballot(pair_of(par, h + opaque_lane(), cur.rows) >= 0);
        if (pairs) end = h + 64 - __clzll(pairs);
      }
      const int frags = (end + MF - 1) / MF - wm;  // fragments wm, wm + 2, ... are this wave's
      live = __builtin_amdgcn_readfirstlane(frags > 0 ? (frags + kWM - 1) / kWM : 0);
    }
#pragma unroll
    for (int i = 0; i < kFM; ++i)
#pragma unroll
      for (int j = 0; j < kFN; ++j) acc[i][j] = Acc{0};
    auto advance = [&] {
      aoff = kStageA - aoff;
      woff = woff == (kWS - 1) * kStageB ? 0 : woff + kStageB;
    };
    // K stage kt but the last, with kLive token fragments: its substep 0,
    // the barrier behind which its slots are free and stage kt + 1 has
    // landed, the refills, its substep 1.  The A refill goes out at once (an
    // A stage has one stage of time to arrive), the W refill behind the
    // MFMAs, so that it does not queue in front of the A loads.
    auto step = [&](auto live_tag, auto last_tag, int kt) {
      constexpr bool kLast = decltype(last_tag)::value;  // stage nk - 2: A moves on to the next item
      read_frags(live_tag, aoff, woff, 1);
      mfmas(live_tag, 0);
      // Issued behind A stage kt + 1: in iterations 1 and 3 the metadata
      // loads of the iteration before, else nothing (A stage 1 landed with
      // stage 0).  Behind W stage kt + 1: W stage kt + 2, and in iterations
      // 0 and 1 the previous item's stores.
      if (role_a) {
        if (kt >= 4) wait_vmcnt_lgkm0<0>();
        else if (kt == 0) wait_vmcnt_lgkm0<63>();
        else if (kt == 2) wait_vmcnt_lgkm0<0>();
        else wait_vmcnt_lgkm0<kMeta>();
      } else {
        if (kt >= kWS - 1) wait_vmcnt_lgkm0<(kWS - 2) * kLB>();
        else wait_past(std::integral_constant<int, (kWS - 2) * kLB>{});
      }
      raw_barrier();
      const int a0 = aoff, w0 = woff;
      if (role_a) {
        if constexpr (kLast) {
          set_rows(par ^ 1, nxt.rows);
          issue_a(nxt.rows, nxt.ok, a0, 0);
        } else {
          issue_a(cur.rows, 1, a0, (kt + 2) * BK);
          if (kt <= 2) {
            if (kt == 0) meta_ids(nxt, par ^ 1);
            if (kt == 2) meta_rows(nxt, par ^ 1);
          }
        }
      }
      advance();
      read_frags(live_tag, aoff, woff, 0);
      mfmas(live_tag, 1);
      if (!role_a) issue_w(nxt, w0);
    };
    // The waves of a block may run different instances: each executes the
    // same barriers and issues the same loads.
    auto stages = [&](auto live_tag) {
      // Stage 0 landed.  Behind it: W stages 1 .. kWS - 1 and the previous
      // item's stores (A stage 1 has landed as well then).
      if (role_a) wait_past(std::integral_constant<int, 0>{});
      else wait_past(std::integral_constant<int, (kWS - 1) * kLB>{});
      raw_barrier();
      read_frags(live_tag, aoff, woff, 0);
#pragma clang loop unroll(disable)
      for (int kt = 0; kt < nk - 2; ++kt) step(live_tag, kNo{}, kt);
      step(live_tag, kYes{}, nk - 2);
      read_frags(live_tag, aoff, woff, 1);
      mfmas(live_tag, 0);
      wait_vmcnt_lgkm0<63>();
      raw_barrier();  // every wave is past its reads of stage nk - 1
      if (role_a) issue_a(nxt.rows, nxt.ok, aoff, BK);
      else issue_w(nxt, woff);
      advance();
      mfmas(live_tag, 1);
    };
    if (live >= 6) stages(std::integral_constant<int, 6>{});
    else if (live == 5) stages(std::integral_constant<int, 5>{});
    else if (live == 4) stages(std::integral_constant<int, 4>{});
    else if (live == 3) stages(std::integral_constant<int, 3>{});
    else if (live == 2) stages(std::integral_constant<int, 2>{});
    else stages(std::integral_constant<int, 1>{});  // at most one (a fragment of zeros if none)
    if (g.topk_w) epilogue(cur, par, live, kYes{});
    else epilogue(cur, par, live, kNo{});
    if (!nxt.ok) break;
    cur = nxt;
    par ^= 1;
    stored = live < kFM ? live : kFM;
  }
  wait_vmcnt_lgkm0<0>();  // no load may write to LDS after the block has ended
#endif  // __HIP_DEVICE_COMPILE__
}

}  // namespace mw8
