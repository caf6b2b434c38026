// Pipelined persistent ring GEMM ("stream" kernel), gfx950 only.
//
// One block per CU (8 waves of 64 x BN/2, v_mfma_i32_16x16x64_i8, a ring of
// two 128-byte K stages moved global -> LDS with buffer_load ... lds) walks
// a list of BM x BN output tiles of a dense grid.  Unlike one tile per
// block, the walk does not drain between tiles:
//
//  * the DMA ring runs on across items: the next item's first two stages
//    are issued during the current item's last two, so they land while the
//    current item finishes its MFMAs and writes its output;
//  * the epilogue writes through a small per-wave LDS slice (8 rows per
//    pass, no block barrier) with a fixed number of 16-byte buffer stores
//    per wave (a row or column outside the output gets an offset past the
//    buffer, which the hardware drops).  Vector memory operations retire in
//    issue order and vmcnt counts stores as well as loads, so the waits for
//    the next item's first stages count the stores exactly and do not wait
//    for them: the output write burst of item i overlaps item i+1's loads;
//  * the item metadata (row and column scales, bias) goes straight into
//    double-buffered LDS tables by buffer_load ... lds, a fixed count per
//    wave issued in the item's first stage behind that stage's refill DMA;
//    the next wait counts it, the one after drains it.  No loaded value is
//    held in registers across the K loop, and the walk never spills (a
//    scratch access would be a vector memory operation the waits do not
//    count; the build checks for it).
//
// An item needs at least 6 K stages (K >= 768); the host uses the one-tile
// kernels otherwise.  bf16 output only (the int32 parity hook stays on the
// one-tile kernels); no K split.
#pragma once

#include "gemm_kernels.h"

namespace mw8 {

// Offsets are 32-bit: the host keeps A, W, the output and every metadata
// array below 2^31 bytes.
struct StreamItem {
  int m0, n0;      // first row; first output column
  int rows_valid;  // rows of the tile that hold rows of A
  int ok;          // 0: no item
};

constexpr int kStreamBM = 256, kStreamBK = 128, kStreamMinStages = 6;

// Dynamic LDS of a stream launch: the ring plus eight 8-row staging slices.
template <int BN>
constexpr int stream_lds_bytes() {
  return 2 * (kStreamBM + BN) * kStreamBK + 8 * 8 * (BN / 2) * 2;
}

template <int BN>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void stream_gemm_kernel(GemmArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int BM = kStreamBM, BK = kStreamBK, WN = 2, kWaves = 8, MF = 16;
  using Mf = MfmaI8<MF>;
  using Acc = typename Mf::Acc;
  constexpr int kWaveM = 64, kWaveN = BN / WN, kFM = kWaveM / MF, kFN = kWaveN / MF;
  constexpr int kStageA = BM * BK, kStageB = BN * BK, kStage = kStageA + kStageB, kRing = 2 * kStage;
  constexpr int kLA = BM / (8 * kWaves), kLB = BN / (8 * kWaves), kL = kLA + kLB;
  // staging: 8 rows of the wave's output columns
  constexpr int kStgRow = kWaveN * 2, kStgChunks = kStgRow / 16, kStg = 8 * kStgRow;
  constexpr int kReadsPerPass = kStg / 1024;          // 16-byte reads (and stores) per lane and pass
  constexpr int kStores = kFM * 2 * kReadsPerPass;     // buffer stores per wave and item
  static_assert(kFN % 2 == 0, "shape");
  static_assert(kStg % 1024 == 0 && (kStgChunks == 8 || kStgChunks == 16), "staging slice");
  static_assert(2 * kL + kStores + 8 < 64, "vmcnt range (two stages, the stores, the metadata loads)");
  static_assert(kRing + 8 * kStg == stream_lds_bytes<BN>(), "LDS layout");

  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ float t_sa[2][BM], t_sw[2][BN];
  __shared__ uint32_t t_bias[2][BN / 2];  // bf16 bias of columns 2 i, 2 i + 1
  static_assert(stream_lds_bytes<BN>() + 4 * (2 * BM + 2 * BN) + 4 * BN <= 163840, "LDS budget");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int frow = lane & 15, fgrp = lane >> 4;
  // The lane id through an empty asm: per-lane values derived from it are
  // recomputed where they are used instead of being hoisted out of the walk
  // (the walk has no registers to keep them in, and a spill would be a
  // vector memory operation that the waits do not count).
  auto opaque_lane = [] {
    int l = static_cast<int>(threadIdx.x) & 63;
    asm volatile("" : "+v"(l));
    return l;
  };

  // ---------------------------------------------------------------- walk
  const int G = gridDim.x, xcd = blockIdx.x % kXcds, local = blockIdx.x / kXcds;
  const int per_xcd = G / kXcds + (xcd < G % kXcds ? 1 : 0);  // blocks on this XCD
  const uint32_t tm_d = static_cast<uint32_t>((g.M + BM - 1) / BM);
  const int tn = static_cast<int>((g.N + BN - 1) / BN), total = static_cast<int>(tm_d) * tn;
  const int base = total / kXcds, rem = total % kXcds;
  const int begin = xcd * base + (xcd < rem ? xcd : rem), count = base + (xcd < rem ? 1 : 0);
  const int rot = xcd * count / kXcds;  // XCD x starts x/8 of the way into its range
  auto item_of = [&](int j) -> StreamItem {
    StreamItem it{0, 0, BM, 0};
    const int pos = local + j * per_xcd;
    if (pos >= count) return it;
    it.ok = 1;
    const uint32_t t = static_cast<uint32_t>(begin + (pos + rot) % count);
    int64_t pm, pn;
    tile_of_index(t, tm_d, static_cast<uint32_t>(tn), pm, pn);
    it.m0 = __builtin_amdgcn_readfirstlane(static_cast<int>(pm) * BM);
    it.n0 = __builtin_amdgcn_readfirstlane(static_cast<int>(pn) * BN);
    const int rv = static_cast<int>(g.M) - it.m0;
    it.rows_valid = __builtin_amdgcn_readfirstlane(rv < BM ? rv : BM);
    return it;
  };

  const int N32 = static_cast<int>(g.N), K32 = static_cast<int>(g.K), lda32 = static_cast<int>(g.lda);
  const int ldo32 = static_cast<int>(g.ldo), M32 = static_cast<int>(g.M);
  // weight row of tile row r of item `it`
  auto w_row_of = [&](const StreamItem& it, int r) -> int { return it.n0 + r < N32 ? it.n0 + r : N32 - 1; };

  // ------------------------------------------------- DMA of the issue item
  // The item whose stages the ring loads (the current item, from its
  // iteration nk-2 on the next one).  The per-lane source offsets are
  // recomputed at every issue from these scalars (a few dozen VALU
  // operations per 128-byte stage) rather than held in registers through the
  // walk.
  StreamItem iss{0, 0, BM, 0};
  auto issue = [&](int slot, int kt) {
    unsigned char* base = lds + slot * kStage;
    const int k0 = kt * BK, ln = opaque_lane();
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        scalar_ptr(const_cast<int8_t*>(g.A + static_cast<int64_t>(iss.m0) * g.lda)), 0, 0x7fffffff, kBufferFlags);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        scalar_ptr(const_cast<int8_t*>(g.W + static_cast<int64_t>(iss.n0) * g.K)), 0, 0x7fffffff, kBufferFlags);
#pragma unroll
    for (int j = 0; j < kLA; ++j) {
      const int unit = (j * kWaves + wave) * 64 + ln, row = unit / 8;
      const int c = (unit % 8) ^ swz_f<BK>(row);
      const int arow = iss.m0 + row < M32 ? row : M32 - 1 - iss.m0;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr_t)(base + (j * kWaves + wave) * 1024), 16,
                                               static_cast<uint32_t>(arow * lda32 + 16 * c), k0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < kLB; ++j) {
      const int unit = (j * kWaves + wave) * 64 + ln, row = unit / 8;
      const int c = (unit % 8) ^ swz_f<BK>(row);
      const uint32_t off = static_cast<uint32_t>((w_row_of(iss, row) - iss.n0) * K32 + 16 * c);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (lds_ptr_t)(base + kStageA + (j * kWaves + wave) * 1024), 16,
                                               off, k0, 0, 0);
    }
  };

  // ------------------------------------------------------------ metadata
  // buffer_load ... lds of 64 table entries each, kMetaLo per wave for waves
  // 0-3 and kMetaHi for waves 4-7 (unconditional: a fixed count):
  //   waves 0-3: row scales t_sa (rows 64 w ..) and weight scales t_sw
  //              (columns 64 w ..);
  //   waves 4-7: bias (waves 4-5: columns 2 l, 2 l + 1 of t_bias entry
  //              l = 64 (w - 4) + lane, one dword each; waves 6-7 reload
  //              entries of waves 4-5), a dummy source when the pointer is
  //              null (the value is then unused).
  constexpr int kMetaLo = 2, kMetaHi = 1;
  auto meta_dma = [&](const StreamItem& cur, int par) {
    const int w4 = wave & 3, r = 64 * w4 + opaque_lane();
    auto rsrc = [](const void* p) {
      return __builtin_amdgcn_make_buffer_rsrc(scalar_ptr(const_cast<void*>(p)), 0, 0x7fffffff, kBufferFlags);
    };
    const int pv = cur.m0 + r < M32 ? cur.m0 + r : M32 - 1;
    const int wr = w_row_of(cur, r);
    if (wave < 4) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc(g.sa), (lds_ptr_t)(&t_sa[par][64 * w4]), 4,
                                               static_cast<uint32_t>(pv * 4), 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc(g.sw), (lds_ptr_t)(&t_sw[par][64 * w4]), 4,
                                               static_cast<uint32_t>(wr * 4), 0, 0, 0);
    } else {
      const int e2 = 64 * (w4 & 1) + opaque_lane();                      // t_bias entry: columns 2 e2, 2 e2 + 1
      const int c2 = cur.n0 + 2 * e2 < N32 ? cur.n0 + 2 * e2 : N32 - 2;  // N % 8 == 0 (staged output)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc(g.bias ? static_cast<const void*>(g.bias) : g.sw),
                                               (lds_ptr_t)(&t_bias[par][64 * (w4 & 1)]), 4,
                                               static_cast<uint32_t>((g.bias ? c2 : 0) * 2), 0, 0, 0);
    }
  };

  // ----------------------------------------------------------- fragments
  // fragment rows wm*64 + 16 i + frow (A) and wn*kWaveN + 16 j + frow (B)
  // share their low 4 bits, and so the chunk swizzle: one lane offset per
  // operand and substep, the fragments 16 rows (2 KB) apart
  const int a_lane[2] = {swz_lds<BK>(wm * kWaveM + frow, 2 * fgrp), swz_lds<BK>(wm * kWaveM + frow, 2 * fgrp + 1)};
  const int b_lane[2] = {kStageA + swz_lds<BK>(wn * kWaveN + frow, 2 * fgrp),
                         kStageA + swz_lds<BK>(wn * kWaveN + frow, 2 * fgrp + 1)};
  v4i fa[2][kFM], fb[kFN];
  Acc acc[kFM][kFN];
  auto read_a = [&](int slot, int ks, int set) {
    const unsigned char* la = lds + slot * kStage + a_lane[ks];
#pragma unroll
    for (int i = 0; i < kFM; ++i) fa[set][i] = *reinterpret_cast<const v4i*>(la + MF * BK * i);
  };
  auto read_b = [&](int slot, int ks, int j) {
    fb[j] = *reinterpret_cast<const v4i*>(lds + slot * kStage + b_lane[ks] + MF * BK * j);
  };
  auto col = [&](int set, int j) {
#pragma unroll
    for (int i = 0; i < kFM; ++i) acc[i][j] = Mf::mma(fa[set][i], fb[j], acc[i][j]);
  };

  // -------------------------------------------------------------- output
  const __amdgpu_buffer_rsrc_t o_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      scalar_ptr(g.out), 0, static_cast<int>(g.M * g.ldo * 2), kBufferFlags);
  unsigned char* stg = lds + kRing + wave * kStg;
  auto sw_row = [](int srow) { return kStgChunks == 16 ? 2 * srow : 2 * (srow >> 1); };
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  auto epilogue_tagged = [&](const StreamItem& it, int par, auto bias_tag) {
    constexpr bool has_bias = decltype(bias_tag)::value;
#pragma unroll
    for (int i = 0; i < kFM; ++i) {
#pragma unroll
      for (int vp = 0; vp < 2; ++vp) {
        const int lane = opaque_lane(), frow = lane & 15, fgrp = lane >> 4;
        const bool odd = (lane & 1) != 0;
        const int srow = 2 * fgrp + (odd ? 1 : 0);  // staged row of this lane's word
        const int v0 = 2 * vp;
        const int r0 = wm * kWaveM + MF * i + 4 * fgrp + v0;  // this lane's rows r0, r0 + 1
        const float sa0 = t_sa[par][r0], sa1 = t_sa[par][r0 + 1];
        auto val = [&](int j, int v) {
          const int c = wn * kWaveN + MF * j + frow;
          float t = epi_scale(acc[i][j][v], v == v0 ? sa0 : sa1, t_sw[par][c]);
          if constexpr (has_bias) t = t + bf16_to_f32(static_cast<uint16_t>(t_bias[par][c >> 1] >> (16 * (c & 1))));
          return t;
        };
        auto put = [&](int cl, float t0, float t1) {  // cl: this lane's column in the slice
          const float send = odd ? t0 : t1;
          const float got = __builtin_bit_cast(
              float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, send), 0xB1, 0xF, 0xF, false));
          const bf16x2 pr = odd ? bf16x2{(__bf16)got, (__bf16)t1} : bf16x2{(__bf16)t0, (__bf16)got};
          const int cc = odd ? cl - 1 : cl;
          *reinterpret_cast<bf16x2*>(stg + srow * kStgRow + (((cc >> 3) ^ sw_row(srow)) << 4) + (cc & 7) * 2) = pr;
        };
#pragma unroll
        for (int j = 0; j < kFN; ++j) put(MF * j + frow, val(j, v0), val(j, v0 + 1));
        // the slice holds tile rows wm*64 + 16 i + 4 (s / 2) + v0 + (s & 1), s = 0..7;
        // each lane writes kReadsPerPass 16-byte chunks of it (the wave's own
        // LDS slice: its LDS operations execute in order, no barrier)
        asm volatile("" ::: "memory");
#pragma unroll
        for (int q = 0; q < kReadsPerPass; ++q) {
          const int u = q * 64 + lane, sr = u / kStgChunks, ch = u % kStgChunks;
          const v4i d = *reinterpret_cast<const v4i*>(stg + sr * kStgRow + ((ch ^ sw_row(sr)) << 4));
          const int r = wm * kWaveM + MF * i + 4 * (sr >> 1) + v0 + (sr & 1);
          const int orow = r < it.rows_valid ? it.m0 + r : -1;
          const int ocol = it.n0 + wn * kWaveN + ch * 8;
          const uint32_t voff = orow >= 0 && ocol < N32
                                    ? static_cast<uint32_t>(orow) * static_cast<uint32_t>(ldo32 * 2) +
                                          static_cast<uint32_t>(ocol * 2)
                                    : 0x80000000u;
          __builtin_amdgcn_raw_buffer_store_b128(d, o_rsrc, voff, 0, kStreamAux);
        }
        asm volatile("" ::: "memory");
      }
    }
  };

  auto epilogue = [&](const StreamItem& it, int par) {
    if (g.bias)
      epilogue_tagged(it, par, std::integral_constant<bool, true>{});
    else
      epilogue_tagged(it, par, std::integral_constant<bool, false>{});
  };

  // ---------------------------------------------------------------- main
  StreamItem cur = item_of(0);
  if (!cur.ok) return;  // block-uniform
  const int nk = static_cast<int>(g.K / BK);
  int par = 0, gbase = 0, jn = 1;
  iss = cur;
  issue(0, 0);
  issue(1, 1);
  bool first = true;
  for (;;) {
    const StreamItem nxt = item_of(jn++);
#pragma unroll
    for (int i = 0; i < kFM; ++i)
#pragma unroll
      for (int j = 0; j < kFN; ++j) acc[i][j] = Acc{0};
    auto slot = [&](int kt) { return (gbase + kt) & 1; };
    // stage 0 landed: after it were issued stage 1 and, past the first
    // item, the previous item's stores
    if (first) wait_vmcnt_lgkm0<kL>(); else wait_vmcnt_lgkm0<kL + kStores>();
    raw_barrier();
    read_a(slot(0), 0, 0);
#pragma unroll
    for (int j = 0; j < kFN; ++j) read_b(slot(0), 0, j);
    for (int kt = 0; kt + 1 < nk; ++kt) {
      read_a(slot(kt), 1, 1);
#pragma unroll
      for (int j = 0; j < kFN; ++j) {
        col(0, j);
        read_b(slot(kt), 1, j);
      }
      // stage kt+1 landed.  Issued after it: in iteration 0 the previous
      // item's stores (kStores per wave), in iteration 1 this item's
      // metadata DMA (kMetaLo / kMetaHi per wave), later nothing
      if (kt == 0) {
        if (first) wait_vmcnt_lgkm0<0>(); else wait_vmcnt_lgkm0<kStores>();
      } else if (kt == 1) {
        if (wave < 4) wait_vmcnt_lgkm0<kMetaLo>(); else wait_vmcnt_lgkm0<kMetaHi>();
      } else {
        wait_vmcnt_lgkm0<0>();
      }
      raw_barrier();  // from kt == 2 on, this item's metadata is in the tables
      read_a(slot(kt + 1), 0, 0);
#pragma unroll
      for (int j = 0; j < kFN; ++j) {
        col(1, j);
        read_b(slot(kt + 1), 0, j);
      }
      if (kt + 2 < nk) {
        issue(slot(kt + 2), kt + 2);
      } else if (nxt.ok) {  // kt == nk - 2: the next item's stage 0
        iss = nxt;
        issue(slot(kt + 2), 0);
      }
      if (kt == 0) meta_dma(cur, par);
    }
    read_a(slot(nk - 1), 1, 1);
#pragma unroll
    for (int j = 0; j < kFN; ++j) {
      col(0, j);
      read_b(slot(nk - 1), 1, j);
    }
    // every wave is past its reads of stage nk-1: its slot takes the next item's stage 1
    wait_vmcnt_lgkm0<63>();
    raw_barrier();
    if (nxt.ok) issue(slot(nk + 1), 1);
#pragma unroll
    for (int j = 0; j < kFN; ++j) col(1, j);
    epilogue(cur, par);
    if (!nxt.ok) break;
    cur = nxt;
    par ^= 1;
    gbase += nk;
    first = false;
  }
#endif  // __HIP_DEVICE_COMPILE__
}

}  // namespace mw8
