// Tile table of the grouped expert GEMMs and the launch of one (element type, epilogue)
// combination.  Each combination is instantiated in its own translation unit
// (moe_gemm_inst_*.hip) so that the library builds in parallel; moe_gemm.hip sees only
// the declaration of dispatch_block.
#pragma once
#include "moe_gemm_quad.h"

namespace fr {

// ---- host side ----------------------------------------------------------------
// Token-block sizes and their tile shapes.  K tiles are 128 bytes per row (256 for
// the 16-row block); every block except 64 streams tiles HBM -> LDS directly.
//   256 / 128 rows: 8 wavefronts, 32x32 MFMA, 2- or 3-slot ring (compute-bound regime);
//                   in the 256-row tile one wavefront per SIMD issues the loads of both;
//   64 rows:        3-slot ring, 8 wavefronts (4 with 256-byte row segments for the gate/up GEMM, persistent);
//                   (the register-staged double buffer of STAGES == 0 is no longer used by any tile);
//   32 / 16 rows:   decode regime, 16x16 MFMA, 2- or 3-slot ring, two or more workgroups per CU (the 16-row tile
//                   persistent or plain, see dispatch_block): weight streaming at HBM rate.  The gate/up GEMM
//                   streams long weight rows faster in 512-byte segments: T32L (when H allows), T16L (rows over 2 KB, fp8 4 KB).
template <typename T> struct Tiles {  // bf16 / fp16
  typedef Cfg<256, 256, 128, 2, 4, 32, 1, 2, 0, 2> T256;
  // The same tile on v_mfma_f32_16x16x32: half the accumulator-register traffic per flop of the 32x32x16 shape.
  // The part's clock under MFMA load follows the power drawn: a pure stream of 16x16x32 MFMAs holds 2.0 GHz where
  // 32x32x16 holds 1.4-1.8 GHz.  One fragment buffer (the second would not fit next to 128 accumulators and two
  // address sets).  Gate/up at 4096 / 16384 tokens: -2.5 % / -5 %, down projection -3 % / -4 %; with a short K loop
  // (2048: half as many K tiles to spread a tile's hand-over on) it loses 4 %, hence kSmallMfmaMinK.
  typedef Cfg<256, 256, 128, 2, 4, 16, 1, 2, 0, 2> T256S;
  typedef T256 T256G;
  typedef Cfg<128, 256, 128, 2, 4, 32, 1, 3, 3> T128;
  typedef Cfg<128, 256, 128, 2, 4, 16, 1, 3, 0, 2> T128P;  // persistent form; one wavefront per SIMD issues the loads (2-4 % over each its own); 16x16x32 MFMAs: 2-3 % over 32x32x16
  // 160 token rows on the same three-slot ring: 159744 bytes, with the walk table all 160 KB of a CU.  A quarter more
  // rows per pass of an expert's weight tiles through LDS, and room for the spread of the experts' loads around a
  // multiple of 128 (n pairs on E experts: n/E +- sqrt(n/E) rows each, so with n/E = 128, 256, 512 every other expert
  // needs one 128-row block more than n/E / 128).  Five token tiles x four weight tiles per wavefront, five of the
  // thirteen loads per issuing wavefront and K tile for the token rows.
  typedef Cfg<160, 256, 128, 2, 4, 16, 1, 3, 0, 2> T160P;
  typedef Cfg<64, 256, 128, 2, 4, 32, 1, 3, 3> T64;    // 3-slot ring like the 128-row tile (5 % over the register-staged form)
  typedef Cfg<64, 128, 256, 2, 2, 32, 1, 3> T64U;      // gate/up: 256-byte row segments, 4 wavefronts (another 5 %)
  typedef Cfg<32, 128, 128, 1, 4, 16, 2, 3> T32;
  // Two slots (40 KB: four workgroups per CU) instead of three (two), for long K slices of rows a power of two long, see dispatch_block
  typedef Cfg<32, 128, 128, 1, 4, 16, 2, 2> T32D;
  typedef Cfg<32, 128, 128, 1, 4, 16, 2, 4> T32S;  // four slots (80 KB) for short K slices, see dispatch_block
  typedef Cfg<16, 64, 256, 1, 2, 16, 2, 3> T16;
  typedef Cfg<32, 128, 512, 1, 4, 16, 1, 2> T32L;
  typedef Cfg<16, 64, 512, 1, 2, 16, 2, 2> T16L;
  typedef Cfg<32, 64, 256, 1, 2, 16, 2, 3> T32N;   // see dispatch_block
  typedef Cfg<64, 256, 128, 2, 4, 16, 1, 3> T64W;
  typedef Cfg<64, 128, 256, 2, 2, 16, 1, 3> T64N;
};
constexpr int kShortRow = 4096;  // bytes of a gate/up weight row up to which the 32- and 64-row tiles of 2-byte operands have forms of their own
template <> struct Tiles<fp8_t> {  // the 16x16x128 MFMA eats 256 bytes of K per two K-steps
  // every wavefront issues its own tile loads: half the address registers per wavefront (the persistent down
  // projection spills 16 instead of 57 registers: 586 vs 595 us at M=4096 although no wavefront can then skip an
  // all-padding half tile; the plain gate/up kernel is unchanged)
  typedef Cfg<256, 256, 128, 2, 4, 32, 1, 2, 0, 1> T256G;  // gate/up GEMM (plain kernel, two fragment buffers)
  typedef Cfg<256, 256, 128, 2, 4, 32, 1, 2, 0, 1> T256;
  typedef T256 T256S;
  typedef Cfg<128, 256, 128, 2, 4, 32, 1, 3, 3> T128;
  typedef Cfg<128, 256, 128, 2, 4, 32, 1, 3, 0, 2> T128P;
  typedef Cfg<160, 256, 128, 2, 4, 16, 1, 3, 0, 2> T160P;  // on the 16x16x128 MFMA (80 rows per wavefront are no multiple of 32)
  typedef Cfg<64, 256, 128, 2, 4, 32, 1, 3, 3> T64;
  typedef Cfg<64, 128, 256, 2, 2, 32, 1, 3> T64U;
  typedef Cfg<32, 128, 256, 1, 4, 16, 2, 2> T32;
  typedef Cfg<16, 64, 256, 1, 2, 16, 2, 3> T16;
  typedef Cfg<32, 128, 512, 1, 4, 16, 1, 2> T32L;
  typedef Cfg<16, 64, 512, 1, 2, 16, 2, 2> T16L;
};

constexpr int kSmallMfmaMinK = 4096;  // K from which the 256-row tile of 2-byte operands takes the 16x16x32 MFMA form

inline bool valid_block(int block) { return block == 16 || block == 32 || block == 64 || block == 128 || block == 160 || block == 256; }
inline int elem_bytes(int dtype) { return dtype == FR_FP8_E4M3 ? 1 : 2; }
inline int tile_k_bytes(int block, int dtype) { return (block == 16 || (block == 32 && dtype == FR_FP8_E4M3)) ? 256 : 128; }
inline int k_multiple(int dtype, int block) { return tile_k_bytes(block, dtype) / elem_bytes(dtype); }

template <typename T, int EPI>
int dispatch_block(GemmArgs a, int block, int splits, int64_t sorted_len, hipStream_t st) {
  typedef Tiles<T> TL;
  auto fill = [&](int BT, int BF, int bkb) {
    const int bk = bkb / static_cast<int>(sizeof(T));
    a.num_t_blocks = static_cast<int>(ceil_div(sorted_len, BT));
    const int fper = (EPI == EPI_SILU) ? BF / 2 : BF;
    a.num_f_tiles = static_cast<int>(ceil_div(a.N, fper));
    a.group_t = tunables().group_m ? tunables().group_m : (BT >= 64 ? 4 : 8);
    a.k_per_split = static_cast<int>(round_up(ceil_div(a.K, splits), bk));
  };
  switch (block) {
    case 256:
      fill(256, TL::T256::BF, TL::T256::BKB);
      // One workgroup per CU: the persistent form hides each tile's ring fill and drain behind its
      // neighbour's.  fp8 runs it with one fragment buffer (registers for the second address set): 4-5 %
      // faster for the down projection, but 6 % slower for the gate/up GEMM (short K, register-starved
      // epilogue: the hand-off K tiles spill; without the hand-off it is within 1 % of the plain kernel),
      // which keeps the plain kernel.
      // Before either: one wavefront per SIMD, tiles as tall as the experts' runs (see moe_gemm_quad.h), where its K loop is
      // long enough.
      if constexpr (EPI != EPI_DOWN) {
        if (!tunables().no_quad) {
          const int rc = launch_gemm_quad<T, EPI>(a, 256, splits, st);
          if (rc != 1) return rc;
        }
      }
      if constexpr (sizeof(T) == 1 && EPI == EPI_SILU) return launch_gemm<T, typename TL::T256G, EPI>(a, splits, st);
      else {
        // 2-byte operands, long K: the 16x16x32 MFMA form (see Tiles::T256S)
        if constexpr (sizeof(T) == 2) {
          if (a.K >= kSmallMfmaMinK) return launch_gemm_persistent<T, typename TL::T256S, EPI>(a, splits, st);
        }
        return launch_gemm_persistent<T, typename TL::T256, EPI>(a, splits, st);
      }
    case 128:
      if constexpr (EPI != EPI_DOWN) {
        if (a.any_height) {  // tiles as tall as the experts' runs
          fill(128, TL::T256::BF, TL::T256::BKB);
          const int rc = a.any_height >= kHeightsByRuns && splits == 1 ? launch_gemm_by_runs<T, typename TL::T128P, EPI>(a, 128, st) : launch_gemm_quad<T, EPI>(a, 128, splits, st);
          if (rc != 1) return rc;
        }
      }
      fill(128, TL::T128::BF, TL::T128::BKB);
      // The gate/up GEMM always takes the persistent form (its walk by expert fetches each expert's
      // weights once per chunk of token blocks); the down projection of the layer (few feature tiles,
      // long K) takes it for the split of the last round, a plain grouped GEMM keeps the plain kernel.
      if constexpr (EPI != EPI_SILU) {
        if (a.long_k) return launch_gemm_persistent<T, typename TL::T128P, EPI>(a, splits, st);
      } else {
        return launch_gemm_persistent<T, typename TL::T128P, EPI>(a, splits, st);
      }
      return launch_gemm<T, typename TL::T128, EPI>(a, splits, st);
    case 160:
      if constexpr (EPI != EPI_DOWN) {
        if (a.any_height) {  // tiles as tall as the experts' runs
          fill(160, TL::T256::BF, TL::T256::BKB);
          const int rc = a.any_height >= kHeightsByRuns && splits == 1 ? launch_gemm_by_runs<T, typename TL::T160P, EPI>(a, 160, st) : launch_gemm_quad<T, EPI>(a, 160, splits, st);
          if (rc != 1) return rc;
        }
      }
      fill(160, TL::T160P::BF, TL::T160P::BKB);
      return launch_gemm_persistent<T, typename TL::T160P, EPI>(a, splits, st);
    case 64:
      // The persistent form hides each tile's ring fill behind its predecessor's last K tiles: the 64-row gate/up
      // GEMM streams the weights at 6.3 instead of 5.9 TB/s (128 tokens: 318 -> 298 us, fp8 192 -> 170 us).  The
      // down projection's 64 x 256 tile gains nothing from it (147 us either way) and stays plain.
      if constexpr (sizeof(T) == 2) {
        // Rows of up to 4 KB: the 128-row tile's walk with half the rows.  Layer in parts of the time on T64U: H = 2048, 64 experts,
        // top-6 100 tokens 0.95, 120 0.95, 150 0.99, 230 0.97; H = 1024, F = 3584 60 0.97, 100 0.975, 200 0.96, 400 0.92; longer rows 1.01 to
        // 1.035 (H = 6144 0.98).
        if (EPI == EPI_SILU && a.K * static_cast<int>(sizeof(T)) <= kShortRow && a.K % (TL::T64W::BKB / static_cast<int>(sizeof(T))) == 0) {
          fill(64, TL::T64W::BF, TL::T64W::BKB);
          return launch_gemm_persistent<T, typename TL::T64W, EPI>(a, splits, st);
        }
        // Fewer tiles of 256 features than CUs, K slices included (by the worst-case block count, which is all the host knows): 128
        // features in 256-byte row pieces.  H = 1024, F = 3584, 8 experts, layer in parts of the time on T64: 60 tokens (156 tiles at
        // most) 0.94, 100 0.93, 200 (226) 0.92, but 400 (326) 1.05.
        if (EPI != EPI_SILU && a.long_k && a.K % (TL::T64N::BKB / static_cast<int>(sizeof(T))) == 0) {
          fill(64, TL::T64N::BF, TL::T64N::BKB);
          if (static_cast<int64_t>(a.num_t_blocks) * ceil_div(a.N, TL::T64::BF) * splits < 256 &&
              static_cast<int64_t>(a.k_per_split) * (splits - 1) < a.K)
            return launch_gemm_persistent<T, typename TL::T64N, EPI>(a, splits, st);
        }
      }
      if (EPI == EPI_SILU && a.K % (TL::T64U::BKB / static_cast<int>(sizeof(T))) == 0) {
        fill(64, TL::T64U::BF, TL::T64U::BKB);
        return launch_gemm_persistent<T, typename TL::T64U, EPI>(a, splits, st);
      }
      fill(64, TL::T64::BF, TL::T64::BKB);
      return launch_gemm<T, typename TL::T64, EPI>(a, splits, st);
    case 32:
      if constexpr (sizeof(T) == 2) {
        // Rows of up to 4 KB: half the features in 256-byte pieces on three slots, two workgroups per CU, whose start-up per tile
        // overlaps (T32L has one).  H = 2048, 64 experts, top-6, layer in parts of the time on T32L: 20 tokens 0.96, 32 0.97, 48 0.96, 80 0.977
        // (persistent 1.04, 1.005, 0.97, 0.95; on two slots 1.025, 0.98, 0.99, 1.00); longer rows 1.035 to 1.05.  Where T32L does not
        // fit either, T32 stays: gate/up in parts of its time H = 640, F = 2560, 8 experts 1.08, Zipf-skewed 1.13 to 1.25, H = 1152
        // 1.07 to 1.25, H = 1408, 16 experts 1.11 to 1.18.
        if (EPI == EPI_SILU && a.K * static_cast<int>(sizeof(T)) <= kShortRow && a.K % (TL::T32L::BKB / static_cast<int>(sizeof(T))) == 0) {
          fill(32, TL::T32N::BF, TL::T32N::BKB);
          return launch_gemm<T, typename TL::T32N, EPI>(a, splits, st);
        }
      }
      if (EPI == EPI_SILU && a.K % (TL::T32L::BKB / static_cast<int>(sizeof(T))) == 0) {
        fill(32, TL::T32L::BF, TL::T32L::BKB);
        return launch_gemm<T, typename TL::T32L, EPI>(a, splits, st);
      }
      fill(32, TL::T32::BF, TL::T32::BKB);
      if constexpr (sizeof(T) == 2 && EPI != EPI_SILU) {
        // The layer's down projection with K slices of 16 KB or more, whose tiles start K at spread places (SPREAD in moe_gemm_kernel.h): half
        // the bytes in flight per workgroup, twice the workgroups.  Layer in parts of the time on three slots, near-uniform / Zipf-skewed:
        // fp16, 16 experts, F = 8192 72 to 160 tokens 0.985 / 0.98, H = 6144, F = 16384, 8 experts 36 to 100 0.975 / 0.965.  Shorter
        // slices leave a CU too few bytes in flight or the workgroups uneven shares: H = 768 1.08, H = 512 1.07, 64 experts,
        // F = 1408 1.01 / 0.98 to 1.02, 16 experts, F = 1408, 200 tokens 0.99 / 1.02, F = 8192 in four slices 1.03 / 1.0.
        if (a.long_k && a.k_per_split * static_cast<int>(sizeof(T)) >= 16384 && (a.K & (a.K - 1)) == 0)
          return launch_gemm<T, typename TL::T32D, EPI>(a, splits, st);
        // Short slices (weight rows of up to 4 KB): a tile's rate is what it has in flight over the latency of memory, and a CU holds two
        // workgroups on four slots as on three.  Layer in parts of the time on three: H = 2048, F = 1408, 64 experts, top-6 24 to 48 tokens 0.995 to
        // 1.00, 64 0.987, 80 0.973, 100 0.988, 120 0.982; long slices lose (H = 4096, F = 14336, 8 experts 36 to 100 tokens 1.00 to 1.02),
        // and a launch that cannot fill two workgroups per CU, by the worst-case tile count, has nothing of it (H = 384 and 512, 8 and 16 experts).
        if (a.long_k && a.k_per_split * static_cast<int>(sizeof(T)) <= kShortRow && static_cast<int64_t>(a.num_t_blocks) * a.num_f_tiles * splits >= 512)
          return launch_gemm<T, typename TL::T32S, EPI>(a, splits, st);
      }
      return launch_gemm<T, typename TL::T32, EPI>(a, splits, st);
    case 16:
      // Plain or persistent.  A plain launch has two workgroups per CU that come and go: every tile pays its start-up
      // (block table -> sorted ids -> first K tiles) and its drain, and rounds of tiles do not overlap.  The persistent
      // form refills the ring across tiles, which pays where a tile's K loop is short or there are several rounds.
      if constexpr (EPI == EPI_SILU) {
        // Rows of up to 2 KB (8 K tiles of 256 bytes; fp8: up to 4 KB): 256-byte segments, persistent from 5 K tiles on and
        // up to 1022 experts, else plain (up to 1 KB).  Kernel in us on weights that no cache holds (several layers' in
        // turn), plain 512-byte segments / this form, 16 tokens, 8 experts unless said otherwise:
        //   bf16  H = 512, F = 3584 (plain) 17.9 / 16.3; 64 experts, top-6, F = 1408 35.9 / 31.8, 64 tokens 45.2 / 40.0
        //         H = 768 22.2 / 20.4, H = 1024 26.1 / 23.8, 64 experts, F = 1408, 32 tokens 65.4 / 59.6
        //   fp8   H = 512 (plain) 14.7 / 13.2, H = 1024 (plain) 18.6 / 16.9, H = 2048, F = 7168 48.6 / 42.2
        //         H = 3072, F = 8192 75.0 / 66.9, H = 3584 85.5 / 76.4
        //         H = 4096, F = 14336, 5 / 16 / 28 tokens 116 / 150 / 151 against 111 / 145 / 145 (another card: 118 / 153 / 153
        //         against 126 / 154 / 155); 64 experts, F = 1536, 32 tokens 124.7 / 125.0; 16 experts, F = 8192 169 / 167
        // bf16, H = 2048, F = 1408, 64 experts, top-6, 32 tokens, layer: 108 / 111 against 116 / 113 (on the previous pass's
        // weights it is the other way round, 102 against 98: part of them is still in the Infinity Cache).  Longer rows
        // stream faster in 512-byte pieces (bf16, H = 4096, layer: 428 against 445 us).
        if (a.K * static_cast<int>(sizeof(T)) <= (sizeof(T) == 1 ? 4096 : 2048)) {
          fill(16, TL::T16::BF, TL::T16::BKB);
          return launch_gemm_persistent<T, typename TL::T16, EPI>(a, splits, st);
        }
        if (a.K % (TL::T16L::BKB / static_cast<int>(sizeof(T))) == 0) {
          fill(16, TL::T16L::BF, TL::T16L::BKB);
          return launch_gemm<T, typename TL::T16L, EPI>(a, splits, st);
        }
      }
      fill(16, TL::T16::BF, TL::T16::BKB);
      // The layer's down projection from 8 KB of K per slice on (32 K tiles): persistent.  Kernel, plain / persistent: bf16,
      // H = 4096, F = 8192, 16 experts, 24 / 64 tokens (two rounds of tiles) 208 / 178 us, H = 2048, F = 4096, 64 experts, top-6,
      // 8 / 40 tokens 114 / 99 and 201 / 159; fp8, 16 experts 102 / 94; one round (8 experts, F = 14336) 151.5 either way,
      // fp8 72 / 71; 2.8 KB (F = 1408) loses 1 %.
      if (EPI != EPI_SILU && a.long_k && a.k_per_split * static_cast<int>(sizeof(T)) >= 8192)
        return launch_gemm_persistent<T, typename TL::T16, EPI>(a, splits, st);
      return launch_gemm<T, typename TL::T16, EPI>(a, splits, st);
    default: return fail(FR_E_SHAPE, "routing block %d not in {16, 32, 64, 128, 160, 256}", block);
  }
}

// Per-device set-up (dynamic LDS limits, occupancy queries) of every kernel dispatch_block<T, EPI> can launch,
// so that no later call has anything left to set up - e.g. a first call under graph capture.
template <typename T, int EPI>
int prepare_tiles() {
  typedef Tiles<T> TL;
  GemmArgs a = {};
  a.setup_only = 1;
  int rc = launch_gemm_persistent<T, typename TL::T256, EPI>(a, 1, nullptr);
  if constexpr (sizeof(T) == 2) {
    if (rc == FR_OK) rc = launch_gemm_persistent<T, typename TL::T256S, EPI>(a, 1, nullptr);
  }
  if constexpr (EPI != EPI_DOWN) {
    if (rc == FR_OK) rc = launch_gemm_quad<T, EPI>(a, 256, 1, nullptr);
    if (rc == FR_OK) rc = launch_gemm_persistent<T, typename TL::T128P, EPI, true>(a, 1, nullptr);
    if (rc == FR_OK) rc = launch_gemm_persistent<T, typename TL::T160P, EPI, true>(a, 1, nullptr);
  }
  if (rc == FR_OK) rc = launch_gemm_persistent<T, typename TL::T128P, EPI>(a, 1, nullptr);
  if (rc == FR_OK) rc = launch_gemm_persistent<T, typename TL::T160P, EPI>(a, 1, nullptr);
  if (rc == FR_OK) rc = launch_gemm<T, typename TL::T128, EPI>(a, 1, nullptr);
  if (rc == FR_OK) rc = launch_gemm<T, typename TL::T64, EPI>(a, 1, nullptr);
  if (rc == FR_OK) rc = launch_gemm<T, typename TL::T32, EPI>(a, 1, nullptr);
  if (rc == FR_OK) rc = launch_gemm_persistent<T, typename TL::T16, EPI>(a, 1, nullptr);  // and its plain form
  if constexpr (sizeof(T) == 2) {
    if constexpr (EPI == EPI_SILU) {
      if (rc == FR_OK) rc = launch_gemm<T, typename TL::T32N, EPI>(a, 1, nullptr);
      if (rc == FR_OK) rc = launch_gemm_persistent<T, typename TL::T64W, EPI>(a, 1, nullptr);
    } else {
      if (rc == FR_OK) rc = launch_gemm_persistent<T, typename TL::T64N, EPI>(a, 1, nullptr);
      if (rc == FR_OK) rc = launch_gemm<T, typename TL::T32D, EPI>(a, 1, nullptr);
      if (rc == FR_OK) rc = launch_gemm<T, typename TL::T32S, EPI>(a, 1, nullptr);
    }
  }
  if constexpr (EPI == EPI_SILU) {
    if (rc == FR_OK) rc = launch_gemm_persistent<T, typename TL::T64U, EPI>(a, 1, nullptr);
    if (rc == FR_OK) rc = launch_gemm<T, typename TL::T32L, EPI>(a, 1, nullptr);
    if (rc == FR_OK) rc = launch_gemm<T, typename TL::T16L, EPI>(a, 1, nullptr);
  }
  return rc;
}

}  // namespace fr
