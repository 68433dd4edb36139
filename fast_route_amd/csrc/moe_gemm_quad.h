// Persistent grouped GEMM with ONE wavefront per SIMD: up to 288 sorted slots x 256 features per workgroup, 16x16x32
// MFMAs (2-byte operands) or 32x32x64 MFMAs (fp8).
//
// Why.  In the eight-wavefront tiles a wavefront owns 128 x 64 outputs and reads twelve operand fragments from
// LDS for thirty-two MFMAs; with 128 x 128 per wavefront it reads sixteen for sixty-four, a third less LDS traffic
// for the same arithmetic and half as many wavefronts issuing instructions, and the part's clock under MFMA load
// follows the energy a flop costs.  The accumulators live in the accumulation half of the register file (one
// wavefront per SIMD has 512 registers per lane), those of a 288-row tile's last token tiles in the ordinary half.
//
// Tile heights.  A tile is 1 to 9 units of 32 token rows: an expert's run of slots is cut into as few tiles as 288 rows
// allow (quad_tiles, quad_walk, quad_tile_at), whatever the routing block.  No tile crosses into the padding behind a
// run: an expert with 1030 pairs is multiplied as 1056 rows in four tiles where 256-row blocks made it 1280 rows in
// five.  Layer in us, 8 experts, H = 4096, F = 14336, top-2, whole and half blocks of 256 / runs: 2048 tokens 1374 / 1190,
// 3000 1814 / 1694, 4096 2325 / 2155, 5800 3154 / 3107, 16384 8567 / 8440; fp8 2048 769 / 680, 3100 1077 / 1007; H = 2048,
// F = 1408, 64 experts, top-6, Zipf-skewed 7000 816 / 790, 8192 922 / 900.  Where the blocks had no padding to lose (every
// expert a multiple of 256) gate/up is even, the down projection 1 % slower with long K loops (8 experts, 256 / 512 / 1024 /
// 2048 rows each 262 / 264, 369 / 374, 689 / 698, 1336 / 1348 us; staged calls, a slice buffer short, 262 / 286 on the first) and
// 2 to 5 % faster with short ones (64 experts, 256 / 512 / 1024 rows 160 / 153, 234 / 222, 424 / 416).  A K loop exists per height (kernel code per height,
// chosen per work unit); the height of the next unit is known a tile ahead, and the hand-over always loads 288 rows' worth of
// addresses (rows beyond the tile are outside the buffer resource and fetch nothing), so any height may follow any other.
//
// Stream.  With a single wavefront per SIMD nobody fills the issue slots a burst of loads or a wait leaves, so the
// wavefront's own instruction stream is even: a K tile of 128 bytes per row is two K-steps; the one barrier per K tile
// sits between them, where every fragment of the tile has been read: the tile's ring slot is free from there on and takes
// the loads of the K tile after next, spread over the second K-step, which leaves them the first K-step of the next K tile
// to land.  The operand the MFMAs walk slowest (2-byte: the eight weight fragments; fp8: the token fragments) has one
// register set, each fragment read again behind its last MFMA of the K-step, except the last ones, whose reads would end
// up right before the barrier; the other operand and those last ones have two sets.
//
// What such a stream cannot hide is a load that misses L2: the ring has two slots, so at most one K tile per
// workgroup is in flight, and a wavefront that finds the memory pipeline backed up stalls at the issue of its
// next load with its MFMAs behind it.  Hence the L2 touch: the workgroups an XCD runs at one time share their
// operand tiles (the token tiles of one chunk share a weight tile, the feature tiles of one token tile its
// rows), and each of them asks for its share of the rows of a K tile several K tiles ahead - one dword per
// 128-byte row piece, into a sink in LDS - so that the tile loads proper find their lines in L2.
//
// Tiles alone on their weight tile.  Where an expert's run is one tile, nobody shares its weight tiles: the touch only passes them
// through L1 twice.  Up to 7 units (fp8: 6) such a tile has a K loop without touches, its weight loads non-temporal, so that the
// stream leaves the token rows in L2; and every run of up to 8 units starts its K loops at spread places (spread_k_start256, why:
// SPREAD_K in moe_gemm_persistent.h), as the eight-wavefront 256-row kernels do.  Layer on these tiles, in
// parts of the time with touches from column 0, without touches / and spread: H = 4096, F = 14336, 8 experts 700 tokens (6 units)
// 0.95 / 0.90, 850 1.00 / 0.95; fp16, 16 experts, F = 8192, 700 (3) 0.90 / 0.855, 1100 0.92 / 0.89, 1500 0.96 / 0.91; H = 6144 700
// 0.93 / 0.89; H = 2048, 64 experts, Zipf-skewed 3000 0.975 / 0.97, 6500 0.99 / 0.98.  With 8 and 9 units it is even or slower (the ring's
// two slots need the L2 hits, and the rows of a start of its own the L2): 1031 tokens 820 without touches, 782 with.  Non-temporal
// touches are evicted before their loads come (20 to 25 % slower); non-temporal loads behind ordinary touches change nothing there
// and cost 14 % where weight tiles are shared.
//
// Same tail split and LDS swizzle as moe_gemm_persistent_kernel; whole tiles are bit-identical to the eight-wavefront 256-row kernels' on
// the same MFMA shape (same K order per accumulator, same roundings in the epilogue).  The 128- and 160-row tiles that this
// kernel stands in for start their K loops elsewhere, and a tile cut along K depends on the tiles' heights.
#pragma once
#include "moe_gemm_persistent.h"

namespace fr {

constexpr int kUnitRows = 32;   // a tile's height in units of
constexpr int kMaxUnits = 9;
// 2 x 2 wavefronts of (half the rows) x 128 features; 16x16x32 MFMAs, fp8 32x32x64.  fp8 tiles of an odd number of units: 1 x 4
// wavefronts of (all rows) x 64 features, a fifth more LDS reads per MFMA (6000 tokens with 1 x 4 throughout: down
// projection 567 against 548 us) but no unit of padding.
template <typename T, int UN>
using QuadCfg = typename std::conditional<sizeof(T) == 2, Cfg<kUnitRows * UN, 256, 128, 2, 2, 16, 1, 2, 0, 1>,
                                          typename std::conditional<UN % 2 == 0, Cfg<kUnitRows * UN, 256, 128, 2, 2, UN % 2 == 0 ? 32 : 16, 1, 2, 0, 1>,
                                                                    Cfg<kUnitRows * UN, 256, 128, 1, 4, 32, 1, 2, 0, 1>>::type>::type;
constexpr int kQuadMinTiles = 8;       // K tiles per work unit, at least (one peeled at its start, five at its end)
constexpr int kQuadXShare = 4;         // ways the touch of a tile's token rows is shared, at most
constexpr int kQuadSink = 1024;        // bytes of LDS the touches land in (256 per wavefront)
// What a tile costs besides its height, in tenths of a unit (weight rows, barriers, epilogue): 64 experts x 8 feature tiles of the
// 22-K-tile down projection, two tiles each (4 rounds), 10 / 12 / 16 / 18 units per expert 183 / 201 / 240 / 259 us with the
// combine: 19.3 us per unit and about 47 + the combine's 40 at none.
constexpr int kTileCost = 26;
// What cutting the last round along K costs besides its slices, in 32nds of a tile, and how much longer than alone, in fifths,
// the slices take behind whole rounds, whose workgroups are no longer in step.  Down projection, 8 experts x 16 feature tiles,
// one round of whole tiles and 128 tiles in two slices / two whole rounds of lower tiles: 20 units per expert 574 / 498 us, 22
// 608 / 547, 24 622 / 562; a round and 32 tiles in eight slices / two rounds, 2048 tokens 445 / 472; nothing but a cut round / a
// whole one: 8 units 264 / 283, 4 experts, 16 units 203 / 231.
constexpr int kCutCost = 4, kCutStretch = 8;
constexpr int kQuadRing = 2 * (kUnitRows * kMaxUnits + 256) * 128;
// Slice buffers of the cut last round, per XCD of 32 workgroups: 32 of 256 x 256 fp32 or, with 288-row tiles, as many of 288 x 256:
// the layers' scratch has room for 32 of these too, a staged caller's (fr_moe_plan.tail_bytes) for 28.  Half a round of 288-row tiles
// takes 32 for two slices each: H = 4096, F = 14336, 8 experts, one tile per expert and feature tile (gate/up: 3 1/2 rounds), layer
// with 28 / 32 buffers 1031 tokens 780 / 769 us, 950 771 / 767; H = 6144, 1031 tokens 1320 / 1311.
// What the fix-up launch needs to know about a cut tile is left next to them (TailCut), in the scratch itself where the
// caller has no other place for it: then there are 31 buffers of 256 rows.  (Working it out again in the fix-up launch instead
// costs staged calls 8 to 12 us: down projection, 8 experts, 1300 tokens 302 / 314, 2048 381 / 393.)
constexpr int kQuadTallBuffers = 28;
__device__ __forceinline__ int quad_buffer_rows(int tallest) { return tallest > 8 ? kUnitRows * kMaxUnits : 256; }
__device__ __forceinline__ int quad_buffers(const GemmArgs& a, int tallest) { return tallest > 8 ? a.tall_buffers : a.tail_buffers; }
static_assert(sizeof(TailCut) * kTailUnits <= kTailDescBytes, "a tile per workgroup");
static_assert(static_cast<int64_t>(kTailUnits) * kUnitRows * kMaxUnits * 256 * 4 == kTallTailBytes, "32 buffers per XCD in the layers' scratch");
static_assert(8 * kQuadTallBuffers * kUnitRows * kMaxUnits * 256 * 4 + kTailDescBytes <= kTailUnits * 256 * 256 * 4 &&
                  8 * 31 * 256 * 256 * 4 + kTailDescBytes <= kTailUnits * 256 * 256 * 4, "fits the scratch");

// Tiles an expert's run of `units` units is cut into when a tile may have `limit` of them: as few as fit, of heights as equal
// as units allow.  With the largest limit a multiple of 256 rows keeps 256-row tiles.
__device__ __forceinline__ int quad_tiles(int units, int limit) {
  return limit == kMaxUnits && units % 8 == 0 ? units / 8 : (units + limit - 1) / limit;
}

// Walk table: off[e] = first routing block of expert e, units[e] = units of its run up to the last one that holds a
// pair, tiles[e] = tiles of the experts before e.  off[kMaxExperts + 1]: the blocks are in no order (legal for the op-level
// GEMM): every block is a tile of its own, tiles and units are not written.
struct QuadWalk {
  int off[kWalkTable], units[kWalkTable], tiles[kWalkTable];
  int tallest;  // units of the tallest tile
  int count[6], high[6];  // tiles and tallest tile under each limit of a tile's height: see quad_walk
};
// all 256 threads; `block` rows per routing block (a multiple of 32, at most 256), nt > 0 blocks, nper workgroups per XCD.
// Nothing of a launch runs beside it, so it is written for few dependent loads and little code (which comes from memory, too):
// from the start of the launch to the first K tile's arrival 64 experts take 11.5 - 12.1 us (gate/up, down projection), 8 experts 9.4 -
// 10.2, of which 3 to 4 are the first tiles' own loads; 15.5 - 16.7 and 11.7 - 12.6 when a wavefront went through its experts' last blocks
// and all limits, the cut tile was worked out apart and the first weights waited for the sorted ids.  Layer H = 2048, 64 experts,
// top-6, 8192 tokens 883 -> 875 us, 6200 703 -> 696; H = 4096, 1031 tokens 773 -> 770; fp8 650 387 -> 384.
// false: the other launch of launch_gemm_by_runs works on these runs
__device__ __forceinline__ bool quad_walk(const GemmArgs& a, QuadWalk& w, int block, int nt, int tid, int nper, int k_tiles) {
  expert_block_offsets(a, nt, w.off, tid, 256);
  if (a.by_runs && !runs_fill_tall_tiles(a, w.off, nt, tid & 63)) return false;
  if (w.off[kMaxExperts + 1]) {
    if (tid == 0) w.tallest = block / kUnitRows;
    __syncthreads();
    return true;
  }
  const int E = a.num_experts, lane = tid & 63, wave = tid >> 6, groups = block / kUnitRows;
  for (int e = tid; e < E; e += 256) w.units[e] = max(w.off[e + 1] - w.off[e] - 1, 0) * groups;
  __syncthreads();
  // the last block of every run: its last 32-slot group with a pair, a group per thread (two at a time), their ids in flight together
  for (int i0 = tid; i0 < E * 8; i0 += 2 * 256) {
    typedef int i32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int V = kUnitRows / 4;
    i32x4_a4 id[2][V];
    int e[2], run[2];  // expert, units of its run up to this group (0: no such group)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int i = min(i0 + p * 256, E * 8 - 1), g = i & 7;
      e[p] = i >> 3;
      const int len = w.off[e[p] + 1] - w.off[e[p]];
      run[p] = len > 0 && g < groups ? (len - 1) * groups + g + 1 : 0;
      const i32x4_a4* ids = reinterpret_cast<const i32x4_a4*>(a.sorted + (run[p] ? (w.off[e[p]] + len - 1) * block + g * kUnitRows : 0));
#pragma unroll
      for (int x = 0; x < V; ++x) id[p][x] = ids[x];
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      int least = id[p][0][0];
#pragma unroll
      for (int x = 0; x < V; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) least = min(least, id[p][x][r]);
      if (least < a.num_valid) atomicMax(&w.units[e[p]], run[p]);
    }
  }
  __syncthreads();
  // The limit of a tile's height.  Tall tiles cost least per row, but a launch of few rounds is over when its busiest
  // workgroup is: a round takes as long as kTileCost + height, and the tiles behind the whole rounds as long as a round
  // unless the schedule cuts them along K.  (Down projection, 8 experts x 16 feature tiles, limit 9 / 8 / 7 / 6 / 5 / 4 in us:
  // 20 units each 574 / 574 / 576 / 498 / 483 / 693 (6 taken), 26 units 715 / 622 / 622 / 790 / 767 / 923 (8 taken), 33 units
  // 752 / 907 / 910 / 867 / 1002 / 1068 (9 taken).  Over 186 launches, 8 to 50 units on 1 to 16 experts, the limit taken costs
  // 1.0 % more than the best on average.)
  constexpr int NL = 6;  // limits 9 to 4: tiles and tallest tile of limits 9 - wave and 5 - wave
  {
    int n[2] = {}, tall[2] = {};
    for (int e0 = 0; e0 < E; e0 += kWave) {
      const int u = e0 + lane < E ? w.units[e0 + lane] : 0;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int c = quad_tiles(u, kMaxUnits - min(wave + 4 * p, NL - 1));
        n[p] += c;
        tall[p] = max(tall[p], c ? (u + c - 1) / c : 0);
      }
    }
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        n[p] += __shfl_xor(n[p], d);
        tall[p] = max(tall[p], __shfl_xor(tall[p], d));
      }
#pragma unroll
    for (int p = 0; p < 2; ++p)
      if (lane == 0 && wave + 4 * p < NL) {
        w.count[wave + 4 * p] = n[p];
        w.high[wave + 4 * p] = tall[p];
      }
  }
  __syncthreads();
  if (wave == 0) {
    unsigned cost;  // lane l: of limit 9 - l
    {
      const int n = w.count[min(lane, NL - 1)], tall = w.high[min(lane, NL - 1)];
      // XCD 0 has the largest share
      const XcdSchedule xs = xcd_schedule(n * a.num_f_tiles, nper, 0, k_tiles, a.tail_ws != nullptr, schedule_by_rounds(n, E),
                                          quad_buffers(a, tall));
      const unsigned tile = kTileCost + 10 * tall, rounds = xs.rounds, slices = xs.slices;
      const unsigned cut = 32 * tile * (rounds ? kCutStretch : 5) / (5 * slices) + kCutCost * tile;
      cost = 32 * rounds * tile + (xs.rest == 0 ? 0 : slices < 2 ? 32 * tile : cut);
    }
    int best = 0;
    unsigned least = __builtin_amdgcn_readlane(cost, 0);
    for (int l = 1; l < NL; ++l) {  // a lower limit has to be 3 % cheaper
      const unsigned c = __builtin_amdgcn_readlane(cost, l);
      if (c < least - least / 32) {
        least = c;
        best = l;
      }
    }
    int base = 0;
    for (int e0 = 0; e0 <= E; e0 += kWave) {
      const int e = e0 + lane, c = e < E ? quad_tiles(w.units[e], kMaxUnits - best) : 0;
      int s = c;
#pragma unroll
      for (int d = 1; d < kWave; d <<= 1) {
        const int up = __shfl_up(s, d);
        if (lane >= d) s += up;
      }
      if (e <= E) w.tiles[e] = base + s - c;
      base += __shfl(s, kWave - 1);
    }
    if (lane == 0) w.tallest = w.high[best];
  }
  __syncthreads();
  return true;
}

// A work unit: an output tile, or a K slice of one.
struct QuadUnit {
  int row0, units;    // first slot, height
  int f, expert;      // feature tile, expert
  int kb, kn, tu;     // K tile it starts at, K tiles (round the end of K), slice buffer (-1: a whole tile)
  int share;          // tiles of its chunk (which share its weight tile) and its index among them: count << 16 | index; 0: blocks in no order
};
constexpr int kUnitTable = 64;  // units a wavefront works out at a time, one per lane

// Tile number lin of the walk: experts in order, an expert's run in chunks of at most group_t tiles, a chunk tile-fastest
// over all feature tiles (see tile_coords).  even_heights: all tiles
// of an expert but the last have the mean height rounded up to even, the last what is left.
__device__ __forceinline__ void quad_tile_at(const GemmArgs& a, const QuadWalk& w, int block, bool even_heights, int lin, int k_all, QuadUnit& u) {
  const int F = a.num_f_tiles, t = lin / F;
  if (w.off[kMaxExperts + 1]) {
    u.row0 = t * block;
    u.units = block / kUnitRows;
    u.f = lin - t * F;
    u.expert = a.expert_ids[t];
    u.share = 0;  // unknown: touched like a tile alone, but its weights are not taken for a stream
    return;
  }
  int lo = 0, hi = a.num_experts - 1;  // the last expert whose tiles start at or before t: it has some
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (w.tiles[mid] <= t) lo = mid;
    else hi = mid - 1;
  }
  const int first = w.tiles[lo], len = w.tiles[lo + 1] - first, un = w.units[lo];
  const int chunks = (len + a.group_t - 1) / a.group_t, base = len / chunks, rem = len - base * chunks;
  int q = lin - first * F, gsz = base + 1, start = 0;
  const int big = rem * gsz * F;  // the first rem chunks hold one tile more
  if (q >= big) {
    q -= big;
    start = rem * gsz;
    gsz = base;
  }
  const int c = q / (gsz * F);
  q -= c * gsz * F;
  start += c * gsz;
  u.f = q / gsz;
  const int index = q - u.f * gsz, b = start + index;
  const int even = (un + 2 * len - 1) / (2 * len) * 2;  // the mean height, rounded up to even
  if (even_heights && un <= 8 * len + 1 && min(even, 8) * (len - 1) < un) {
    const int h = min(even, 8);
    u.row0 = w.off[lo] * block + b * h * kUnitRows;
    u.units = b < len - 1 ? h : un - h * (len - 1);
  } else {
    const int ub = un / len, ur = un - ub * len;  // the first ur tiles are one unit taller
    u.row0 = w.off[lo] * block + (b * ub + min(b, ur)) * kUnitRows;
    u.units = ub + (b < ur ? 1 : 0);
  }
  u.expert = lo;
  u.share = gsz << 16 | index;
  if (un <= 8 && a.spread_k) u.kb = spread_k_start256(lo, u.f, F, u.kb, k_all);
}

// One MFMA, written out so that an accumulator stays in the registers it has: those of the first kQuadAgpr token tiles in
// the accumulation half of the register file (all 256 of them in a tile of 256 rows or more), the rest in the ordinary
// half.  Left to the compiler's three-operand form, with no register of that half to spare, accumulators wandered through
// ordinary registers around the K loop and address registers were spilled inside it (288 rows, 4096 tokens: down projection
// 906 against 740 us).  What the compiler sees to for MFMAs of its own, and not for these: a result may be read by another
// instruction 18 wait states after the last MFMA on it at the earliest (run_unit's s_nops wait 20; MFMAs on one accumulator are
// as many MFMAs apart as a K-step has), and no vector instruction may write an operand right before the MFMA (two wait states).
// Operands are LDS reads, which are waited for, and accumulators start from zero in an MFMA, so there is nothing to write one;
// a change here is checked in the assembly: the 6720 MFMAs of a 2-byte kernel and the 1148 of an fp8 one have no vector write
// of an operand among the four instructions before.
constexpr int kQuadAgpr = 8;
#if defined(__HIP_DEVICE_COMPILE__)
#define FQ_MFMA(name_, reg_)                                                                                     \
  if constexpr (FIRST) asm volatile(name_ " %0, %1, %2, 0" : "=&" reg_(acc) : "v"(wf), "v"(xf));                 \
  else asm volatile(name_ " %0, %1, %2, %0" : "+" reg_(acc) : "v"(wf), "v"(xf));
template <typename T, bool AGPR, bool FIRST, typename AccT>
__device__ __forceinline__ void quad_mfma(AccT& acc, const u32x4* w, const u32x4* x) {
  if constexpr (sizeof(T) == 1) {
    const i32x8 wf = Elem<T>::join(w), xf = Elem<T>::join(x);
    if constexpr (AGPR) { FQ_MFMA("v_mfma_f32_32x32x64_f8f6f4", "a") } else { FQ_MFMA("v_mfma_f32_32x32x64_f8f6f4", "v") }
  } else {
    const u32x4 wf = w[0], xf = x[0];
    if constexpr (std::is_same<T, bf16_t>::value) {
      if constexpr (AGPR) { FQ_MFMA("v_mfma_f32_16x16x32_bf16", "a") } else { FQ_MFMA("v_mfma_f32_16x16x32_bf16", "v") }
    } else {
      if constexpr (AGPR) { FQ_MFMA("v_mfma_f32_16x16x32_f16", "a") } else { FQ_MFMA("v_mfma_f32_16x16x32_f16", "v") }
    }
  }
}
#undef FQ_MFMA
#endif

// Epilogue of a tile [row0, row_end) x columns from f0 on.  Every column exists (a width below a tile's is not taken, the last
// tile starts early), rows from row_end on belong to another tile, in whole token tiles: one scalar test each.  With one
// wavefront per SIMD nothing runs beside it, so a token tile has one row address and its columns are immediate offsets of
// the stores, which are 16 bytes wide (join_features), and fp8's weight scales come in 16-byte loads.  A token tile is fetched, computed and stored before the next
// is looked at: what the compiler may not do across a fence is hold all accumulators in ordinary registers.  Against the
// epilogue that the other kernels share (column tests and an address per group, ids loaded one by one): down projection,
// H = 2048, F = 1408, 64 experts, 8192 tokens 332 -> 309 us, 256 rows each 170 -> 153; H = 4096, F = 14336, 8 experts, 4096 tokens
// 727 -> 720; gate/up in fp8, 2048 tokens 478 -> 456.
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));  // a caller's scale array is aligned to its elements
// a loaded value is waited for here and not where it is used
template <typename V>
__device__ __forceinline__ void arrived(V& v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(v));
#endif
}
template <typename T, typename C, int EPI, typename AccT>
__device__ __forceinline__ void quad_epilogue(const GemmArgs& a, AccT (&acc)[C::JF][C::IT], int row0, int row_end, int f0, int expert,
                                              int wt, int wf, int frow, int kgrp) {
  typedef Elem<T> E;
  typedef typename E::out_t out_t;
  typedef typename E::out4 out4;
  constexpr int GROUPS = (C::TILE == 32) ? 4 : 1;  // groups of 4 consecutive features of a lane and accumulator tile
  constexpr int HJ = C::JF / 2;                    // EPI_SILU: gate tiles, then as many up tiles
  constexpr int TF = (EPI == EPI_SILU) ? C::TF / 2 : C::TF;
  const int slot0 = row0 + wt * C::TT, col0 = f0 + wf * TF + kgrp * 4;
  // What the rows need from memory, in two rounds: all loads of a round go out before the first is waited for, and the last
  // wait is behind them, not between the stores (a wait there is one for the stores before it, too).
  int sids[C::IT];
  float scale[C::IT];  // routed weight of the lane's pair in each token tile, times the token row's scale (fp8)
  f32x4 wscale[E::SCALED ? C::JF * GROUPS : 1];
  if constexpr (E::SCALED) {
    const float* wsc = a.w_scale + static_cast<int64_t>(expert) * a.w_rows + col0;
#pragma unroll
    for (int j = 0; j < C::JF; ++j)
#pragma unroll
      for (int g = 0; g < GROUPS; ++g)
        wscale[j * GROUPS + g] = *reinterpret_cast<const f32x4_a4*>(
            EPI == EPI_SILU ? wsc + (j / HJ) * static_cast<int64_t>(a.N) + (j % HJ) * C::TILE + g * 8 : wsc + j * C::TILE + g * 8);
  }
  if constexpr (EPI != EPI_SILU || E::SCALED) {
#pragma unroll
    for (int i = 0; i < C::IT; ++i) sids[i] = a.sorted[min(slot0 + i * C::TILE + frow, row_end - 1)];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < C::IT; ++i) {
      arrived(sids[i]);
      if (slot0 + i * C::TILE + frow >= row_end) sids[i] = a.num_valid;
      scale[i] = 1.f;
    }
    float xs[C::IT];
    if constexpr (EPI != EPI_SILU) {
      if (a.mul_weight) {
#pragma unroll
        for (int i = 0; i < C::IT; ++i) scale[i] = a.topk_w[min(sids[i], a.num_valid - 1)];
      }
    }
    if constexpr (E::SCALED) {  // a padding row's scale is not used
#pragma unroll
      for (int i = 0; i < C::IT; ++i)
        xs[i] = a.x_scale[a.top_k > 0 ? min(sids[i], a.num_valid - 1) / a.top_k : min(slot0 + i * C::TILE + frow, row_end - 1)];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < C::IT; ++i) {
      arrived(scale[i]);
      if constexpr (E::SCALED) {
        arrived(xs[i]);
        scale[i] *= xs[i];
      }
    }
    if constexpr (E::SCALED) {
#pragma unroll
      for (int x = 0; x < C::JF * GROUPS; ++x) arrived(wscale[x]);
    }
  }
  // pairs of accumulator groups, joined into 16-byte stores: (MFMA tile j, j + 1) or, with 32 x 32 tiles, groups (g, g + 1)
  constexpr int JS = GROUPS == 1 ? 2 : 1, PAIRS = GROUPS == 1 ? 1 : GROUPS / 2;
  typedef out_t out8 __attribute__((ext_vector_type(8), aligned(8)));  // rows of a width that is a multiple of 4
  const int colw = f0 + wf * TF + kgrp * 8;
#pragma unroll
  for (int i = 0; i < C::IT; ++i) {
    if (slot0 + i * C::TILE >= row_end) break;
    auto fetch = [&](int j) { return i < kQuadAgpr ? acc_fetch(acc[j][i]) : acc[j][i]; };
    if constexpr (EPI == EPI_SILU) {
      out_t* row = static_cast<out_t*>(a.out) + static_cast<int64_t>(slot0 + i * C::TILE + frow) * a.ldo + colw;
      auto value = [&](const AccT& ga, const AccT& ua, int j, int g) {
        out4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float gv = ga[g * 4 + r], uv = ua[g * 4 + r];
          if constexpr (E::SCALED) {
            gv *= scale[i] * wscale[j * GROUPS + g][r];
            uv *= scale[i] * wscale[(j + HJ) * GROUPS + g][r];
          }
          o[r] = round_once<out_t>(silu(gv) * uv);
        }
        return o;
      };
#pragma unroll
      for (int j = 0; j < HJ; j += JS) {
        const AccT ga = fetch(j), ua = fetch(j + HJ);
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
          out4 lo = value(ga, ua, j, GROUPS == 1 ? 0 : 2 * p), hi;
          if constexpr (GROUPS == 1) hi = value(fetch(j + 1), fetch(j + 1 + HJ), j + 1, 0);
          else hi = value(ga, ua, j, 2 * p + 1);
          join_features<C::TILE>(lo, hi);
          *reinterpret_cast<out8*>(row + j * C::TILE + p * 16) = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      const bool valid = sids[i] < a.num_valid;
      auto value = [&](const AccT& c, int j, int g) {
        out4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = c[g * 4 + r] * scale[i];
          if constexpr (E::SCALED) v *= wscale[j * GROUPS + g][r];
          o[r] = r < 2 ? round_twice<out_t>(v) : round_once<out_t>(v);
        }
        return o;
      };
      if (a.add_div) {  // top-k combine in the epilogue
        out_t* row = static_cast<out_t*>(a.out) + static_cast<int64_t>(sids[i] / a.add_div) * a.ldo + col0;
#pragma unroll
        for (int j = 0; j < C::JF; ++j) {
          const AccT c = fetch(j);
#pragma unroll
          for (int g = 0; g < GROUPS; ++g)
            if (valid) atomic_add4(row + j * C::TILE + g * 8, value(c, j, g));
        }
      } else {
        out_t* row = static_cast<out_t*>(a.out) + static_cast<int64_t>(sids[i]) * a.ldo + colw;
#pragma unroll
        for (int j = 0; j < C::JF; j += JS) {
          const AccT c = fetch(j);
#pragma unroll
          for (int p = 0; p < PAIRS; ++p) {
            out4 lo = value(c, j, GROUPS == 1 ? 0 : 2 * p), hi;
            if constexpr (GROUPS == 1) hi = value(fetch(j + 1), j + 1, 0);
            else hi = value(c, j, 2 * p + 1);
            join_features<C::TILE>(lo, hi);
            if (valid) *reinterpret_cast<out8*>(row + j * C::TILE + p * 16) = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          }
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// What the workgroups of an XCD have to do: all 256 threads, the walk table behind it.
struct QuadPlan {
  XcdSchedule xs;
  int tallest;
  bool even_heights;
  bool works;  // see quad_walk
};
template <typename T>
__device__ __forceinline__ QuadPlan quad_plan(const GemmArgs& a, QuadWalk& walk, int block, int xcd, int nper, int tid) {
  const int nt = min(a.npost[0] / block, a.num_t_blocks), k_tiles = a.K / (QuadCfg<T, kMaxUnits>::BKB / static_cast<int>(sizeof(T)));
  QuadPlan p;
  // fp8's even heights have the geometry with fewer LDS reads, and short K loops are better off with whole tiles and one
  // short one than with equal ones: layer in us, equal / even, fp8 2500 tokens 926 / 894, 4878 1570 / 1515; H = 2048, F = 1408
  // (32 and 22 K tiles), 64 experts, 8192 tokens 952 / 940, 7000 806 / 800; H = 4096, F = 14336 (64 and 224) 2300 1460 / 1495,
  // 3000 1713 / 1733, 5800 3116 / 3142.
  p.even_heights = sizeof(T) == 1 || k_tiles <= 32;
  int tiles = 0;
  p.tallest = 0;
  p.works = true;
  if (nt > 0) {
    p.works = quad_walk(a, walk, block, nt, tid, nper, k_tiles);
    if (!p.works) return p;
    tiles = __builtin_amdgcn_readfirstlane(walk.off[kMaxExperts + 1] ? nt : walk.tiles[a.num_experts]);
    p.tallest = __builtin_amdgcn_readfirstlane(walk.tallest);
  }
  p.xs = xcd_schedule(tiles * a.num_f_tiles, nper, xcd, k_tiles, a.tail_ws != nullptr, schedule_by_rounds(tiles, a.num_experts),
                      quad_buffers(a, p.tallest));
  return p;
}
template <typename T, int EPI>
__global__ __launch_bounds__(256, 1) void moe_gemm_quad_kernel(const GemmArgs a, int block) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef QuadCfg<T, kMaxUnits> CM;
  typedef Elem<T> E;
  typedef __attribute__((address_space(3))) void* lptr_t;
  typedef typename std::conditional<CM::TILE == 32, f32x16, f32x4>::type acc_t;
  constexpr int ES = static_cast<int>(sizeof(T));
  constexpr int BF = CM::BF, CPR = CM::CPR, BKB = CM::BKB, BK = BKB / ES, FC = E::FC;
  constexpr int TILE = CM::TILE, KG = CM::KGROUPS;
  constexpr int COLS = EPI == EPI_SILU ? BF / 2 : BF;
  constexpr int kAloneUnits = sizeof(T) == 1 ? 6 : 7;  // tallest tile with a loop of its own for being alone on its weight tile
  constexpr int NW = 4, XI = kMaxUnits, WI = 8;        // tile loads per wavefront and K tile, at most: a load per unit of rows
  constexpr int XBYTES = kUnitRows * kMaxUnits * BKB, SLOT = XBYTES + BF * BKB;  // a ring slot: X rows, then W rows
  static_assert(2 * SLOT == kQuadRing && CM::WIW == WI && CM::XIW == XI && CPR == 8 && CPR / (KG * FC) == 2, "two K-steps per K tile");

  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  __shared__ QuadWalk walk;
  __shared__ QuadUnit unit_table[2][kUnitTable];

  // ---- schedule (as in moe_gemm_persistent_kernel, over the tiles of quad_walk) -----------------
  const int tid = threadIdx.x, lane = tid & 63;
  const int xcd = blockIdx.x & 7, nper = gridDim.x >> 3, loc = blockIdx.x >> 3;
  const int k_all = a.K / BK;
  const QuadPlan plan = quad_plan<T>(a, walk, block, xcd, nper, tid);
  if (!plan.works) return;
  const XcdSchedule& xs = plan.xs;
  // what the fix-up launch asks for: tile `loc` of the XCD's last round, if that is cut (then it is this workgroup's last unit)
  TailCut* const cut_at = a.tail_desc != nullptr ? reinterpret_cast<TailCut*>(a.tail_desc) + (xcd * nper + loc) : nullptr;
  const bool cut = xs.slices > 1 && loc < xs.rest;
  if (cut_at && !cut && tid == 0) *cut_at = TailCut{};
  const int n_units = xs.rounds + (loc < xs.rest * xs.slices ? 1 : 0);
  if (n_units == 0) return;

  const int wave_u = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wstep = a.w_tiled ? (BKB / kTileBytes) * kTilePiece : BKB;  // bytes from one K tile of W to the next
  const T* X = static_cast<const T*>(a.X);

  // Units j0 .. j0 + 63, one per lane, into the table's half (j0 / 64) & 1.  Every wavefront writes the same values and
  // reads what it wrote itself; no wavefront is a whole unit ahead of another, so the other half is never in use.
  // With equal heights the workgroups of an XCD move on by one tile per round: tiles of a chunk differ by a unit, and with a
  // power of two of them a workgroup would meet the same one in every round (5800 tokens 3133 -> 3107 us).
  auto fill_units = [&](int j0) {
    const int j = min(j0 + lane, n_units - 1);
    QuadUnit u = {};
    int lin;
    if (j < xs.rounds) {
      int l = plan.even_heights ? loc : loc + j;
      l -= l / nper * nper;
      lin = xcd_round_tile(xs, nper, xcd, l, j);
      u.kb = 0;
      u.kn = k_all;
      u.tu = -1;
    } else {
      const int s = loc / xs.rest, t = loc - s * xs.rest;
      lin = xs.tail_base + t;
      u.kb = s * k_all / xs.slices;
      u.kn = (s + 1) * k_all / xs.slices - u.kb;
      u.tu = xs.slices > 1 ? s * xs.rest + t : -1;
    }
    quad_tile_at(a, walk, block, plan.even_heights, lin, k_all, u);
    unit_table[(j0 / kUnitTable) & 1][lane] = u;
    if (cut_at && cut && tid < kUnitTable && tid == n_units - 1 - j0)  // (thread = lane: u is unit j0 + tid)
      *cut_at = TailCut{u.row0, u.units, u.f, u.expert, xs.slices, xs.rest, quad_buffers(a, plan.tallest), quad_buffer_rows(plan.tallest)};
  };
  auto unit_at = [&](int j) {
    const QuadUnit& s = unit_table[(j / kUnitTable) & 1][j % kUnitTable];
    QuadUnit u;
    u.row0 = __builtin_amdgcn_readfirstlane(s.row0);
    u.units = __builtin_amdgcn_readfirstlane(s.units);
    u.f = __builtin_amdgcn_readfirstlane(s.f);
    u.expert = __builtin_amdgcn_readfirstlane(s.expert);
    u.kb = __builtin_amdgcn_readfirstlane(s.kb);
    u.kn = __builtin_amdgcn_readfirstlane(s.kn);
    u.tu = __builtin_amdgcn_readfirstlane(s.tu);
    u.share = __builtin_amdgcn_readfirstlane(s.share);
    return u;
  };
  // Features of a tile: the last tile of a width that is no multiple of the tile's starts early instead of ending short
  // (its first columns are the previous tile's last ones, same operands, same sums).
  auto first_col = [&](int f) { return min(f * COLS, a.N - COLS); };
  // row of W behind row r of a weight tile whose first column is f0
  auto w_row = [&](int f0, int r) { return EPI == EPI_SILU ? (r / COLS) * a.N + f0 + r % COLS : f0 + r; };

  // sorted id -> token row, by multiplication (ids below 2^31; a.div_mul and a.div_shift from quad_divisor)
  auto div_top_k = [&](int sid) { return a.top_k == 1 ? static_cast<unsigned>(sid) : __umulhi(static_cast<unsigned>(sid), a.div_mul) >> a.div_shift; };
  const unsigned xpitch = static_cast<unsigned>(a.ldx * ES);

  // ---- per-lane addresses ------------------------------------------------------------------
  // Tile load q of wavefront w fills LDS rows [32 q + 8 w, + 8) of the X or W tile, lane -> (row, 16-byte chunk); rows 32
  // apart share their swizzle key, so the weight rows of the eight loads differ by wavefront-uniform distances only.
  const int lrow = wave_u * 8 + lane / CPR, lchunk = swizzle<CPR>(lrow, lane % CPR);
  const unsigned wlane = static_cast<unsigned>(w_byte_offset(a.w_tiled, a.ldw, a.K, lrow, lchunk * 16, ES));
  const unsigned wgap1 = static_cast<unsigned>(w_byte_offset(a.w_tiled, a.ldw, a.K, 32, 0, ES));
  const unsigned wgap2 = static_cast<unsigned>(w_byte_offset(a.w_tiled, a.ldw, a.K, 64, 0, ES));
  // fragments: one address per operand and K-step, the fragments at immediate offsets
  const int frow = lane % TILE, kgrp = lane / TILE;
  const int key0 = swizzle<CPR>(frow, 0);
  int xadr[2][FC];  // byte addresses in slot 0 of the chunks of row frow of the X tile (the W tile: XBYTES further)
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int c = 0; c < FC; ++c) xadr[s][c] = (frow * CPR + (((s * KG + kgrp) * FC + c) ^ key0)) * 16;
#define FQ_XD(i_) ((i_) * TILE * CPR * 16)
#define FQ_WD(j_) ((acc_tile_col<C, EPI>(0, (j_)) - acc_tile_col<C, EPI>(0, 0)) * CPR * 16)

  // ---- address sets: A = unit being multiplied, B = the workgroup's next unit ---------------------
  QuadUnit uA, uB;
  int n_sid[XI], n_tsid = 0;
  unsigned xsrcA[XI], xsrcB[XI];
  unsigned wlA = 0, whA = 0, wlB = 0, whB = 0;          // W: byte offset of loads 0..3 and 4..7 of the tile
  unsigned twA = 0, txA = 0, twB = 0, txB = 0;          // touch offsets (weight rows, token rows) of this lane
  __amdgpu_buffer_rsrc_t xrsA, wrsA, xrsB, wrsB;
  // Touch shares.  Weight K tile (256 rows): shared by the share >> 16 token tiles of the chunk, tile `index` asks for
  // rows [index * per, + per), per = ceil(256 / count), a quarter of them per wavefront.  Token K tile: shared by
  // the feature tiles of the token tile an XCD holds at one time, about 32 / count of them, at most kQuadXShare.
#define FQ_TOUCH_ROWS(u_, wrow_, xrow_, xon_)                                                  \
  {                                                                                            \
    const int cnt_ = max(1, min((u_).share >> 16, 32));                                        \
    const int per_ = (BF + cnt_ - 1) / cnt_, pw_ = (per_ + NW - 1) / NW;                       \
    wrow_ = min(((u_).share & 0xFFFF) * per_ + wave_u * pw_ + (lane < pw_ ? lane : 0), BF - 1); \
    const int xs_ = max(1, min(kQuadXShare, 32 / cnt_)), rows_ = (u_).units * kUnitRows;       \
    const int xper_ = (rows_ + xs_ - 1) / xs_, xw_ = (xper_ + NW - 1) / NW;                    \
    xrow_ = ((u_).f % xs_) * xper_ + wave_u * xw_ + (lane < xw_ ? lane : 0);                   \
    xon_ = lane < xw_ && xrow_ < rows_;                                                        \
    xrow_ = min(xrow_, rows_ - 1);                                                             \
  }
  // A lane constant as if it came to be here: the compiler works what depends on it out in place, instead of ahead of all
  // units and keeping it in registers through the K loops (which cost 40 to 140 spilled registers, some of them reloaded
  // in a K loop).
#define FQ_HERE(v_) asm volatile("" : "+v"(v_));
  // sorted ids of the unit's load rows; a row beyond the tile counts as padding
#define FQ_IDS(u_, sid_, tsid_)                                                                \
  {                                                                                            \
    const int rows_i = (u_).units * kUnitRows;                                                 \
    int lrow_ = lrow;                                                                          \
    FQ_HERE(lrow_)                                                                             \
    _Pragma("unroll") for (int q = 0; q < XI; ++q) {                                           \
      const int rr = q * kUnitRows + lrow_;                                                    \
      sid_[q] = a.sorted[(u_).row0 + min(rr, rows_i - 1)];                                     \
    }                                                                                          \
    int wr_, xr_; bool xo_;                                                                    \
    FQ_TOUCH_ROWS(u_, wr_, xr_, xo_)                                                           \
    (void)wr_; (void)xo_;                                                                      \
    tsid_ = a.sorted[(u_).row0 + xr_];                                                         \
  }
  // The set of unit u_ in parts, so that the parts can stand between MFMAs.  Offsets are bytes within 4 GiB (checked by the
  // launcher).  live_: 1, or 0 for the set behind a workgroup's last unit, whose loads all fall outside empty resources.
#define FQ_SET_RSRC(u_, live_, wl_, wh_, xrs_, wrs_)                                                         \
  {                                                                                                          \
    const int64_t xrow0_ = a.top_k > 0 ? 0 : static_cast<int64_t>((u_).row0);                                \
    xrs_ = uniform_rsrc(X + xrow0_ * a.ldx, (a.x_span ? a.x_span : 0xFFFFFFFFu) * static_cast<unsigned>(live_)); \
    wrs_ = uniform_rsrc(static_cast<const T*>(a.W) + static_cast<int64_t>((u_).expert) * a.w_expert_stride, 0xFFFFFFFFu * static_cast<unsigned>(live_)); \
    const int f0_ = first_col((u_).f);                                                                       \
    wl_ = static_cast<unsigned>(w_byte_offset(a.w_tiled, a.ldw, a.K, f0_, 0, ES));                           \
    wh_ = static_cast<unsigned>(w_byte_offset(a.w_tiled, a.ldw, a.K, w_row(f0_, BF / 2), 0, ES));            \
  }
#define FQ_SET_ROW(u_, sid_, q_, xsrc_)                                                                      \
  {                                                                                                          \
    int lrow_ = lrow;                                                                                        \
    FQ_HERE(lrow_)                                                                                           \
    const bool pad_ = (q_) >= (u_).units || (sid_) >= a.num_valid;                                           \
    unsigned row_ = a.top_k > 0 ? div_top_k(sid_) : (q_) * kUnitRows + lrow_;                                \
    row_ = pad_ ? 0u : row_;                                                                                 \
    const unsigned off_ = row_ * xpitch + lchunk * 16;                                                       \
    xsrc_ = a.x_span && pad_ ? kSkipOffset : off_;                                                           \
  }
#define FQ_SET_TOUCH(u_, tsid_, tw_, tx_)                                                                    \
  {                                                                                                          \
    int wrow_, xrow_; bool xon_;                                                                             \
    FQ_TOUCH_ROWS(u_, wrow_, xrow_, xon_)                                                                    \
    tw_ = static_cast<unsigned>(w_byte_offset(a.w_tiled, a.ldw, a.K, w_row(first_col((u_).f), wrow_), 0, ES)); \
    const bool tpad_ = !xon_ || (tsid_) >= a.num_valid;                                                      \
    unsigned trow_ = a.top_k > 0 ? div_top_k(tsid_) : static_cast<unsigned>(xrow_);                          \
    trow_ = tpad_ ? 0u : trow_;                                                                              \
    tx_ = a.x_span && tpad_ ? kSkipOffset : trow_ * xpitch;                                                  \
  }
  // tile load q (weight rows first) of K tile tile_ of set SET into ring slot slot_
#define FQ_ISSUE(SET, tile_, slot_, q_)                                                                     \
  {                                                                                                         \
    if ((q_) < WI) {                                                                                        \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(                                                             \
          wrs##SET, (lptr_t)(lds_raw + (slot_) * SLOT + XBYTES + ((q_) * NW + wave_u) * (kWave * 16)),      \
          16, wlane, (((q_) & 4) ? wh##SET : wl##SET) + (((q_) & 2) ? wgap2 : 0) + (((q_) & 1) ? wgap1 : 0) + (tile_) * wstep, 0, WAUX); \
    } else {                                                                                                \
      __builtin_amdgcn_raw_ptr_buffer_load_lds(                                                             \
          xrs##SET, (lptr_t)(lds_raw + (slot_) * SLOT + (((q_) - WI) * NW + wave_u) * (kWave * 16)),        \
          16, xsrc##SET[(q_) < WI ? 0 : (q_) - WI], (tile_) * BKB, 0, 0);                                   \
    }                                                                                                       \
  }
  // touch of K tile tile_ of set SET
#define FQ_TOUCH_ISSUE(SET, tile_)                                                                          \
  {                                                                                                         \
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs##SET, (lptr_t)(lds_raw + 2 * SLOT + wave_u * 256), 4, tw##SET, (tile_) * wstep, 0, 0);  \
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs##SET, (lptr_t)(lds_raw + 2 * SLOT + wave_u * 256), 4, tx##SET, (tile_) * BKB, 0, 0); \
  }
#define FQ_FENCE __builtin_amdgcn_sched_barrier(0);
  // One K-step: the MFMAs of fragment set S.  FIRST: the accumulators start from zero.  RD: the fragments of K-step
  // S ^ 1 are read from ring slot rsl_.  NLD_ (0: none): the first NLD_ loads of K tile ltile_ of set LSET go into slot
  // lsl_, and behind the last MFMA the touch of K tile ttile_ of set TSET goes out.
  // Read r goes behind MFMA r * span / N2, load q behind MFMA (q + 1/2) * (NM - 1) / NLD_, out of the reads' way.
#define FQ_KSTEP(S, FIRST, RD, rsl_, NLD_, LSET, ltile_, lsl_, TSET, ttile_, HOOK)                         \
  {                                                                                                        \
    _Pragma("unroll") for (int m = 0; m < NM; ++m) {                                                       \
      const int j = WOUT ? m / IN : m % IN, i = WOUT ? m % IN : m / IN;                                    \
      if (i < kQuadAgpr) quad_mfma<T, true, FIRST>(acc[j][i], fw[WOUT && j < OUT - KEEP2 ? 0 : (S)][j], fx[!WOUT && i < OUT - KEEP2 ? 0 : (S)][i]); \
      else quad_mfma<T, false, FIRST>(acc[j][i], fw[WOUT && j < OUT - KEEP2 ? 0 : (S)][j], fx[!WOUT && i < OUT - KEEP2 ? 0 : (S)][i]); \
      FQ_FENCE                                                                                             \
      HOOK(m)                                                                                              \
      if (RD) {                                                                                            \
        if (m % IN == IN - 1 && m / IN < OUT - KEEP2) {                                                    \
          if (WOUT) { FQ_READ_W(0, m / IN, (S) ^ 1, rsl_) } else { FQ_READ_X(0, m / IN, (S) ^ 1, rsl_) }   \
        }                                                                                                  \
        const int span_ = (S) == 0 ? RSPAN0 : RSPAN1, r = (m * N2 + span_ - 1) / span_;                    \
        if (r < N2 && r * span_ < (m + 1) * N2) {                                                          \
          if (r < IN) {                                                                                    \
            if (WOUT) { FQ_READ_X((S) ^ 1, r, (S) ^ 1, rsl_) } else { FQ_READ_W((S) ^ 1, r, (S) ^ 1, rsl_) } \
          } else {                                                                                         \
            if (WOUT) { FQ_READ_W((S) ^ 1, OUT - KEEP2 + r - IN, (S) ^ 1, rsl_) }                          \
            else { FQ_READ_X((S) ^ 1, OUT - KEEP2 + r - IN, (S) ^ 1, rsl_) }                               \
          }                                                                                                \
        }                                                                                                  \
      }                                                                                                    \
      if ((NLD_) > 0) {                                                                                    \
        _Pragma("unroll") for (int x = 0; x < ((NLD_) + NM - 2) / (NM - 1) + 1; ++x) {                         \
          const int q = (2 * m * (NLD_) + NM - 1) / (2 * (NM - 1)) + x;                                    \
          if (q < (NLD_) && (2 * q + 1) * (NM - 1) < 2 * (m + 1) * (NLD_)) {                               \
            FQ_ISSUE(LSET, ltile_, lsl_, q)                                                                \
            FQ_FENCE                                                                                       \
          }                                                                                                \
        }                                                                                                  \
        if (m == NM - 1 && TOUCH) {                                                                        \
          FQ_TOUCH_ISSUE(TSET, ttile_)                                                                     \
          FQ_FENCE                                                                                         \
        }                                                                                                  \
      }                                                                                                    \
    }                                                                                                      \
  }
#define FQ_READ_W(set_, j_, s_, sl_)                                                                       \
  {                                                                                                        \
    _Pragma("unroll") for (int c = 0; c < FC; ++c) {                                                       \
      fw[set_][j_][c] = *reinterpret_cast<const u32x4*>(lds_raw + xadr[s_][c] + wbase + (sl_) * SLOT + FQ_WD(j_)); \
      FQ_FENCE                                                                                             \
    }                                                                                                      \
  }
#define FQ_READ_X(set_, i_, s_, sl_)                                                                       \
  {                                                                                                        \
    _Pragma("unroll") for (int c = 0; c < FC; ++c) {                                                       \
      fx[set_][i_][c] = *reinterpret_cast<const u32x4*>(lds_raw + xadr[s_][c] + xbase + (sl_) * SLOT + FQ_XD(i_)); \
      FQ_FENCE                                                                                             \
    }                                                                                                      \
  }
  // the two newest memory operations of a wavefront at the barrier are the touches of the K tile before:
  // everything older - the tile loads the barrier publishes - has landed
#define FQ_SYNC(newest_)                                                                 \
  {                                                                                      \
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(newest_) : "memory");            \
    __builtin_amdgcn_s_barrier();                                                        \
    FQ_FENCE                                                                             \
  }
  // K tile t of the unit from ring slot par; its slot takes K tile ltile_ of set LSET
#define FQ_PERIOD(FIRST, RDLAST, NLD_, LSET, ltile_, TSET, ttile_, HOOK)                 \
  {                                                                                      \
    FQ_KSTEP(0, FIRST, true, par, 0, LSET, 0, 0, TSET, 0, HOOK)                          \
    FQ_SYNC((FIRST) || !TOUCH ? 0 : 2)                                                   \
    FQ_KSTEP(1, false, RDLAST, par ^ 1, NLD_, LSET, ltile_, par, TSET, ttile_, FQ_NO_HOOK) \
    par ^= 1;                                                                            \
  }
#define FQ_NO_HOOK(m_)
  // The next unit's coordinates and the loads of its sorted ids, behind the second MFMA of a K tile; its address set between
  // the MFMAs of the next K tile, a row in each gap.
#define FQ_HOOK_IDS(m_)                                                                  \
  if ((m_) == 1) {                                                                       \
    uB = unit_at(unit + live);                                                           \
    FQ_IDS(uB, n_sid, n_tsid)                                                            \
    FQ_FENCE                                                                             \
  }
#define FQ_HOOK_SET(m_)                                                                  \
  if ((m_) == 0) {                                                                       \
    FQ_SET_RSRC(uB, live, wlB, whB, xrsB, wrsB)                                          \
    FQ_FENCE                                                                             \
  }                                                                                      \
  _Pragma("unroll") for (int x = 0; x < HPER; ++x)                                       \
    if ((m_) >= 1 && ((m_) - 1) * HPER + x < XI) {                                       \
      FQ_SET_ROW(uB, n_sid[((m_) - 1) * HPER + x < XI && (m_) >= 1 ? ((m_) - 1) * HPER + x : 0], ((m_) - 1) * HPER + x, \
                 xsrcB[((m_) - 1) * HPER + x < XI && (m_) >= 1 ? ((m_) - 1) * HPER + x : 0]) \
      FQ_FENCE                                                                           \
    }                                                                                    \
  if ((m_) == NM - 1) {                                                                  \
    FQ_SET_TOUCH(uB, n_tsid, twB, txB)                                                   \
    FQ_FENCE                                                                             \
  }

  fill_units(0);
  uA = unit_at(0);
  // K tiles the next loads and the next touches ask for: a unit's follow each other round the end of K
  auto next_k = [&](int k) { return k + 1 == k_all ? 0 : k + 1; };
  int lw = uA.kb, tw;
  {
    // fill: the first two K tiles into slots 0 and 1, the weights while the sorted ids are on their way
    constexpr int WAUX = 0;
    const int k1 = next_k(lw);
    int sid0[XI], tsid0;
    FQ_IDS(uA, sid0, tsid0)
    FQ_SET_RSRC(uA, 1, wlA, whA, xrsA, wrsA)
    FQ_FENCE
#pragma unroll
    for (int q = 0; q < WI; ++q) FQ_ISSUE(A, lw, 0, q)
#pragma unroll
    for (int q = 0; q < WI; ++q) FQ_ISSUE(A, k1, 1, q)
    FQ_FENCE
#pragma unroll
    for (int q = 0; q < XI; ++q) FQ_SET_ROW(uA, sid0[q], q, xsrcA[q])
#pragma unroll
    for (int q = WI; q < WI + XI; ++q) FQ_ISSUE(A, lw, 0, q)
#pragma unroll
    for (int q = WI; q < WI + XI; ++q) FQ_ISSUE(A, k1, 1, q)
    FQ_SET_TOUCH(uA, tsid0, twA, txA)
    lw = next_k(k1);
    tw = next_k(lw);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(XI) : "memory");
  __builtin_amdgcn_s_barrier();
  int par = 0, unit = 0;

  // One work unit of UN units of rows (or fewer: rows beyond the tile are padding): kn >= kQuadMinTiles K tiles; ALONE: the only
  // tile on its weight tile (no touch, weights non-temporal).  The ring
  // holds the unit's first two K tiles when it starts.  The next unit's routing data is asked for five K tiles before the end
  // and turned into the address set B in the next one (the K loop proper keeps one set in registers); the last three K tiles
  // touch its first three, and its first two refill the ring during the last two.
  auto run_unit = [&](auto height, auto alone) __attribute__((always_inline)) {
    constexpr int UN = decltype(height)::value;
    constexpr bool ALONE = decltype(alone)::value, TOUCH = !ALONE;
    constexpr int WAUX = ALONE ? 2 : 0;  // cache policy of the weight loads (2: non-temporal)
    typedef QuadCfg<T, UN> C;
    // the operand walked slowest: the weights, or the token rows where a wavefront has all of them
    constexpr bool WOUT = C::WT == 2;
    constexpr int KEEP2 = FC == 1 ? 2 : 1;              // its last fragments, which have two register sets like the other operand
    constexpr int IT = C::IT, JF = C::JF, OUT = WOUT ? JF : IT, IN = WOUT ? IT : JF, NM = OUT * IN;
    const int wt = wave_u / C::WF, wf = wave_u % C::WF;
    const int wbase = XBYTES + acc_tile_col<C, EPI>(wf, 0) * CPR * 16;
    constexpr int N2 = IN + KEEP2;                      // fragments with two register sets
    constexpr int HPER = (XI + NM - 3) / (NM - 2);      // rows of the next unit's address set per MFMA
    // MFMAs their reads are spread over: in the first K-step they end well before the barrier that waits for them
    constexpr int RSPAN0 = NM * 5 / 8 < N2 ? N2 : NM * 5 / 8, RSPAN1 = NM * 7 / 8 < N2 ? N2 : NM * 7 / 8;
    const int xbase = wt * C::TT * CPR * 16;
    acc_t acc[JF][IT];
    u32x4 fw[2][JF][FC], fx[2][IT][FC];
#pragma unroll
    for (int i = 0; i < IT; ++i) FQ_READ_X(0, i, 0, par)
#pragma unroll
    for (int j = 0; j < JF; ++j) FQ_READ_W(0, j, 0, par)
    const int live = min(n_units - 1 - unit, 1);  // 0: this is the workgroup's last unit
    const int kn = uA.kn;
#define FQ_NEXT { lw = next_k(lw); tw = next_k(tw); }
    FQ_PERIOD(true, true, WI + UN, A, lw, A, tw, FQ_NO_HOOK)
    FQ_NEXT
    __builtin_amdgcn_s_waitcnt(0xC07F); /* lgkmcnt(0): no scalar load pending inside the loop */
    for (int t = 1; t < kn - 5; ++t) {
      FQ_PERIOD(false, true, WI + UN, A, lw, A, tw, FQ_NO_HOOK)
      FQ_NEXT
    }
    FQ_PERIOD(false, true, WI + UN, A, lw, A, tw, FQ_HOOK_IDS)
    FQ_NEXT
    FQ_PERIOD(false, true, WI + UN, A, lw, A, tw, FQ_HOOK_SET)
    lw = next_k(lw);
    tw = uB.kb;
    FQ_PERIOD(false, true, WI + UN, A, lw, B, tw, FQ_NO_HOOK)
    lw = tw;
    tw = next_k(tw);
    FQ_PERIOD(false, true, WI + XI, B, lw, B, tw, FQ_NO_HOOK)
    FQ_NEXT
    FQ_PERIOD(false, false, WI + XI, B, lw, B, tw, FQ_NO_HOOK)
    FQ_NEXT
#undef FQ_NEXT
    // the last MFMA's result is up to 19 wait states away, which the compiler does not know
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory");
    FQ_FENCE
    int frow_e = frow, kgrp_e = kgrp;
    FQ_HERE(frow_e)
    FQ_HERE(kgrp_e)
    if (uA.tu < 0)
      quad_epilogue<T, C, EPI>(a, acc, uA.row0, uA.row0 + uA.units * kUnitRows, first_col(uA.f), uA.expert, wt, wf, frow_e, kgrp_e);
    else
      tail_store<C, EPI, kQuadAgpr>(
          a.tail_ws + static_cast<int64_t>(xcd * quad_buffers(a, plan.tallest) + uA.tu) * (quad_buffer_rows(plan.tallest) * BF),
          acc, wt, wf, frow_e, kgrp_e);
  };
  for (;; ++unit) {
    // a loop of its own for every height from 4 on (fp8: 9 and the even ones), 2 and 4 for those below; alone: 7, 6, 4 and 2
    const int height = uA.units;
    if (unit + 1 < n_units && (unit + 1) % kUnitTable == 0) fill_units(unit + 1);
    if (uA.share == 1 << 16 && height <= kAloneUnits && a.spread_k) {
      if (height == 7) run_unit(std::integral_constant<int, kAloneUnits>(), std::true_type());
      else if (height >= 5) run_unit(std::integral_constant<int, 6>(), std::true_type());
      else if (height >= 3) run_unit(std::integral_constant<int, 4>(), std::true_type());
      else run_unit(std::integral_constant<int, 2>(), std::true_type());
    } else if (height == 9) run_unit(std::integral_constant<int, 9>(), std::false_type());
    else if (height == 8 || (sizeof(T) == 1 && height == 7)) run_unit(std::integral_constant<int, 8>(), std::false_type());
    else if (sizeof(T) != 1 && height == 7) {
      if constexpr (sizeof(T) != 1) run_unit(std::integral_constant<int, 7>(), std::false_type());
    } else if (height == 6 || (sizeof(T) == 1 && height == 5)) run_unit(std::integral_constant<int, 6>(), std::false_type());
    else if (sizeof(T) != 1 && height == 5) {
      if constexpr (sizeof(T) != 1) run_unit(std::integral_constant<int, 5>(), std::false_type());
    } else if (height >= 3) run_unit(std::integral_constant<int, 4>(), std::false_type());
    else run_unit(std::integral_constant<int, 2>(), std::false_type());
    if (unit + 1 >= n_units) break;
    uA = uB; xrsA = xrsB; wrsA = wrsB; wlA = wlB; whA = whB; twA = twB; txA = txB;
#pragma unroll
    for (int q = 0; q < XI; ++q) xsrcA[q] = xsrcB[q];
  }
  // the loads behind the last unit fetched nothing, but none may be pending when the workgroup gives its LDS back
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#undef FQ_HOOK_SET
#undef FQ_HOOK_IDS
#undef FQ_NO_HOOK
#undef FQ_PERIOD
#undef FQ_SYNC
#undef FQ_KSTEP
#undef FQ_FENCE
#undef FQ_READ_X
#undef FQ_READ_W
#undef FQ_TOUCH_ISSUE
#undef FQ_ISSUE
#undef FQ_SET_TOUCH
#undef FQ_SET_ROW
#undef FQ_SET_RSRC
#undef FQ_HERE
#undef FQ_IDS
#undef FQ_TOUCH_ROWS
#undef FQ_XD
#undef FQ_WD
#endif
}

// Sums the K slices of the last round's tiles and applies the epilogue: one workgroup per 32 rows of a tile.  What a tile is
// the GEMM launch has written down; a launch without a cut tile costs 5 us (11 with the walk worked out again here).
template <typename T, int EPI>
__global__ __launch_bounds__(256) void quad_fixup_kernel(const GemmArgs a, int nper) {
  constexpr int BF = QuadCfg<T, kMaxUnits>::BF;
  const int half = nper / 2;
  const int xcd = blockIdx.x / (half * kMaxUnits), t = (blockIdx.x / kMaxUnits) % half, rb = blockIdx.x % kMaxUnits;
  const TailCut c = reinterpret_cast<const TailCut*>(a.tail_desc)[xcd * nper + t];
  if (rb >= c.units || c.slices < 2) return;
  const int64_t buffer = static_cast<int64_t>(c.buffer_rows) * BF;
  const float* first = a.tail_ws + (xcd * c.buffers + t) * buffer;
  // widths that are no multiple of a tile's are not cut: no tile starts early here
  fixup_rows<T, BF, EPI>(a, first, c.rest * buffer, c.slices, c.row0, rb * kUnitRows, c.f * (EPI == EPI_SILU ? BF / 2 : BF), c.expert);
}

// Workgroups resident at once on the current device: one per CU (a multiple of 8, one share per XCD).
template <typename T, int EPI>
int quad_grid(int* grid_out) {
  constexpr int kMaxDevices = 64;
  constexpr int kLds = kQuadRing + kQuadSink;
  static int cached[kMaxDevices] = {};  // per device; a race between threads writes the same value twice
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) return fail(FR_E_LAUNCH, "quad GEMM: device %d (%s)", dev, hipGetErrorString(e));
  if (!cached[dev]) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&moe_gemm_quad_kernel<T, EPI>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    int cus = 0, per_cu = 0;
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, moe_gemm_quad_kernel<T, EPI>, 256, kLds);
    if (e != hipSuccess) {
      (void)hipGetLastError();  // reported here: not to be found again by the next launch check
      return fail(FR_E_LAUNCH, "quad GEMM set-up (%d B LDS): %s", kLds, hipGetErrorString(e));
    }
    if (per_cu < 1 || cus < 8) return fail(FR_E_LAUNCH, "quad GEMM: occupancy %d on %d CUs", per_cu, cus);
    cached[dev] = cus / 8 * 8;  // one workgroup per CU: a second would share the SIMDs' MFMA pipes
  }
  *grid_out = cached[dev];
  return FR_OK;
}

// n / d as umulhi(n, mul) >> shift for n < 2^31 and 2 <= d < 2^31 (round-up reciprocal of 31 + ceil(log2 d) bits: its error
// times n stays below one unit in the last place of the quotient).
inline void quad_divisor(int d, unsigned* mul, int* shift) {
  int l = 0;
  while (l < 31 && (int64_t(1) << l) < d) ++l;
  *mul = d >= 2 ? static_cast<unsigned>((uint64_t(1) << (31 + l)) / d + 1) : 0u;
  *shift = l > 0 ? l - 1 : 0;
}

// The list of cut tiles where the caller has no place for it but the scratch
inline int* tail_desc_in(float* tail_ws) { return reinterpret_cast<int*>(tail_ws + kTailUnits * 256 * 256) - kTailDescBytes / 4; }

// nper: workgroups per XCD of the GEMM launch
template <typename T, int EPI>
int launch_quad_fixup(const GemmArgs& a, int nper, hipStream_t st) {
  if (nper < 2) return FR_OK;
  hipLaunchKernelGGL((quad_fixup_kernel<T, EPI>), dim3(8 * (nper / 2) * kMaxUnits), dim3(256), 0, st, a, nper);
  return check_launch("quad_fixup_kernel");
}

// Launches the one-wavefront-per-SIMD kernel on routing arrays of `block` rows (a multiple of 32, at most 256; num_t_blocks
// and num_f_tiles filled for `block` rows and 256 features) for a single K split with at least kQuadMinTiles K tiles per work
// unit.  Returns 1 when the shape is not one it takes (nothing launched: the caller takes another kernel).
template <typename T, int EPI>
int launch_gemm_quad(const GemmArgs& a_in, int block, int splits, hipStream_t st) {
  typedef QuadCfg<T, kMaxUnits> C;
  GemmArgs a = a_in;
  constexpr int ES = static_cast<int>(sizeof(T)), BK = C::BKB / ES;
  constexpr int COLS = (EPI == EPI_SILU) ? C::BF / 2 : C::BF;
  if (a.setup_only) {
    int resident = 0;
    return quad_grid<T, EPI>(&resident);
  }
  // a K slice of the split tail has at least k tiles / kTailMaxSplit K tiles (and never under kTailMinSlice)
  if (splits != 1 || a.K % BK != 0 || a.K / BK < 2 * kQuadMinTiles || a.num_experts < 1 || a.num_experts > kMaxExperts) return 1;
  // a width below a tile's has no last tile to start early; one that is no multiple adds columns twice in the atomic epilogue
  if (a.N < COLS || (a.add_div && a.N % COLS != 0)) return 1;
  const int64_t x_rows = a.top_k > 0 ? a.num_valid / a.top_k : C::BT;
  const int64_t w_rows = EPI == EPI_SILU ? 2 * static_cast<int64_t>(a.N) : a.N;
  const int64_t lim = int64_t(1) << 32;
  if (x_rows * a.ldx * ES >= lim || w_rows * a.ldw * ES >= lim)
    return fail(FR_E_SHAPE, "token rows (%lld x %lld) or one expert's weights (%lld x %lld) span 4 GiB or more",
                (long long)x_rows, (long long)a.ldx, (long long)w_rows, (long long)a.ldw);
  a.group_t = tunables().group_m ? tunables().group_m : kChunkBlocks;
  if (tunables().no_tail_split) a.tail_ws = nullptr;
  a.spread_k = a.N % COLS == 0;
  quad_divisor(a.top_k, &a.div_mul, &a.div_shift);
  a.x_span = x_rows * a.ldx * ES < (int64_t(1) << 31) ? static_cast<unsigned>(x_rows * a.ldx * ES) : 0u;
  int resident = 0;
  const int rc = quad_grid<T, EPI>(&resident);
  if (rc != FR_OK) return rc;
  const int64_t worst = static_cast<int64_t>(a.num_t_blocks) * a.num_f_tiles;
  // After many whole rounds the workgroups are no longer in step (tiles of several heights, hand-overs), and cutting the last
  // round buys less than its slices' fp32 round trip costs - the sooner the shorter a tile's K loop is: gate/up
  // (64 K tiles) with / without the split 681 / 684 us at 8.8 rounds (1536 tokens), 832 / 816 at 10.5, 1030 / 988
  // at 12.5, 1521 / 1505 at 17.5, 5743 / 5723 at 70; the down projection (224 K tiles) 785 / 915 at 2.7 rounds,
  // 2803 / 2979 at 11; fp8 down projection (112 K tiles) 1743 / 1794 at 8.5 rounds; 96 K tiles (H = 6144) 1138 / 1135
  // at 10 rounds, 1442 / 1437 at 12.
  const int64_t max_rounds = a.K / BK >= 112 ? 16 : 8;
  const bool tail = a.tail_ws && a.K / BK >= kTailMinTiles && a.N % COLS == 0 && worst * block < max_rounds * resident * 256;
  a.tail_buffers = 32;
  a.tall_buffers = a.tail_tall ? 32 : kQuadTallBuffers;
  if (a.tail_ws && !a.tail_desc) a.tail_desc = tail_desc_in(a.tail_ws);
  if (a.tail_ws && a.tail_desc == tail_desc_in(a.tail_ws)) a.tail_buffers = 31;
  if (!tail) a.tail_ws = nullptr;
  if (!tail && !a.by_runs) a.tail_desc = nullptr;
  int64_t grid = resident;
  if (grid > kTailUnits && (tail || a.by_runs)) grid = kTailUnits;
  hipLaunchKernelGGL((moe_gemm_quad_kernel<T, EPI>), dim3(static_cast<unsigned>(grid)), dim3(256), kQuadRing + kQuadSink, st, a, block);
  int lrc = check_launch("moe_gemm_quad_kernel");
  if (lrc != FR_OK || !tail || a.by_runs) return lrc;
  return launch_quad_fixup<T, EPI>(a, static_cast<int>(grid / 8), st);
}

// A GEMM whose tile form only the experts' runs can decide: tall tiles and the tiles C of the routing block are both launched, and
// the device has one of them return at once (runs_fill_tall_tiles).  The one that works lists the tiles it cuts, which one
// fix-up launch sums.  a: filled for `block` rows and 256 features.  Returns 1 as launch_gemm_quad does.
// Near-uniform loads, which is all the host can price, are multiplied up to a fifth faster by tall tiles, skewed ones up to a
// quarter slower: an expert with several tiles leaves the others' short ones to wait for its rounds.
template <typename T, typename C, int EPI>
int launch_gemm_by_runs(const GemmArgs& a_in, int block, hipStream_t st) {
  GemmArgs a = a_in;
  int tall_grid = 0, block_grid = 0;
  int rc = quad_grid<T, EPI>(&tall_grid);
  if (rc == FR_OK) rc = persistent_grid<T, C, EPI, true>(&block_grid);
  if (rc != FR_OK) return rc;
  if (tall_grid != block_grid) return 1;  // the list of cut tiles is one per workgroup
  if (tunables().no_tail_split) a.tail_ws = nullptr;
  if (!a.tail_ws) a.tail_desc = nullptr;
  else if (!a.tail_desc) a.tail_desc = tail_desc_in(a.tail_ws);
  a.by_runs = a.any_height - kHeightsByRuns + 1;
  rc = launch_gemm_quad<T, EPI>(a, block, 1, st);
  if (rc != FR_OK) return rc;
  GemmArgs b = a;
  if (sizeof(T) == 1 && EPI == EPI_SILU) b.tail_ws = nullptr;  // fp8's gate/up GEMM does not cut these tiles
  rc = launch_gemm_persistent<T, C, EPI, true>(b, 1, st);
  if (rc != FR_OK || !a.tail_desc) return rc;
  return launch_quad_fixup<T, EPI>(a, (tall_grid < kTailUnits ? tall_grid : kTailUnits) / 8, st);
}

}  // namespace fr
