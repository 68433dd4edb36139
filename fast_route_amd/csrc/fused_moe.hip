// Composite entry points: tile plan, workspace carving, and the whole layer as
// one sequence of launches on the caller's stream.
#include "fr_common.h"
#include <cmath>

namespace fr {
namespace {

constexpr int64_t kAlign = 256;
int64_t aligned(int64_t bytes) { return round_up(bytes, kAlign); }

fr_moe_tunables g_tunables = {0, 0, 0, 0, 0};
constexpr int64_t kStaticScratchBytes = int64_t(64) << 20;  // see fr_fused_moe_noalloc

// expected multiples of `rows` that hold an expert's pairs: `avg` pairs per expert, spread as under uniform routing
double expected_blocks(double avg, int E, int rows) {
  const double sigma = sqrt(avg * (1.0 - 1.0 / E)) + 1e-9;
  double sum = 1.0;
  for (int k = 1; k * rows < avg + 8 * sigma; ++k) sum += 0.5 * erfc((static_cast<double>(k) * rows - avg) / (sigma * 1.4142135623730951));
  return sum;
}

// A layer whose plan routes for 128 or 160 rows and runs the one-wavefront-per-SIMD kernel all the same, with tiles as tall as
// the experts' runs (moe_gemm_quad.h).  Layer in us, the plan's own tiles / that kernel:
//   H = 4096, F = 14336, 8 experts   bf16 1240 tokens (310 pairs per expert) 973 / 893, 1280 995 / 908, 1430 1078 / 945, 1500
//                                    1133 / 969, 2300 1480 / 1406, 2420 1520 / 1478; fp8 1250 614 / 556
//   16 experts, F = 8192, fp16       2490 (311) 1108 / 1065, 4400 1727 / 1581
//   H = 3072, F = 4096, 16 experts   4500 (562) 0.96, 5000 0.92 of the plan's tiles
//   H = 2048, F = 1408, 64 experts, top-6, Zipf-skewed: 5600 (525) 1.04 to 1.06, 5900 (553) 0.96, 6200 0.96 to 0.99, 7100 0.97
//   H = 2048, F = 8192, 8 experts    2200 (550) 0.98, 2500 0.92; fp8 0.92, 0.85
//   H = 1024, F = 3584, 8 experts    2200 to 4096 0.93 to 1.03, 4142 (1036) 0.87
// With fewer pairs (H >= 4096), where an expert's run is one tile of it and the plan's rows make it two: the weights pass through the
// CUs once.  Up to 7 units (fp8: 6) such a tile streams its weights (moe_gemm_quad.h); 8 and 9 units gain less and lose to
// the plan's tiles in a launch of few.  That holds for runs of about the same length, which is all that is priced here: with skewed loads the
// plan's tiles are faster, so the device chooses by the runs (launch_gemm_by_runs; its second launch of either GEMM costs 4 to 5 us).
// Layer in parts of the time with the plan's tiles, near-uniform load tall tiles / chosen by runs, and Zipf-skewed load tall / by runs:
//   H = 4096, F = 14336, 8 experts   645 tokens 0.845 / 0.855, 1.10 / 1.00; 850 0.94 / 0.94, 1.13 / 1.005; 1031 0.96 / 0.965, 1.07 / 1.01
//                                    fp8 640 0.83 / 0.84, 1.10 / 1.03, but 700 (175 pairs) 0.99 / 1.005, 1.06 / 1.02: up to 167
//   H = 6144, F = 16384              900 0.925 / 0.93, 1.20 / 1.01;  H = 5120, F = 8192, 16 experts 1350 0.86 / 0.865, 1.18 / 1.00
//   16 experts, F = 8192, fp16       1300 0.84 / 0.85, 1.11 / 1.00;  H = 7168, F = 2048, 64 experts, top-8 1350 0.88 / 0.885, 1.09 / 1.005
//   H = 4096, F = 4096, 8 experts    640 0.835 / 0.86, 1.15 / 1.025; F = 1536, 32 experts, top-4 1350 0.955 / 0.97, 1.15 / 1.02
// Tall tiles for every load, near-uniform, the plan's tiles / tall:
//   H = 4096, F = 14336, 8 experts   645 (161) 735 / 635, 700 735 / 637, 850 783 / 702, 950 802 / 778, 1031 (258) 832 / 797, 1080
//                                    845 / 826, but 1120 (280: some experts two tiles) 841 / 851, 1160 855 / 881, 1200 880 / 890
//                                    fp8 640 441 / 397, 700 426 / 401, but 740 (185) 437 / 433, 800 442 / 452, 950 475 / 473
//   H = 6144, F = 16384              700 1280 / 1108, 1000 1425 / 1342; one block of 160 rows per expert: 580 (145) 958 / 1097
//   16 experts, F = 8192, fp16       1240 (155) 753 / 679, 1300 837 / 688, 1900 963 / 866, 2200 (275) 1008 / 1037; one block: 700
//                                    593 / 611, 960 (120) 610 / 650, 1100 652 / 668
//   H = 5120, F = 8192, 16 experts   1350 (169) 1075 / 922, 2000 1214 / 1099; H = 7168, F = 2048, 64 experts, top-8 1350 1487 / 1311
//   H = 4096, F = 4096, 8 experts    640 250 / 203, 750 251 / 220, but 1000 (250; 256 gate/up tiles) 270 / 281; F = 1536, 32
//                                    experts, top-4 1350 358 / 333, 1700 382 / 367, 2000 (250; 384) 400 / 409
// A few tiles leave the chip idle whatever their height, and the smaller ones less of it: one expert, F = 4096 (64 gate/up
// tiles) 350 tokens 1.20, 570 1.11, F = 2048 1.21, 1.13; 8 experts, F = 1024 (128 and 192 tiles) 1400 1.02, 2300 1.07; but one
// expert, F = 14336 (224) 0.97, 8 experts, F = 2048 (256) 1400 0.87.
// Only where the plan has a single K slice: that kernel writes a pair's row once, in the operands' 2-byte type, where several
// slices are summed from fp32 rows.
int any_height(int64_t M, int64_t H, int64_t F, int E, int topk, int dtype, const fr_moe_plan& p) {
  const fr_moe_tunables& t = g_tunables;
  if ((p.block != 128 && p.block != 160) || p.split_k > 1 || t.no_quad || t.block || E > 1022) return kHeightsOfBlock;
  const int es = dtype == FR_FP8_E4M3 ? 1 : 2;
  if (H * es < 2048 || F * es < 2048) return kHeightsOfBlock;  // 16 K tiles in both GEMMs
  const double avg = static_cast<double>(M) * topk / E, tall = expected_blocks(avg, E, 288), tiles = E * tall * (F / 128);
  if (avg >= (H >= 4096 ? 310.0 : H >= 2048 ? 550.0 : 1030.0)) return tiles >= 200.0 ? kHeightsAny : kHeightsOfBlock;
  if (H < 4096 || expected_blocks(avg, E, p.block) < 1.3) return kHeightsOfBlock;
  if (!((expected_blocks(avg, E, es == 2 ? 224 : 180) <= 1.13 && tiles >= 200.0) || (es == 2 && tall <= 1.13 && tiles >= 450.0))) return kHeightsOfBlock;
  if (p.block != 128 || avg < 222.0) return kHeightsByRuns;
  const int64_t up = E * ceil_div(F, 128);  // gate/up tiles with one per expert and feature tile; the plan has two
  return up % 256 != 0 && 2 * up % 256 == 0 ? kHeightsByLongRuns128 : kHeightsByRuns128;
}

struct Carve {
  float* topk_w;
  int32_t* topk_ids;
  int32_t* sorted;
  int32_t* expert_ids;
  int32_t* npost;
  void* align_ws;
  int64_t align_ws_bytes;
  void* act;
  float* partial;
  float* tail;       // scratch for splitting the last round of 256-row tiles, or nullptr
  int* tail_cuts;    // and the list of the tiles cut
  int any_height;    // the GEMMs' tiles need not be the plan's blocks
  bool tall;         // the buffers in `tail` hold tiles of 288 rows
  void* xq;          // fp8 layer only
  float* x_scale;
  void* actq;
  float* act_scale;
  int64_t total;
  TailScratch tail_scratch() const { return TailScratch{tail, tail_cuts, any_height, tail && tall}; }
};

// the activated intermediate is stored in half precision also on the fp8 path
int act_elem_size(int) { return 2; }

// tall: slice buffers for tiles of 288 rows; without them kTallTailBytes - tail_bytes (8.4 MB) less
Carve carve(void* base, int64_t M, int64_t H, int64_t F, int E, int topk, int dtype, const fr_moe_plan& p, bool tall = true) {
  Carve c;
  c.tall = tall;
  const int64_t n = M * topk;
  char* b = static_cast<char*>(base);
  int64_t off = 0;
  auto take = [&](int64_t bytes) { char* r = b ? b + off : nullptr; off += aligned(bytes); return r; };
  c.topk_w = reinterpret_cast<float*>(take(n * 4));
  c.topk_ids = reinterpret_cast<int32_t*>(take(n * 4));
  c.sorted = reinterpret_cast<int32_t*>(take(p.sorted_len * 4));
  c.expert_ids = reinterpret_cast<int32_t*>(take((n + E) * 4));
  c.npost = reinterpret_cast<int32_t*>(take(4));
  c.align_ws_bytes = fr_moe_align_workspace_bytes(n, E);
  c.align_ws = take(c.align_ws_bytes);
  c.act = take(p.sorted_len * F * act_elem_size(dtype));
  c.partial = reinterpret_cast<float*>(take(static_cast<int64_t>(p.split_k) * n * H * 4));
  c.tail = p.tail_bytes > 0 ? reinterpret_cast<float*>(take(tall && p.tail_bytes < kTallTailBytes ? kTallTailBytes : p.tail_bytes)) : nullptr;
  c.any_height = any_height(M, H, F, E, topk, dtype, p);
  c.tail_cuts = p.tail_bytes > 0 ? reinterpret_cast<int*>(take(kTailDescBytes)) : nullptr;
  c.xq = nullptr; c.x_scale = nullptr; c.actq = nullptr; c.act_scale = nullptr;
  if (dtype == FR_FP8_E4M3) {
    c.xq = take(M * H);
    c.x_scale = reinterpret_cast<float*>(take(M * 4));
    c.actq = take(p.sorted_len * F);
    c.act_scale = reinterpret_cast<float*>(take(p.sorted_len * 4));
  }
  c.total = off;
  return c;
}

int check_layer_shapes(const char* who, int64_t M, int64_t H, int64_t F, int E, int topk, int dtype) {
  FR_REQUIRE(dtype == FR_F16 || dtype == FR_BF16 || dtype == FR_FP8_E4M3, FR_E_DTYPE, "%s: dtype %d not in {f16, bf16, fp8_e4m3}", who, dtype);
  FR_REQUIRE(M >= 0 && H > 0 && F > 0, FR_E_SHAPE, "%s: M=%lld H=%lld F=%lld", who, (long long)M, (long long)H, (long long)F);
  FR_REQUIRE(E >= 1 && E <= 1024 && topk >= 1 && topk <= E, FR_E_SHAPE, "%s: E=%d topk=%d", who, E, topk);
  const int mult = dtype == FR_FP8_E4M3 ? 256 : 128;
  FR_REQUIRE(H % mult == 0 && F % mult == 0, FR_E_SHAPE, "%s: H=%lld and F=%lld must be multiples of %d", who, (long long)H, (long long)F, mult);
  FR_REQUIRE(M * topk < (int64_t(1) << 30), FR_E_SHAPE, "%s: M*topk too large", who);
  return FR_OK;
}

}  // namespace
const fr_moe_tunables& tunables() { return g_tunables; }

int plan_leaves_heights(int64_t M, int64_t H, int64_t F, int E, int topk, int dtype, int block) {
  const int mult = dtype == FR_FP8_E4M3 ? 256 : 128;
  if ((block != 128 && block != 160) || H % mult || F % mult || E > 1022 || topk > E) return kHeightsOfBlock;  // shapes without a plan among them
  fr_moe_plan p;
  return fr_moe_get_plan(M, H, F, E, topk, dtype, &p) == FR_OK && p.block == block ? any_height(M, H, F, E, topk, dtype, p) : kHeightsOfBlock;
}
}  // namespace fr

using namespace fr;

extern "C" int fr_moe_set_tunables(const fr_moe_tunables* t) {
  if (!t) {
    g_tunables = fr_moe_tunables{0, 0, 0, 0, 0, 0};
    return FR_OK;
  }
  FR_REQUIRE(t->block == 0 || t->block == 16 || t->block == 32 || t->block == 64 || t->block == 128 || t->block == 160 || t->block == 256,
             FR_E_SHAPE, "fr_moe_set_tunables: block=%d not in {0, 16, 32, 64, 128, 160, 256}", t->block);
  FR_REQUIRE(t->split_k >= 0 && t->split_k <= 64, FR_E_SHAPE, "fr_moe_set_tunables: split_k=%d outside [0, 64]", t->split_k);
  FR_REQUIRE(t->group_m >= 0 && t->group_m <= 64, FR_E_SHAPE, "fr_moe_set_tunables: group_m=%d outside [0, 64]", t->group_m);
  FR_REQUIRE(t->no_tail_split == 0 || t->no_tail_split == 1, FR_E_SHAPE, "fr_moe_set_tunables: no_tail_split=%d", t->no_tail_split);
  FR_REQUIRE(t->epilogue_combine == 0 || t->epilogue_combine == 1, FR_E_SHAPE, "fr_moe_set_tunables: epilogue_combine=%d", t->epilogue_combine);
  FR_REQUIRE(t->no_quad == 0 || t->no_quad == 1, FR_E_SHAPE, "fr_moe_set_tunables: no_quad=%d", t->no_quad);
  g_tunables = *t;
  return FR_OK;
}

extern "C" int fr_moe_get_tunables(fr_moe_tunables* t) {
  FR_REQUIRE(t, FR_E_NULL, "fr_moe_get_tunables: null pointer");
  *t = g_tunables;
  return FR_OK;
}

namespace fr {
namespace {
// the plan's routing block
int plan_block(int64_t M, int64_t H, int64_t F, int E, int topk, int dtype) {
  const int64_t n = M * topk;
  const double avg = static_cast<double>(n) / E;  // expected pairs per expert under uniform load
  // Routing block = token rows per GEMM tile.  Decode sizes want one block per expert
  // (weights are streamed once); from ~32 pairs per expert on, the 128-row MFMA tile
  // wins even with its padding, and 256 rows once runs are long enough to amortise it.
  // The 256-row tile's advantage grows with the K of the gate/up GEMM (its start-up per
  // tile is amortised over more K tiles); measured crossovers: 512..640 pairs per expert
  // at H = 4096 (F = 14336, E = 8: 2048 tokens 1380 us with 128 rows against 1435 with 256, 2560 tokens
  // 1810 against 1662).  At H = 2048 (F = 1408, E = 64, top-6: 32 and 22 K tiles per output tile) the 128-row
  // tile stays ahead as far as measured: 768 / 1536 pairs per expert 960 / 1738 us against 1002 / 1776.
  const double t256 = H >= 4096 ? 560.0 : (H <= 2048 ? 4096.0 : 4096.0 - (H - 2048) * (3536.0 / 2048.0));
  // Between 26 and 52 pairs per expert with a long gate/up K the 64-row tile wins: one block per expert
  // where 32-row blocks stream every expert's weights through the CUs twice, and half the MFMA and LDS work
  // of the 128-row tile (measured at H = 4096, F = 14336, E = 8: M = 112..192 4-6 % faster than either;
  // at H = 2048, F = 1408, E = 64 with skewed load it is slower than the 128-row tile, hence the K condition).
  int block;
  if (avg <= 8) block = 16;
  else if (avg < 26 || (avg < 32 && H < 4096)) block = 32;
  else if (avg < 52 && H >= 4096) block = 64;
  else if (avg < t256) block = 128;
  else block = 256;
  // 160-row blocks (a gate/up K of at least 32 K tiles): the same three-slot ring as the 128-row
  // tile with a quarter more rows per pass of an expert's weights through LDS.  Under uniform routing an expert
  // gets avg +- sqrt(avg) pairs, so with avg = 128, 256, 384, 512 every other expert needs one 128-row block more
  // than avg / 128; 160 rows absorb the spread.  Taken where the expected number of blocks per expert drops by an
  // eighth or more (1 / 1.15), or the expected rows the MFMAs multiply (whole half-blocks: a wavefront row is skipped when
  // all its rows are padding) by 2 %; measured on 8 experts, H = 4096, 128 / 160 / 256 rows:
  //   tokens  512  681 / 618         us      1536  1143 / 1112 / 1132       3072        1906 / 1939
  //           640  753 / 749                 1792  1236 / 1179 / 1192       4096        2433 / 2485
  //           768  715 / 743 (128 stays)     2048  1393 / 1386 / 1441       5120        2988 / 2975
  //           896  828 / 770                 2560  1706 / 1623 / 1685       6144        3507 / 3478
  //          1024  874 / 801                                                8192        4658 / 4512
  // With a 160-row candidate the 256-row tile takes over at 1200 pairs per expert (H >= 4096).  Below 112 pairs per expert one
  // block holds an expert either way and the smaller tile is cheaper (256 / 384 tokens: 548 / 556, 580 / 602 us);
  // with H = 1024 (16 K tiles) the 160-row tile loses (700 tokens: 85 / 96 us).
  // fp8 (16x16x128 MFMAs for this tile; its gate/up kernel spills 46 registers): only where a sixth of the blocks
  // go - 128 / 160 / 256 rows: 512 tokens 435 / 392, 1024: 543 / 505, 2560: 1145 / 1006 / 1063 us, but 2048: 853 / 877
  // / 899 - and below 900 pairs per expert (4096 tokens: 1506 against 1495 us with 256 rows).
  const bool two_byte = dtype == FR_BF16 || dtype == FR_F16;
  auto expected = [&](int rows) { return expected_blocks(avg, E, rows); };
  if ((block == 128 || block == 256) && H >= 2048 && F >= 1024 && E <= 1022 && avg >= 112 &&
      avg < (H >= 4096 ? (two_byte ? 1200.0 : 900.0) : t256)) {
    const double b128 = expected(128), b160 = expected(160);
    const double c128 = expected(64) * 64, c160 = expected(80) * 80;
    const bool take160 = two_byte ? (b160 * 1.15 < b128 || c160 <= 0.98 * c128) : b160 * 1.2 < b128;
    if (take160) block = 160;
  }
  // 256 rows, where both GEMMs run the one-wavefront-per-SIMD kernel (16 K tiles or more in both).  Its tiles follow the experts'
  // runs in units of 32 rows (moe_gemm_quad.h), so the block decides the padding of the routing arrays only; what is priced
  // here, the mean of whole and half blocks of 256 rows, bounds that padding.  Layer in us, 128 or 160 rows without that kernel
  // / 256: H = 4096, F = 14336, 8 experts 1536 tokens 1117 / 983, 1792 1222 / 1077, 2048 1422 / 1184, 2560 1657 / 1547, 3000
  // 1878 / 1694; fp8 1280 596 / 558, 1600 707 / 607, 2048 848 / 694, 2400 916 / 902; H = 2048, F = 1408, 64 experts, top-6,
  // Zipf-skewed 7468 0.96, 8192 0.99, 10000 0.94.  Layers that keep smaller blocks by this rule may run that kernel, too
  // (any_height); what it costs with one or two experts and F up to 4096 is that of few tiles (400 tokens, one expert 1.19).
  if (!g_tunables.no_quad && (block == 128 || block == 160) && H >= 2048 && F >= 2048 / (two_byte ? 2 : 1) && E <= 1022 &&
      avg >= (H >= 4096 ? (two_byte ? 350.0 : 300.0) : 700.0)) {
    const double other = expected(block) * block;
    const double quad = 0.5 * (expected(256) * 256 + expected(128) * 128);
    if (quad <= (two_byte ? 1.08 : 1.18) * other) block = 256;
  }
  if (g_tunables.block) block = g_tunables.block;
  // the fp8 160-row tile exists in the persistent form only (five K tiles per K slice at least, 1022 experts at most)
  if (block == 160 && !two_byte && (H < 640 || F < 1024 || E > 1022)) block = 128;
  return block;
}

// The plan for that block: K slices of the down projection, scratch.
fr_moe_plan plan_for(int64_t M, int64_t H, int64_t F, int E, int topk, int dtype, int block) {
  const int64_t n = M * topk;
  const double avg = static_cast<double>(n) / E;
  auto expected = [&](int rows) { return expected_blocks(avg, E, rows); };
  // Down projection: N = H gives few feature tiles, so K is split.
  const int bf = block == 16 ? 64 : (block == 32 ? 128 : 256);
  // expected token blocks: one per pair or per expert in the decode regime, else the expected blocks per expert
  const int64_t blocks = n <= E ? n : (block >= 128 ? static_cast<int64_t>(E * expected(block) + 0.5) : E);
  const int64_t tiles = blocks * ceil_div(H, bf);
  const int bk_elems = dtype == FR_FP8_E4M3 ? (block <= 32 ? 256 : 128) : (block == 16 ? 128 : 64);
  // 256-row tiles of 2-byte operands with a long K balance their last round themselves (its
  // tiles are cut along K over the idle workgroups); both GEMMs share the scratch for that.
  const int64_t tail_up = tail_scratch_bytes(block, dtype, H, F, true), tail_down = tail_scratch_bytes(block, dtype, F, H, false);
  int split = 1;
  if (tail_down > 0 && (tiles >= 192 || tiles <= 64)) {
    // whole rounds plus a split last round, or so few tiles that every one is cut into 4..8 slices;
    // in between (most of one round: no idle workgroups to cut for) all tiles are split alike
  } else if (block >= 128) {
    // one workgroup per CU: the split that minimises GEMM time (at ~0.9 PFLOP/s, stretched by how long the
    // busiest workgroup works: the persistent launch gives each of `sp` slices 256 / sp workgroups, rounded down
    // to whole XCD shares, and a workgroup does ceil(tiles / those) units of 1 / sp of a tile) plus the partial
    // traffic it causes (one 2-byte slice, or `split` fp32 slices, written and read back at ~4 TB/s: with many
    // pairs per weight byte that traffic decides).  Measured on 8 experts with one block each (128 tiles), down
    // projection with 1 / 2 / 3 / 4 slices: 384 tokens 185 / 174 / 212 / 196 us, 512 tokens 202 / 194 / 233 / 214.
    double best = 1e30;
    const double rows = static_cast<double>(blocks) * block, pairs = static_cast<double>(n);
    for (int sp = 1; sp <= 4; ++sp) {
      if (F / sp < 8 * bk_elems) break;
      const int64_t wgs = 256 / sp / 8 * 8;
      const double busiest = static_cast<double>(ceil_div(tiles, wgs)) / sp;  // in tiles
      const double fill = (static_cast<double>(tiles) / 256.0) / busiest;
      const double t_gemm = 2.0 * rows * H * F / 0.9e15 / (fill < 1.0 ? fill : 1.0);
      const double t_part = pairs * H * (sp == 1 ? 2.0 : 4.0 * sp) * 2.0 / 4e12;
      if (t_gemm + t_part < best) { best = t_gemm + t_part; split = sp; }
    }
  } else {
    // several workgroups per CU: aim at ~512 workgroups
    // (the 64-row tile runs one workgroup per CU: ~256)
    const int64_t target = block == 64 ? 256 : 512;
    while (split < 16 && tiles * split * 2 <= target && F / (split * 2) >= 8 * bk_elems) split *= 2;
    // between half a pair and one pair per expert: collisions are common (some experts get two rows,
    // some none) and the grid is partly filled by tiles of unequal luck; four slices even that out
    // (measured at 3 and 4 tokens on 8 experts, top-2: -9 % and -13 % on the down projection; with
    // fewer pairs the blocks are as many as the pairs and the rule above already fills the grid)
    if (n <= E && 2 * n > E && tiles <= 512)
      while (split < 4 && F / (split * 2) >= 8 * bk_elems) split *= 2;
  }
  int64_t tail_bytes = tail_up > tail_down ? tail_up : tail_down;
  if (g_tunables.split_k) {  // as many slices as asked for, as far as every slice keeps 8 K tiles
    split = g_tunables.split_k;
    while (split > 1 && F / split < 8 * bk_elems) --split;
  }
  if (g_tunables.no_tail_split) tail_bytes = 0;
  fr_moe_plan plan;
  plan.block = block;
  plan.split_k = split;
  plan.sorted_len = n + static_cast<int64_t>(E) * (block - 1);
  plan.tail_bytes = tail_bytes;
  plan.workspace_bytes = carve(nullptr, M, H, F, E, topk, dtype, plan).total;
  return plan;
}

// The layers route for another block than the plan's where that has been found faster (2-byte operands; a block set by hand
// stands).  Never for fewer K slices that are summed from fp32 rows: a single slice's rows are rounded.  Only sizes are known here, so every
// range holds for near-uniform as well as Zipf-skewed loads.  Layer in parts of the time with the plan's block, near-uniform / Zipf (two
// routings):
//   Many narrow experts (shapes: H, F, experts, top-k).  The heavy experts of a skewed load take several small tiles.  Up to 128 experts
//   and F = 2816: the routing blocks' padding is E x block rows of F activated values.
//     plan 16, 32 rows from 2 pairs per expert, where gate/up rows are short enough for the narrow 32-row tile (moe_gemm_tiles.h):
//       2048, 1408, 64, 6   2 pairs 1.00 / 0.98, 3 0.99 / 0.96, 6 1.01 / 0.88, 8 1.01 / 0.905, but 1.1 1.01 / 1.02
//       2048, 768, 128, 8   2 1.01 / 0.97, 4 1.00 / 0.96, 8 1.00 / 0.85;   2048, 1024, 60, 4   2 0.99 / 0.98, 3 1.03 / 1.01, 5 1.02 / 0.93, 8 0.995 / 0.90
//       2048, 1408, 32, 2   3 1.00 / 0.95, 6 1.00 / 0.98;   2048, 2048, 64, 6   3 0.97 / 0.88, 8 0.96 / 0.88
//       2048, 2816, 64, 6   3 1.06 / 0.965;   2560, 1536, 64, 8   3 1.03 / 0.98;   3072, 1536, 32, 4   2 1.01 / 1.055, 6 1.01 / 1.05
//     64 rows instead of 32 from 12 pairs:
//       2048, 1408, 64, 6   12 1.015 / 0.94, 16 1.01 / 0.87, 20 1.00 / 0.83, 27 0.89 / 0.805;   2048, 768, 128, 8   12 1.01 / 0.89, 20 1.00 / 0.82
//       2048, 1024, 60, 4   8.5 0.95 / 1.07, 12 0.95 / 0.99, 20 0.95 / 0.84;   2048, 1408, 32, 2   12 1.02 / 0.875, 16 1.02 / 0.985, 24 0.92 / 0.86
//       3072, 1536, 32, 4   8.5 1.02 / 1.07, 12 1.015 / 1.015, 16 0.995 / 0.89;   2560, 1536, 64, 8   12 1.02 / 0.93;   3072, 1024, 96, 4   12 1.00 / 0.84
//       2048, 2816, 64, 6   12 1.02 / 0.875;   3072, 2816, 100, 8   12 1.00 / 0.88
//       2048, 1024, 128, 8   12 0.98 / 0.91;   3584, 640, 64, 6   12 0.97 / 0.83
//     but from 24 pairs where w2 has short rows, or rows of a power of two of 4 KB or more, whose 32-row tiles start K at spread places and 64-row
//     ones do not:   2048, 512, 128, 8   12 1.08 / 1.01, 18 1.08 / 0.88, 26 0.97 / 0.81;   2048, 256, 64, 6   12 1.145 / 1.20, 26 1.00 / 0.99, 128 rows 28.5 1.08 / 1.07
//       2048, 2048, 64, 6   12 1.12 / 0.96, 20 1.11 / 0.89, 24 1.04 / 0.81, 27 0.98 / 0.85
//     128 rows from 28 pairs (64 rows): 2048, 1408, 64, 6 28.5 0.89 / 0.78 (0.83 / 0.83); 3072, 1024, 96, 4 0.90 / 0.62 (0.87 / 0.71)
//   H = 640 to 1024, up to 16 experts: the plan's 64-row range begins at H = 4096, and the 128-row tile has up to 16 short K tiles there.
//   t = gate/up tiles with one block per expert.
//     plan 32, 64 rows where t is most of a round and leaves room for an expert's second block, H = 1024:
//       F = 3584, 8 experts (t = 224) 8.5 0.915 / 0.91, 12 0.925 / 0.91, 20 0.90 / 0.94, 30 0.815 / 0.91;   F = 1536, 16 experts (192) 12 0.905 / 0.91, 30 0.89 / 0.895
//       F = 7168, 4 (224) 12 0.91 / 0.91, 30 0.84 / 0.82;   F = 14336, 2 (224) 12 0.98, 30 0.90;   F = 4096, 8 (256) 12 0.93 / 0.84, 20 0.92 / 1.07
//       F = 2048, 8 (128) 12 1.05 / 0.95;   H = 768, F = 2048, 16 (256) 1.05 / 1.04;   H = 896, F = 5120, 6 (240) 1.12 / 1.125;   t = 22 to 80 1.2 to 1.3
//     plan 32, 16 rows up to 10 pairs from a whole round on: F = 4096, 8 experts (256) 10 0.965 / 0.94, H = 768, F = 2048, 16 (256) 0.905 / 0.945, F = 3072, 16
//       (384) 0.91 / 0.96, F = 14336, 8 (896) 0.91 / 0.95;   but F = 2048, 8 (128) 0.955 / 1.02, H = 768, F = 3584, 8 (224) 0.925 / 1.12
//     plan 128, 64 rows up to 48 pairs: F = 3584, 8 40 0.74 / 0.97, F = 14336, 8 0.86 / 0.92, H = 768, F = 3072, 16 0.79 / 0.76, F = 1024, 16 (128; two K slices)
//       0.89 / 0.92;   but F = 1536, 16 (192; three K slices) 0.89 / 1.04, 48 0.89 / 1.12
//     up to 90 pairs (t above 128: 104) with t up to 224 and one K slice: F = 3584, 8 64 1.00 / 0.80, 80 0.96 / 0.765, 100 0.95 / 0.75, F = 7168, 4 1.01 / 0.95, 0.89 / 0.76, F = 2048, 8 0.84 / 0.85, 0.74 / 0.77;
//       but t = 256 F = 4096, 8 80 1.05 / 0.895, H = 768, F = 2048, 16 1.025 / 0.875;   F = 2048, 8 100 0.74 / 1.09
//     up to 125 pairs with t up to 80: F = 4096, 2 0.62, F = 2816, 1 0.63, F = 1024, 8 0.90 / 0.91, H = 640, F = 2560, 4 0.74 / 0.74
//   160 rows instead of 128 where an expert is likely to exceed 128 rows: a block more costs a round of tiles, the larger tile 1 %.
//     16 experts, F = 8192, fp16: 920 tokens (115 pairs) 0.895 / 1.005, 800 (100; no expert above 128) 0.99; H = 6144, F = 16384 460 0.87 / 1.045; H = 4096,
//     F = 14336, 8 experts 460 0.955 / 1.005, none above 128: 300 and 420 1.01; 16 experts, F = 1536, top-4 460 0.86 / 0.955; 4 experts, F = 2048 230 0.985 / 1.045
int layer_block(int64_t M, int64_t H, int64_t F, int E, int topk, int dtype, const fr_moe_plan& p) {
  if ((dtype != FR_F16 && dtype != FR_BF16) || g_tunables.block) return p.block;
  const double avg = static_cast<double>(M) * topk / E;
  if (E >= 32 && E <= 128 && H >= 2048 && H < 4096 && F <= 2816 && p.block <= 32) {
    if (F >= 512 && avg >= 28) return 128;
    if (F >= 512 && avg >= (F < 640 || (F > 1024 && (F & (F - 1)) == 0) ? 24 : 12)) return 64;
    return avg >= 2 && H <= 2048 && F <= 2048 ? 32 : p.block;
  }
  if (E <= 16 && H >= 640 && H <= 1024 && F >= 1024) {
    const int64_t t = E * ceil_div(F, 128);
    if (p.block == 32) return H > 896 && t >= 192 && t <= 240 ? 64 : t >= 256 && avg <= 10 ? 16 : 32;
    if (p.block == 128 && ((avg <= 48 && (p.split_k == 1 || t <= 128)) || (avg <= (t > 128 ? 104 : 90) && p.split_k == 1 && t <= 224) || (avg < 126 && t <= 80))) return 64;
  }
  if (E <= 16 && H >= 4096 && F >= 1024 && p.block == 128 && avg < 128 && E * (expected_blocks(avg, E, 128) - 1.0) >= 0.15) return 160;
  return p.block;
}
// `p`: the plan.  A block taken where the plan cuts no last round cuts none either (at 28 to 32 pairs per expert, 128 rows for 32, the layer is
// 1 % faster for it and the scratch 64 MiB smaller), and a block whose scratch is more than fr_fused_moe_noalloc has is not taken
// where the plan's is not: the same sizes run the same kernels there.
fr_moe_plan layer_plan(int64_t M, int64_t H, int64_t F, int E, int topk, int dtype, const fr_moe_plan& p) {
  const int block = layer_block(M, H, F, E, topk, dtype, p);
  if (block == p.block) return p;
  fr_moe_plan q = plan_for(M, H, F, E, topk, dtype, block);
  if (p.tail_bytes == 0) q.tail_bytes = 0;
  q.workspace_bytes = carve(nullptr, M, H, F, E, topk, dtype, q).total;
  if (q.workspace_bytes > kStaticScratchBytes && carve(nullptr, M, H, F, E, topk, dtype, p).total <= kStaticScratchBytes) return p;
  return p.split_k > 1 && q.split_k == 1 ? p : q;
}

// The blocks, slices and buffers of a layer call in the workspace it was given (p: fr_moe_get_plan's result, whose bytes hold all of
// them).  A smaller workspace, as a caller may have kept it for these sizes, is enough while it holds the plan's own block with slice
// buffers of 256 rows: the call then does without what does not fit.
int layer_carve(const char* who, int64_t M, int64_t H, int64_t F, int E, int topk, int dtype, fr_moe_plan& p, void* workspace, int64_t bytes,
                Carve& c) {
  FR_REQUIRE(workspace, FR_E_WORKSPACE, "%s: no workspace (%lld bytes needed)", who, (long long)p.workspace_bytes);
  bool tall = true;
  fr_moe_plan q = layer_plan(M, H, F, E, topk, dtype, p);
  if (bytes < p.workspace_bytes) {
    const int64_t least = carve(nullptr, M, H, F, E, topk, dtype, p, false).total;
    FR_REQUIRE(bytes >= least, FR_E_WORKSPACE, "%s: workspace %lld < %lld bytes", who, (long long)bytes, (long long)least);
    if (carve(nullptr, M, H, F, E, topk, dtype, q, false).total > bytes) q = p;
    tall = carve(nullptr, M, H, F, E, topk, dtype, q).total <= bytes;
  }
  FR_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255u) == 0, FR_E_ALIGN, "%s: workspace must be 256-byte aligned", who);
  p = q;
  c = carve(workspace, M, H, F, E, topk, dtype, p, tall);
  return FR_OK;
}
}  // namespace
}  // namespace fr

extern "C" int fr_moe_get_plan(int64_t M, int64_t H, int64_t F, int E, int topk, int dtype, fr_moe_plan* plan) {
  FR_REQUIRE(plan, FR_E_NULL, "fr_moe_get_plan: null plan");
  dtype &= ~FR_W_TILED;  // the plan does not depend on the weight layout
  int rc = check_layer_shapes("fr_moe_get_plan", M, H, F, E, topk, dtype);
  if (rc != FR_OK) return rc;
  *plan = plan_for(M, H, F, E, topk, dtype, plan_block(M, H, F, E, topk, dtype));
  const int64_t layer_bytes = layer_plan(M, H, F, E, topk, dtype, *plan).workspace_bytes;
  if (layer_bytes > plan->workspace_bytes) plan->workspace_bytes = layer_bytes;
  return FR_OK;
}

extern "C" int fr_moe_get_layer_plan(int64_t M, int64_t H, int64_t F, int E, int topk, int dtype, fr_moe_plan* plan) {
  int rc = fr_moe_get_plan(M, H, F, E, topk, dtype, plan);
  if (rc != FR_OK) return rc;
  const int64_t bytes = plan->workspace_bytes;
  *plan = layer_plan(M, H, F, E, topk, dtype & ~FR_W_TILED, *plan);
  plan->workspace_bytes = bytes;
  if (plan->tail_bytes > 0) plan->tail_bytes = kTallTailBytes + kTailDescBytes;
  return FR_OK;
}

namespace fr {
namespace {
// top-k gating of the logits and the routing arrays of the result: one launch for small
// batches, gating then align otherwise.  qx (fp8 layer): the bf16 token rows [M, H], quantised per row into
// c.xq / c.x_scale - by the same launch for small batches, by one of its own otherwise.
int route_and_align(const void* logits, int logits_dtype, int64_t M, int E, int topk, int renormalize, int block,
                    const Carve& c, const void* qx, int64_t H, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (route_align_fits(M, E, topk, qx != nullptr))
    return route_align_small(logits, logits_dtype, M, E, topk, renormalize, block, c.topk_w, c.topk_ids, c.sorted,
                             c.expert_ids, c.npost, qx, H, c.xq, c.x_scale, st);
  int rc = fr_gating_topk(logits, logits_dtype, M, E, E, topk, renormalize, c.topk_w, c.topk_ids, stream);
  if (rc != FR_OK) return rc;
  rc = fr_moe_align(c.topk_ids, FR_I32, M * topk, E, block, c.sorted, c.expert_ids, c.npost, c.align_ws, c.align_ws_bytes, stream);
  if (rc != FR_OK || !qx) return rc;
  return quant_rows(qx, FR_BF16, M, RowFilter{}, H, H, c.xq, c.x_scale, st);
}
}  // namespace
}  // namespace fr

extern "C" int fr_fused_experts(const void* x, const void* w1, const void* w2, const float* topk_weights,
                                const int32_t* topk_ids, int64_t M, int64_t H, int64_t F, int E, int topk,
                                int dtype, void* out, void* workspace, int64_t workspace_bytes, void* stream) {
  fr_moe_plan p;
  int rc = fr_moe_get_plan(M, H, F, E, topk, dtype, &p);
  if (rc != FR_OK) return rc;
  if (M == 0) return FR_OK;
  FR_REQUIRE(x && w1 && w2 && topk_weights && topk_ids && out, FR_E_NULL, "fr_fused_experts: null pointer");
  Carve c;
  rc = layer_carve("fr_fused_experts", M, H, F, E, topk, dtype & ~FR_W_TILED, p, workspace, workspace_bytes, c);
  if (rc != FR_OK) return rc;
  rc = fr_moe_align(topk_ids, FR_I32, M * topk, E, p.block, c.sorted, c.expert_ids, c.npost, c.align_ws, c.align_ws_bytes, stream);
  if (rc != FR_OK) return rc;
  rc = gateup_impl(x, nullptr, w1, nullptr, c.sorted, c.expert_ids, c.npost, M, H, F, E, topk, p.block, dtype & ~FR_W_TILED, c.act, c.tail_scratch(),
                   static_cast<hipStream_t>(stream), "fr_fused_experts", (dtype & FR_W1_TILED) ? 1 : 0);
  if (rc != FR_OK) return rc;
  return down_impl(c.act, nullptr, w2, nullptr, topk_weights, c.sorted, c.expert_ids, c.npost, M, H, F, E, topk, p.block,
                   p.split_k, dtype & ~FR_W_TILED, dtype & ~FR_W_TILED, c.partial, out, c.tail_scratch(), static_cast<hipStream_t>(stream),
                   "fr_fused_experts", (dtype & FR_W2_TILED) ? 1 : 0, topk_ids);
}

namespace fr {
namespace {
// p: fr_moe_get_plan's result
int fused_moe_run(fr_moe_plan p, const void* x, const void* w1, const void* w2, const void* logits, int logits_dtype,
                  int64_t M, int64_t H, int64_t F, int E, int topk, int renormalize, int dtype, void* out, void* workspace,
                  int64_t workspace_bytes, void* stream) {
  int rc;
  FR_REQUIRE(x && w1 && w2 && logits && out, FR_E_NULL, "fr_fused_moe: null pointer");
  Carve c;
  rc = layer_carve("fr_fused_moe", M, H, F, E, topk, dtype & ~FR_W_TILED, p, workspace, workspace_bytes, c);
  if (rc != FR_OK) return rc;
  // a handful of tokens: the gate/up launch gates and sorts by itself (row-major weights only)
  rc = (dtype & FR_W1_TILED) ? 1
                            : gateup_rows_routed(x, w1, logits, logits_dtype, M, H, F, E, topk, renormalize, p.block, dtype, c.act, c.topk_w,
                                                 c.topk_ids, c.sorted, c.expert_ids, c.npost, static_cast<hipStream_t>(stream));
  if (rc < 0) return rc;
  if (rc == 1) {
    rc = route_and_align(logits, logits_dtype, M, E, topk, renormalize, p.block, c, nullptr, H, stream);
    if (rc != FR_OK) return rc;
    rc = gateup_impl(x, nullptr, w1, nullptr, c.sorted, c.expert_ids, c.npost, M, H, F, E, topk, p.block, dtype & ~FR_W_TILED, c.act, c.tail_scratch(),
                   static_cast<hipStream_t>(stream), "fr_fused_moe", (dtype & FR_W1_TILED) ? 1 : 0);
    if (rc != FR_OK) return rc;
  }
  return down_impl(c.act, nullptr, w2, nullptr, c.topk_w, c.sorted, c.expert_ids, c.npost, M, H, F, E, topk, p.block,
                   p.split_k, dtype & ~FR_W_TILED, dtype & ~FR_W_TILED, c.partial, out, c.tail_scratch(), static_cast<hipStream_t>(stream),
                   "fr_fused_moe", (dtype & FR_W2_TILED) ? 1 : 0, c.topk_ids);
}
}  // namespace
}  // namespace fr

extern "C" int fr_fused_moe(const void* x, const void* w1, const void* w2, const void* logits, int logits_dtype,
                            int64_t M, int64_t H, int64_t F, int E, int topk, int renormalize, int dtype,
                            void* out, void* workspace, int64_t workspace_bytes, void* stream) {
  fr_moe_plan p;
  int rc = fr_moe_get_plan(M, H, F, E, topk, dtype, &p);
  if (rc != FR_OK) return rc;
  if (M == 0) return FR_OK;
  return fused_moe_run(p, x, w1, w2, logits, logits_dtype, M, H, F, E, topk, renormalize, dtype, out, workspace, workspace_bytes, stream);
}

extern "C" int fr_fused_moe_fp8(const void* x, int x_dtype, const void* w1q, const float* w1_scale, const void* w2q,
                                const float* w2_scale, const void* logits, int logits_dtype, int64_t M, int64_t H,
                                int64_t F, int E, int topk, int renormalize, void* out, void* workspace,
                                int64_t workspace_bytes, void* stream) {
  fr_moe_plan p;
  int rc = fr_moe_get_plan(M, H, F, E, topk, FR_FP8_E4M3, &p);
  if (rc != FR_OK) return rc;
  if (M == 0) return FR_OK;
  const int w2_flag = x_dtype & FR_W2_TILED;
  x_dtype &= ~FR_W_TILED;
  FR_REQUIRE(x_dtype == FR_BF16, FR_E_DTYPE, "fr_fused_moe_fp8: activations must be bf16 (dtype %d)", x_dtype);
  FR_REQUIRE(x && w1q && w1_scale && w2q && w2_scale && logits && out, FR_E_NULL, "fr_fused_moe_fp8: null pointer");
  hipStream_t st = static_cast<hipStream_t>(stream);
  Carve c;
  rc = layer_carve("fr_fused_moe_fp8", M, H, F, E, topk, FR_FP8_E4M3, p, workspace, workspace_bytes, c);
  if (rc != FR_OK) return rc;
  rc = route_and_align(logits, logits_dtype, M, E, topk, renormalize, p.block, c, x, H, stream);
  if (rc != FR_OK) return rc;
  // the eight-wavefront kernels' gate/up GEMM does not cut its last round in fp8
  rc = gateup_impl(c.xq, c.x_scale, w1q, w1_scale, c.sorted, c.expert_ids, c.npost, M, H, F, E, topk, p.block, FR_FP8_E4M3, c.act,
                   p.block == 256 || c.any_height ? c.tail_scratch() : TailScratch{}, st, "fr_fused_moe_fp8", 0);
  if (rc != FR_OK) return rc;
  // only slots that hold a pair: nothing of a padding slot's row is used by the down projection
  rc = quant_rows(c.act, FR_BF16, p.sorted_len, RowFilter{c.npost, c.sorted, M * topk}, F, F, c.actq, c.act_scale, st);
  if (rc != FR_OK) return rc;
  return down_impl(c.actq, c.act_scale, w2q, w2_scale, c.topk_w, c.sorted, c.expert_ids, c.npost, M, H, F, E, topk, p.block,
                   p.split_k, FR_FP8_E4M3, x_dtype, c.partial, out, c.tail_scratch(), st, "fr_fused_moe_fp8", w2_flag ? 1 : 0, nullptr);
}

// ---- one entry point that allocates nothing ------------------------------------
// The layer's scratch lives in a device array of this library instead of a caller's buffer.
// Host code may not pass the array's name to a kernel (on the host it is a stand-in, not a
// device address): its address on the current device is looked up once per device and kept.
namespace fr {
namespace {
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

int static_scratch(void** out) {
  constexpr int kMaxDevices = 64;
  static void* ptrs[kMaxDevices] = {};  // per device; two threads racing here store the same address
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) return fail(FR_E_NO_DEVICE, "fr_fused_moe_noalloc: device %d (%s)", dev, hipGetErrorString(e));
  if (!ptrs[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      (void)hipGetLastError();
      return fail(FR_E_NO_DEVICE, "fr_fused_moe_noalloc: hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
    }
    ptrs[dev] = p;
  }
  *out = ptrs[dev];
  return FR_OK;
}
}  // namespace
int prepare_static_scratch() {
  void* p = nullptr;
  return static_scratch(&p);
}
}  // namespace fr

extern "C" int fr_fused_moe_noalloc(const void* x, const void* w1, const void* w2, const void* logits, int logits_dtype,
                                    int64_t M, int64_t H, int64_t F, int E, int topk, int renormalize, int dtype,
                                    void* out, void* stream) {
  fr_moe_plan p;
  int rc = fr_moe_get_plan(M, H, F, E, topk, dtype, &p);
  if (rc != FR_OK) return rc;
  FR_REQUIRE((dtype & ~FR_W_TILED) == FR_F16 || (dtype & ~FR_W_TILED) == FR_BF16, FR_E_DTYPE, "fr_fused_moe_noalloc: dtype %d not in {f16, bf16}", dtype);
  const int64_t own_bytes = plan_for(M, H, F, E, topk, dtype & ~FR_W_TILED, p.block).workspace_bytes;  // where they fit, the layer's do (layer_plan)
  FR_REQUIRE(own_bytes <= kStaticScratchBytes, FR_E_WORKSPACE,
             "fr_fused_moe_noalloc: these sizes need %lld bytes of scratch, the library's static scratch holds %lld; use fr_fused_moe with a workspace",
             (long long)own_bytes, (long long)kStaticScratchBytes);
  if (M == 0) return FR_OK;
  void* ws = nullptr;
  rc = static_scratch(&ws);
  if (rc != FR_OK) return rc;
  return fused_moe_run(p, x, w1, w2, logits, logits_dtype, M, H, F, E, topk, renormalize, dtype, out, ws, kStaticScratchBytes, stream);
}
