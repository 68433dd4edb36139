// Block-aligned stable counting sort of (expert, token) pairs on gfx950.
//
// The n flat pairs are cut into segments of seg_len consecutive pairs, one
// wavefront per segment.  (1) every wavefront builds an LDS histogram of its
// segment; (2) an exclusive scan over segments gives each (expert, segment) its
// offset inside the expert's run, and an exclusive scan over the padded expert
// totals gives each run its start; (3) every wavefront walks its segment again
// 64 pairs at a time and ranks the pairs of one expert among themselves with
// wavefront ballots, so flat order survives inside each expert: the result is
// the stable sort.  Small inputs run all three phases in one workgroup with the
// tables in LDS; large ones take two launches, between which only the sums of every count
// workgroup go through memory (count, scatter + block table), or, with many experts, three
// on a table of every segment's counts (count, per-expert segment scan, scatter + block table).
#include "gating_core.h"
#include "quant_core.h"

namespace fr {
namespace {

constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / kWave;
constexpr int kSmallMaxE = 256;
// One workgroup sorts up to this many pairs.  As kernels two launches are the faster form from about 4000 pairs on (replayed from a graph,
// Zipf-skewed, one workgroup / two launches, us: 8 experts 4096 pairs 6.0 / 6.4, 5120 6.9 / 6.4, 6144 7.8 / 6.5; 64 experts 3072 5.75 / 6.2, 4096 6.6 / 6.6, 5120
// 7.7 / 6.6, 6144 8.6 / 6.6; 256 experts 2048 6.9 / 7.2, 3072 7.8 / 7.3, 6144 10.8 / 8.0).  But a program that calls moe_align_block_size by itself waits for the
// host side of the call, to which a second launch adds 2.5 us and more: 64 experts, 4200 / 6144 pairs 8.9 and 8.9 us with one, 11.7 and 11.7 with
// two among other calls, 21.7 and 22.5 against 23.1 and 23.2 alone; with topk_softmax in front 14.6 and 14.5 against 17.5 and 17.6.  The layers, whose
// GEMMs hide their host side, take the same line, at a cost of up to 2 us, 3 to 5 with 256 experts (H = 2048, F = 1408, 64 experts, 4200 pairs 234.0 / 232.6,
// 6144 240.7 / 236.7; H = 1024, F = 512, 256 experts, 4800 181.1 / 177.7; H = 1024, F = 3584, 8 experts, 5200 153.5 / 154.2, 6144 164.1 / 162.4).
constexpr int64_t kSmallMaxN = 6144;
// Gating and sort in ONE launch up to this many pairs (above, the gating kernel spread over the CUs plus the
// one-workgroup sort win: 2048 pairs 31.6 against 29.5 us for a small layer, 1536 pairs on 64 experts 51.8 against 26.5)
constexpr int64_t kRouteAlignMaxN = 1024;
constexpr int kMaxE = 1024;
constexpr int kSegThreads = 256;
constexpr int kSegWaves = kSegThreads / kWave;

__device__ __forceinline__ int64_t min64(int64_t a, int64_t b) { return a < b ? a : b; }

__host__ __device__ inline int bits_for(int E) {
  int b = 0;
  while ((1 << b) < E) ++b;
  return b;
}

// lanes (among `valid` ones) holding the same expert as this lane
__device__ __forceinline__ unsigned long long same_expert_lanes(int e, bool valid, int nbits) {
  unsigned long long m = __ballot(valid);
  for (int b = 0; b < nbits; ++b) {
    const bool bit = (e >> b) & 1;
    const unsigned long long vote = __ballot(bit);
    m &= bit ? vote : ~vote;
  }
  return m;
}

__device__ __forceinline__ int wave_inclusive_scan(int v) {
  // inside the rows of 16 lanes (row_shr), then each row's last value into the rows behind it (row_bcast): eight vector
  // instructions where six __shfl_up steps are six LDS round trips one behind the other
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);
  return v;
}

template <typename IdT>
__device__ __forceinline__ void segment_histogram(const IdT* __restrict__ ids, int64_t lo, int64_t hi,
                                                  int E, int lane, int* hist) {
  for (int64_t p = lo + lane; p < hi; p += kWave) {
    const int e = static_cast<int>(ids[p]);
    if (e >= 0 && e < E) atomicAdd(&hist[e], 1);
  }
}

// Walk [lo, hi) in flat order; cnt[e] holds the next free slot of expert e for
// this wavefront and is advanced as pairs are placed.
constexpr int kScatterPF = 4;  // rounds of 64 pairs whose ids are fetched together: the rounds themselves depend on
                               // one another through cnt[], their loads need not wait for that chain
template <typename IdT>
__device__ __forceinline__ void segment_ids(const IdT* __restrict__ ids, int64_t base0, int64_t hi, int lane, int (&ev)[kScatterPF]) {
#pragma unroll
  for (int r = 0; r < kScatterPF; ++r) {
    const int64_t p = base0 + r * kWave + lane;
    ev[r] = (p < hi) ? static_cast<int>(ids[p]) : -1;
  }
}
// Histogram of [lo, hi); `first` holds the ids of its first kScatterPF rounds (segment_ids), -1 behind hi: they are asked
// for together instead of each round waiting for its own.
template <typename IdT>
__device__ __forceinline__ void segment_histogram(const IdT* __restrict__ ids, int64_t lo, int64_t hi,
                                                  int E, int lane, int* hist, const int (&first)[kScatterPF]) {
#pragma unroll
  for (int r = 0; r < kScatterPF; ++r)
    if (first[r] >= 0 && first[r] < E) atomicAdd(&hist[first[r]], 1);
  segment_histogram(ids, lo + kScatterPF * kWave, hi, E, lane, hist);
}
// `first`: the ids of the first kScatterPF rounds, fetched by the caller ahead of time (segment_ids), or nullptr
template <typename IdT>
__device__ __forceinline__ void segment_scatter(const IdT* __restrict__ ids, int64_t lo, int64_t hi,
                                                int E, int nbits, int lane, volatile int* cnt,
                                                int32_t* __restrict__ sorted, const int* first = nullptr) {
  const unsigned long long below = (1ull << lane) - 1ull;
  for (int64_t base0 = lo; base0 < hi; base0 += kScatterPF * kWave) {
    int ev[kScatterPF];
    if (first != nullptr && base0 == lo) {
#pragma unroll
      for (int r = 0; r < kScatterPF; ++r) ev[r] = first[r];
    } else {
      segment_ids(ids, base0, hi, lane, ev);
    }
#pragma unroll
    for (int r = 0; r < kScatterPF; ++r) {
      const int64_t base = base0 + r * kWave;
      if (base >= hi) break;
      const int64_t p = base + lane;
      int e = ev[r];
      const bool valid = (p < hi) && e >= 0 && e < E;
      if (!valid) e = 0;
      const unsigned long long same = same_expert_lanes(e, valid, nbits);
      if (valid) {
        const int rank = __popcll(same & below);
        const int total = __popcll(same);
        const int old = cnt[e];
        sorted[old + rank] = static_cast<int32_t>(p);
        if (rank == total - 1) cnt[e] = old + total;
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// start[e] = exclusive scan of the padded totals, start[E] = padded length.
// Executed by one wavefront; total/start live in LDS.
__device__ __forceinline__ void scan_padded_totals(const int* total, int* start, int E, int B, int lane) {
  int running = 0;
  for (int base = 0; base < E; base += kWave) {
    const int e = base + lane;
    const int c = (e < E) ? (total[e] + B - 1) / B * B : 0;
    const int incl = wave_inclusive_scan(c);
    if (e < E) start[e] = running + incl - c;
    running += __builtin_amdgcn_readlane(incl, kWave - 1);
  }
  if (lane == 0) start[E] = running;
}

// ---------------------------------------------------------------- small path
// table[w][e]: pairs of expert e in segment w -> in the segments before w; total[e]: in all.  The counts are read before
// any of them is overwritten: the reads then do not wait for one another (16 LDS latencies, about a microsecond).
__device__ __forceinline__ void scan_segments(int* table, int* total, int E, int tid) {
  for (int e = tid; e < E; e += kSmallThreads) {
    int c[kSmallWaves];
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) c[w] = table[w * E + e];
    int running = 0;
#pragma unroll
    for (int w = 0; w < kSmallWaves; ++w) {
      table[w * E + e] = running;
      running += c[w];
    }
    total[e] = running;
  }
}

struct SmallTables {
  int table[kSmallWaves * kSmallMaxE];  // [segment][expert]: counts, then next free slots
  int total[kSmallMaxE];
  int first_block[kSmallMaxE + 1];  // of an expert's run; [E]: blocks in all
};
// The sort of one workgroup: the segment of each wavefront is [lo, hi), `first` its first ids (segment_ids), the table is
// zero and published.  A chain of dependent LDS steps that nothing runs beside, so it has few of them: up to 64 experts one
// wavefront turns counts into slots without a barrier (a lane per expert), a wavefront then places its pairs from its own row of the table and the block
// table and the padding are written behind that, by groups of lanes per expert instead of a search per block.
template <typename IdT>
__device__ __forceinline__ void small_sort(SmallTables& t, const IdT* ids, const int (&first)[kScatterPF], int64_t lo, int64_t hi,
                                           int64_t n, int E, int B, int64_t sorted_len, int tid, int32_t* __restrict__ sorted,
                                           int32_t* __restrict__ expert_ids, int32_t* __restrict__ npost_out) {
  const int lane = tid % kWave, wave = tid / kWave;
  int* mine = t.table + wave * E;
  segment_histogram(ids, lo, hi, E, lane, mine, first);
  __syncthreads();
  if (E <= kWave) {
    if (wave == 0) {
      int c[kSmallWaves], all = 0;
#pragma unroll
      for (int w = 0; w < kSmallWaves; ++w) c[w] = lane < E ? t.table[w * E + lane] : 0;
#pragma unroll
      for (int w = 0; w < kSmallWaves; ++w) all += c[w];
      const int blocks = static_cast<int>(static_cast<unsigned>(all + B - 1) / static_cast<unsigned>(B)), end = wave_inclusive_scan(blocks);
      if (lane < E) {
        int slot = (end - blocks) * B;
#pragma unroll
        for (int w = 0; w < kSmallWaves; ++w) {
          t.table[w * E + lane] = slot;
          slot += c[w];
        }
        t.total[lane] = all;
        t.first_block[lane] = end - blocks;
        if (lane == E - 1) t.first_block[E] = end;
      }
    }
    __syncthreads();
  } else {
    scan_segments(t.table, t.total, E, tid);
    __syncthreads();
    if (wave == 0) {
      int running = 0;
      for (int base = 0; base < E; base += kWave) {
        const int e = base + lane;
        const int blocks = e < E ? static_cast<int>(static_cast<unsigned>(t.total[e] + B - 1) / static_cast<unsigned>(B)) : 0;
        const int end = running + wave_inclusive_scan(blocks);
        if (e < E) t.first_block[e] = end - blocks;
        running = __builtin_amdgcn_readlane(end, kWave - 1);
      }
      if (lane == 0) t.first_block[E] = running;
    }
    __syncthreads();
    for (int e = lane; e < E; e += kWave) mine[e] += t.first_block[e] * B;
    __builtin_amdgcn_wave_barrier();
  }
  segment_scatter(ids, lo, hi, E, bits_for(E), lane, mine, sorted, first);
  const int group = E <= kSmallWaves ? 6 : 4;  // log2 of the lanes an expert gets
  for (int e = tid >> group; e < E; e += kSmallThreads >> group) {
    const int sub = tid & ((1 << group) - 1), b0 = t.first_block[e], b1 = t.first_block[e + 1];
    for (int b = b0 + sub; b < b1; b += 1 << group) expert_ids[b] = e;
    for (int s = b0 * B + t.total[e] + sub; s < b1 * B; s += 1 << group) sorted[s] = static_cast<int32_t>(n);
  }
  const int npost = t.first_block[E] * B;
  for (int64_t s = npost + tid; s < sorted_len; s += kSmallThreads) sorted[s] = static_cast<int32_t>(n);
  if (tid == 0) npost_out[0] = npost;
}

// bf16 token rows [M, K] to quantise to e4m3 alongside (x == nullptr: none)
struct RowQuant {
  const bf16_t* x;
  unsigned char* q;
  float* scale;
  int K;
};

// Workgroups 1 and up of the one-launch routing: the fp8 layer's token rows.  A workgroup to a row has all of the row's loads in flight at
// once (a wavefront to a row, in two passes, was the longest chain of the launch: 8.2 us against 5.0 without the rows at 16 tokens, H = 4096);
// rows beyond its registers take a wavefront each.  So do short rows, of which most of a workgroup's threads have nothing.  Layer with F = 256, 8 experts, top-1, a wavefront / a workgroup to a row, us:
//   16 tokens     H = 256 16.5 / 16.7, 1024 17.5 / 17.6, 1280 20.5 / 20.2, 2048 21.7 / 21.2, 4096 28.9 / 25.6, 8192 45.8 / 37.8, 16384 81.3 / 58.5
//   128           1024 21.6 / 21.65, 1280 22.8 / 22.4, 1792 24.1 / 23.8, 2048 25.6 / 25.0, 4096 36.2 / 32.7, 8192 58.8 / 48.8
//   512           1024 31.9 / 32.4, 1792 36.9 / 37.6, 2048 39.95 / 39.1, 3072 50.0 / 49.5, 4096 57.6 / 55.6, 8192 89.9 / 82.4
//   700           1280 36.9 / 36.7, 2048 42.4 / 42.8, 3072 53.5 / 53.5, 4096 60.7 / 59.6, 5120 74.7 / 71.6
//   1024          1024 38.9 / 39.4, 2048 48.4 / 48.7, 3072 58.5 / 58.8, 4096 63.5 / 64.0, 8192 104.7 / 100.3, 16384 184.5 / 161.1
constexpr int kRowOfBlock = 2 * 8 * kSmallThreads;  // longest row of a workgroup
__host__ __device__ inline bool block_per_row(int64_t M, int K) {
  return K <= kRowOfBlock && (M <= 128 ? K > 1024 : K >= 2048);
}
__host__ __device__ inline int64_t quant_blocks(int64_t M, int K) { return block_per_row(M, K) ? M : (M + kSmallWaves - 1) / kSmallWaves; }
__device__ __forceinline__ void quant_rows_beside(const RowQuant& rq, int64_t M, int tid, float* red) {
  const int64_t block = static_cast<int64_t>(blockIdx.x) - 1;
  const bool whole = block_per_row(M, rq.K);
  const int64_t row = whole ? block : block * kSmallWaves + tid / kWave;
  if (row >= M) return;
  const bf16_t* x = rq.x + row * rq.K;
  unsigned char* q = rq.q + row * rq.K;
  if (!whole) quant_row(x, rq.K, q, rq.scale + row, tid % kWave);
  else if (rq.K <= kRowOfBlock / 2) quant_row_block<bf16_t, 1, kSmallWaves>(x, rq.K, q, rq.scale + row, tid, red);
  else quant_row_block<bf16_t, 2, kSmallWaves>(x, rq.K, q, rq.scale + row, tid, red);
}

template <typename IdT>
__global__ __launch_bounds__(kSmallThreads) void align_small_kernel(
    const IdT* __restrict__ ids, int64_t n, int E, int B, int seg_len, int64_t sorted_len,
    int32_t* __restrict__ sorted, int32_t* __restrict__ expert_ids, int32_t* __restrict__ npost_out) {
  __shared__ SmallTables t;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int64_t lo = min64(n, static_cast<int64_t>(wave) * seg_len);
  const int64_t hi = min64(n, lo + seg_len);
  int first[kScatterPF];  // read once for the histogram and the placement
  segment_ids(ids, lo, hi, lane, first);
  for (int i = tid; i < kSmallWaves * E; i += kSmallThreads) t.table[i] = 0;
  __syncthreads();
  small_sort(t, ids, first, lo, hi, n, E, B, sorted_len, tid, sorted, expert_ids, npost_out);
}

// Small batches, whole routing in one launch: the workgroup first gates every token (a group of G lanes per token,
// 1024/G tokens per pass; weights and ids go to their global arrays), then sorts the ids it has just written.  The gating of
// one workgroup is bound by vector instructions.  NV > 0: each lane keeps 4 * NV logits (gate_token_blocked), which is
// a quarter of them for 64 experts.
template <typename T, int G, int VPL, int NV>
__global__ __launch_bounds__(kSmallThreads) void route_align_small_kernel(
    const T* __restrict__ logits, int64_t M, int E, int topk, int renorm, int B, int seg_len, int64_t sorted_len,
    float* __restrict__ w_out, int32_t* __restrict__ ids_out, int32_t* __restrict__ sorted,
    int32_t* __restrict__ expert_ids, int32_t* __restrict__ npost_out, RowQuant rq) {
  __shared__ SmallTables t;
  __shared__ int32_t pair_id[kRouteAlignMaxN];  // the ids stay here for the sort: no way out to memory and back
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  if (blockIdx.x > 0) {  // the fp8 layer's token rows are quantised by further workgroups of the same launch
    quant_rows_beside(rq, M, tid, reinterpret_cast<float*>(t.total));
    return;
  }
  for (int i = tid; i < kSmallWaves * E; i += kSmallThreads) t.table[i] = 0;
  constexpr int kPerPass = kSmallThreads / G;
  for (int64_t base = 0; base < M; base += kPerPass) {  // uniform trip count: every lane joins the cross-lane ops
    const int64_t token = base + tid / G;
    const bool live = token < M;
    const T* row = logits + (live ? token : 0) * E;
    float* w_row = w_out + token * topk;
    int32_t* id_row = pair_id + static_cast<int>(live ? token : 0) * topk;
    if constexpr (NV > 0) {
      if (base + wave * (kWave / G) >= M) break;  // a wavefront without a token (it has none in later passes)
      gate_token_blocked<G, NV, true>([&](int e0) { return load4_as_float(row + e0); }, [&](int e) { return to_float(row[e]); }, live, E, topk, renorm, w_row, id_row);
    } else {
      gate_token<G, VPL>([&](int e) { return to_float(row[e]); }, live, E, topk, renorm, w_row, id_row);
    }
  }
  __syncthreads();
  const int64_t n = M * topk;
  const int64_t lo = min64(n, static_cast<int64_t>(wave) * seg_len);
  const int64_t hi = min64(n, lo + seg_len);
  int first[kScatterPF];
  segment_ids(pair_id, lo, hi, lane, first);
  for (int i = tid; i < n; i += kSmallThreads) ids_out[i] = pair_id[i];
  small_sort(t, pair_id, first, lo, hi, n, E, B, sorted_len, tid, sorted, expert_ids, npost_out);
}

// ---------------------------------------------------------------- large path
// counts is [E][S]: after align_segscan_kernel, counts[e][s] is the offset of
// segment s inside expert e's run and totals[e] the length of the run.
template <typename IdT>
__global__ __launch_bounds__(kSegThreads) void align_count_kernel(
    const IdT* __restrict__ ids, int64_t n, int E, int seg_len, int S, int* __restrict__ counts) {
  extern __shared__ int hist[];  // [kSegWaves][E]
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int seg = blockIdx.x * kSegWaves + wave;
  int* mine = hist + wave * E;
  for (int e = lane; e < E; e += kWave) mine[e] = 0;
  __builtin_amdgcn_wave_barrier();
  if (seg >= S) return;
  const int64_t lo = static_cast<int64_t>(seg) * seg_len;
  const int64_t hi = min64(n, lo + seg_len);
  segment_histogram(ids, lo, hi, E, lane, mine);
  __builtin_amdgcn_wave_barrier();
  for (int e = lane; e < E; e += kWave) counts[static_cast<int64_t>(e) * S + seg] = mine[e];
}

// One workgroup per expert: exclusive scan of that expert's per-segment counts
// (in place) and its total.
__global__ __launch_bounds__(kSegThreads) void align_segscan_kernel(int* __restrict__ counts,
                                                                     int* __restrict__ totals, int S) {
  __shared__ int wave_sum[kSegWaves];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  int* row = counts + static_cast<int64_t>(e) * S;
  int running = 0;
  for (int base = 0; base < S; base += kSegThreads) {
    const int s = base + tid;
    const int c = (s < S) ? row[s] : 0;
    const int incl = wave_inclusive_scan(c);
    if (lane == kWave - 1) wave_sum[wave] = incl;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kSegWaves; ++w) {
      const int ws = wave_sum[w];
      before += (w < wave) ? ws : 0;
      all += ws;
    }
    if (s < S) row[s] = running + before + incl - c;
    running += all;
    __syncthreads();
  }
  if (tid == 0) totals[e] = running;
}

// Scatter pass.  Every workgroup rebuilds the run starts from the E totals (cheap),
// workgroup e < E also writes expert e's block table and padding, workgroup 0 the
// tail and the padded length; then each wavefront places its segment.
template <typename IdT>
__global__ __launch_bounds__(kSegThreads) void align_scatter_kernel(
    const IdT* __restrict__ ids, int64_t n, int E, int B, int seg_len, int S, int64_t sorted_len,
    const int* __restrict__ counts, const int* __restrict__ totals, int32_t* __restrict__ sorted,
    int32_t* __restrict__ expert_ids, int32_t* __restrict__ npost_out) {
  extern __shared__ int hist[];  // [kSegWaves][E]
  __shared__ int start[kMaxE + 1];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  if (wave == 0) scan_padded_totals(totals, start, E, B, lane);
  __syncthreads();
  if (static_cast<int>(blockIdx.x) < E) {
    const int e = blockIdx.x;
    for (int b = start[e] / B + tid; b < start[e + 1] / B; b += kSegThreads) expert_ids[b] = e;
    for (int s = start[e] + totals[e] + tid; s < start[e + 1]; s += kSegThreads) sorted[s] = static_cast<int32_t>(n);
  }
  if (blockIdx.x == 0) {
    for (int64_t s = start[E] + tid; s < sorted_len; s += kSegThreads) sorted[s] = static_cast<int32_t>(n);
    if (tid == 0) npost_out[0] = start[E];
  }
  const int seg = blockIdx.x * kSegWaves + wave;
  if (seg >= S) return;
  int* mine = hist + wave * E;
  for (int e = lane; e < E; e += kWave) mine[e] = start[e] + counts[static_cast<int64_t>(e) * S + seg];
  __builtin_amdgcn_wave_barrier();
  const int64_t lo = static_cast<int64_t>(seg) * seg_len;
  const int64_t hi = min64(n, lo + seg_len);
  segment_scatter(ids, lo, hi, E, bits_for(E), lane, mine, sorted);
}

// ---------------------------------------------------------------- large path, two launches
// The per-expert scan over segments costs a launch of its own only because every scatter workgroup needs
// (a) each expert's total and (b) the pairs of each expert in the segments before its own.  Here a count
// workgroup covers 16 segments and leaves their sums in wgcnt[b][e]; a scatter workgroup gets (a) and (b) from one pass
// over the NB x E sums (12288 values for 64 experts and 393 216 pairs: twelve loads per thread, all of one expert, summed in
// registers before two integer LDS atomics, so the order does not matter), and counts its own 16 segments again while these are
// on their way: the ids are in its registers anyway.  Used while NB x E stays small.
// A wavefront places its 64-pair rounds one behind the other, so segments are short (two_level_seg_len); 256 pairs and more each left most
// CUs without a wavefront.  Both launches, ids that change from call to call, us, segments of 256 pairs (a 2048th from 524 288 on)
// and a table of every segment's counts in memory / now:
//   64 experts    6200 pairs 8.9 / 6.4, 20000 9.5 / 7.1, 100000 10.3 / 7.8, 200000 10.9 / 8.2, 393216 11.5 / 9.1, 1000000 16.7 / 12.8, 4000000 42.6 / 32.3
//   8 experts     20000 9.0 / 6.5, 100000 9.1 / 6.7, 400000 9.4 / 9.3, 1000000 14.3 / 11.4, 4000000 38.1 / 26.7
//   256 experts   200000 15.8 / 11.9;  512 50000 20.1 / 11.2
constexpr int kSeg2Threads = 1024;
constexpr int kSeg2Waves = kSeg2Threads / kWave;
constexpr int64_t kTwoLevelMaxEntries = 16384;

template <typename IdT>
__global__ __launch_bounds__(kSeg2Threads) void align_count2_kernel(
    const IdT* __restrict__ ids, int64_t n, int E, int seg_len, int* __restrict__ wgcnt) {
  extern __shared__ int hist[];  // [E]
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int64_t lo = min64(n, (static_cast<int64_t>(blockIdx.x) * kSeg2Waves + wave) * seg_len);
  const int64_t hi = min64(n, lo + seg_len);
  int first[kScatterPF];
  segment_ids(ids, lo, hi, lane, first);
  for (int e = tid; e < E; e += kSeg2Threads) hist[e] = 0;
  __syncthreads();
  segment_histogram(ids, lo, hi, E, lane, hist, first);
  __syncthreads();
  for (int e = tid; e < E; e += kSeg2Threads) wgcnt[static_cast<int64_t>(blockIdx.x) * E + e] = hist[e];
}

template <typename IdT>
__global__ __launch_bounds__(kSeg2Threads) void align_scatter2_kernel(
    const IdT* __restrict__ ids, int64_t n, int E, int B, int seg_len, int NB, int64_t sorted_len,
    const int* __restrict__ wgcnt, int32_t* __restrict__ sorted,
    int32_t* __restrict__ expert_ids, int32_t* __restrict__ npost_out) {
  extern __shared__ int hist[];  // [kSeg2Waves][E]
  __shared__ int start[kMaxE + 1];
  __shared__ int total[kMaxE];
  __shared__ int before[kMaxE];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int wg = blockIdx.x;
  const int64_t lo = min64(n, (static_cast<int64_t>(wg) * kSeg2Waves + wave) * seg_len);
  const int64_t hi = min64(n, lo + seg_len);
  int first[kScatterPF];
  segment_ids(ids, lo, hi, lane, first);
  for (int e = tid; e < E; e += kSeg2Threads) total[e] = before[e] = 0;
  for (int i = tid; i < kSeg2Waves * E; i += kSeg2Threads) hist[i] = 0;
  __syncthreads();
  // expert e: all pairs, and the pairs in the workgroups before this one.  A thread keeps one expert and sums every
  // (1024 / E)-th workgroup in registers: independent loads, two LDS atomics at the end.  E <= 512 (the launcher).
  const int per_pass = kSeg2Threads / E, my_e = tid % E, b0 = tid / E;
  if (E * NB <= kSeg2Threads) {
    const int c = tid < E * NB ? wgcnt[tid] : 0;
    if (c != 0) {
      atomicAdd(&total[my_e], c);
      if (b0 < wg) atomicAdd(&before[my_e], c);
    }
  } else if (b0 < per_pass) {
    int all = 0, below = 0;
#pragma unroll 4
    for (int b = b0; b < NB; b += per_pass) {
      const int c = wgcnt[static_cast<int64_t>(b) * E + my_e];
      all += c;
      below += b < wg ? c : 0;
    }
    if (all != 0) atomicAdd(&total[my_e], all);
    if (below != 0) atomicAdd(&before[my_e], below);
  }
  int* mine = hist + wave * E;
  segment_histogram(ids, lo, hi, E, lane, mine, first);
  __syncthreads();
  if (wave == 0) scan_padded_totals(total, start, E, B, lane);
  __syncthreads();
  // a segment's counts -> its next free slots
  for (int e = tid; e < E; e += kSeg2Threads) {
    int c[kSeg2Waves], slot = start[e] + before[e];
#pragma unroll
    for (int w = 0; w < kSeg2Waves; ++w) c[w] = hist[w * E + e];
#pragma unroll
    for (int w = 0; w < kSeg2Waves; ++w) {
      hist[w * E + e] = slot;
      slot += c[w];
    }
  }
  if (wg < E) {
    const int e = wg;
    for (int b = start[e] / B + tid; b < start[e + 1] / B; b += kSeg2Threads) expert_ids[b] = e;
    for (int s = start[e] + total[e] + tid; s < start[e + 1]; s += kSeg2Threads) sorted[s] = static_cast<int32_t>(n);
  }
  if (wg == 0) {
    for (int64_t s = start[E] + tid; s < sorted_len; s += kSeg2Threads) sorted[s] = static_cast<int32_t>(n);
    if (tid == 0) npost_out[0] = start[E];
  }
  __syncthreads();
  segment_scatter(ids, lo, hi, E, bits_for(E), lane, mine, sorted, first);
}

bool use_small_path(int64_t n, int E) { return n <= kSmallMaxN && E <= kSmallMaxE; }

int large_seg_len(int64_t n) {
  const int64_t want = round_up(ceil_div(n, 2048), kWave);
  return static_cast<int>(want < 256 ? 256 : want);
}
// Pairs per segment of the two launches: one 64-pair round up to 524 288 pairs and an 8192nd beyond, or as many more as keep the workgroup sums
// within kTwoLevelMaxEntries (a 2048th of the pairs from the start: 393216 pairs on 64 experts 9.8 us and not 9.1, 1000000 on 8 16.4 and not 11.4);
// 0: too many sums all the same, the three launches.
int two_level_seg_len(int64_t n, int E) {
  if (E > 512) return 0;
  const int longest = large_seg_len(n);
  for (int64_t len = n > 0 ? round_up(ceil_div(n, 8192), kWave) : kWave; len <= longest; len += kWave)
    if (E * ceil_div(ceil_div(n, len), kSeg2Waves) <= kTwoLevelMaxEntries) return static_cast<int>(len);
  return 0;
}
// workgroups of the count launch, a set of sums each
int two_level_groups(int64_t n, int len) { return static_cast<int>(n > 0 ? ceil_div(ceil_div(n, len), kSeg2Waves) : 1); }

template <typename IdT>
int run(const void* ids_v, int64_t n, int E, int B, int32_t* sorted, int32_t* expert_ids,
        int32_t* npost, void* ws, hipStream_t st) {
  const IdT* ids = static_cast<const IdT*>(ids_v);
  const int64_t sorted_len = n + static_cast<int64_t>(E) * (B - 1);
  if (use_small_path(n, E)) {
    int seg_len = static_cast<int>(round_up(ceil_div(n, kSmallWaves), kWave));
    if (seg_len == 0) seg_len = kWave;
    hipLaunchKernelGGL((align_small_kernel<IdT>), dim3(1), dim3(kSmallThreads), 0, st, ids, n, E, B,
                       seg_len, sorted_len, sorted, expert_ids, npost);
    return check_launch("align_small_kernel");
  }
  const int seg_len = large_seg_len(n);
  const int S = static_cast<int>(n > 0 ? ceil_div(n, seg_len) : 1);
  int* counts = static_cast<int*>(ws);
  int* run_start = counts + static_cast<int64_t>(E) * S;
  const unsigned blocks = static_cast<unsigned>(ceil_div(S, kSegWaves));
  const unsigned scatter_blocks = blocks > static_cast<unsigned>(E) ? blocks : static_cast<unsigned>(E);
  const size_t lds = sizeof(int) * kSegWaves * E;
  if (const int len = two_level_seg_len(n, E)) {  // workgroup sums, scatter: two launches
    const int NB = two_level_groups(n, len);
    hipLaunchKernelGGL((align_count2_kernel<IdT>), dim3(NB), dim3(kSeg2Threads), sizeof(int) * E, st, ids, n, E, len, counts);
    hipLaunchKernelGGL((align_scatter2_kernel<IdT>), dim3(NB > E ? NB : E), dim3(kSeg2Threads), sizeof(int) * kSeg2Waves * E, st, ids, n, E, B,
                       len, NB, sorted_len, counts, sorted, expert_ids, npost);
    return check_launch("align kernels");
  }
  hipLaunchKernelGGL((align_count_kernel<IdT>), dim3(blocks), dim3(kSegThreads), lds, st, ids, n, E,
                     seg_len, S, counts);
  hipLaunchKernelGGL(align_segscan_kernel, dim3(E), dim3(kSegThreads), 0, st, counts, run_start, S);
  hipLaunchKernelGGL((align_scatter_kernel<IdT>), dim3(scatter_blocks), dim3(kSegThreads), lds, st, ids, n, E, B,
                     seg_len, S, sorted_len, counts, run_start, sorted, expert_ids, npost);
  return check_launch("align kernels");
}

// Rows that 4-element vector loads can read, 17 to 64 experts: a few lanes per token in the one-workgroup form.  Renormalised weights
// only: their sum is taken in the order of rank, as gate_token takes it, so that a weight has the same bits from either.
// (Above 64 experts the two forms order NaN differently.)  Any topk: from 24 tokens on the several logits win at each, with fewer tokens the two are within
// 0.3 us.  Layer with H = F = 128, one / several, us: 64 experts, 48 tokens, top-1 16.4 / 15.0, top-2 16.8 / 14.9, 32 tokens, top-8 19.2 / 16.9, top-16 23.9 / 20.2, top-32
// 34.8 / 27.7, 16 tokens, top-64 39.4 / 39.6; 32 experts, 64 tokens, top-8 20.25 / 17.7, top-16 31.2 / 27.0, 32, top-32 33.1 / 31.9; fp8 layers (F = 256), 64 experts, 64 tokens,
// top-16 39.1 / 29.3, 170, top-6 42.2 / 29.4, 250, top-1 32.05 / 24.2, 32 experts, 250, top-4 33.0 / 25.0.
bool gated_blocked(const void* logits, size_t elem, int E, int topk, int renorm) {
  return renorm && E > 16 && E <= 64 && E % 4 == 0 && reinterpret_cast<uintptr_t>(logits) % (4 * elem) == 0 && topk <= kBlockedSlots * (E <= 32 ? 8 : 16);
}

template <typename T, int G, int VPL, int NV>
void launch_route_align(const void* logits, int64_t M, int E, int topk, int renorm, int B, int64_t sorted_len,
                        float* w, int32_t* ids, int32_t* sorted, int32_t* expert_ids, int32_t* npost, RowQuant rq,
                        hipStream_t st) {
  int seg_len = static_cast<int>(round_up(ceil_div(M * topk, kSmallWaves), kWave));
  if (seg_len == 0) seg_len = kWave;
  const unsigned grid = 1 + (rq.x ? static_cast<unsigned>(quant_blocks(M, rq.K)) : 0u);
  hipLaunchKernelGGL((route_align_small_kernel<T, G, VPL, NV>), dim3(grid), dim3(kSmallThreads), 0, st,
                     static_cast<const T*>(logits), M, E, topk, renorm, B, seg_len, sorted_len, w, ids, sorted,
                     expert_ids, npost, rq);
}

template <typename T>
void dispatch_route_align(const void* logits, int64_t M, int E, int topk, int renorm, int B, int64_t sorted_len,
                          float* w, int32_t* ids, int32_t* sorted, int32_t* expert_ids, int32_t* npost, RowQuant rq,
                          hipStream_t st) {
#define FR_RA(G, VPL, NV) launch_route_align<T, G, VPL, NV>(logits, M, E, topk, renorm, B, sorted_len, w, ids, sorted, expert_ids, npost, rq, st)
  if (gated_blocked(logits, sizeof(T), E, topk, renorm)) {
    if (E <= 32) FR_RA(8, 1, 1);
    else FR_RA(16, 1, 1);
  } else if (E <= 1) FR_RA(1, 1, 0);
  else if (E <= 2) FR_RA(2, 1, 0);
  else if (E <= 4) FR_RA(4, 1, 0);
  else if (E <= 8) FR_RA(8, 1, 0);
  else if (E <= 16) FR_RA(16, 1, 0);
  else if (E <= 32) FR_RA(32, 1, 0);
  else if (E <= 64) FR_RA(64, 1, 0);
  else if (E <= 128) FR_RA(64, 2, 0);
  else FR_RA(64, 4, 0);
#undef FR_RA
}

}  // namespace

// Gating and routing arrays in one launch for small batches; false when the shape is
// outside what one workgroup should do (the caller then runs the two stages separately).
// One workgroup's gating is a chain of rounds of 16 wavefronts x 64 / G tokens, G = next power of two of E; two launches cost 1 to 3 us more and
// spread the gating over the CUs.  A layer with H = F = 128, one / two launches, us (the sort of then, a microsecond longer in either):
//   16 experts, top-2   192 tokens (3 rounds) 18.7 / 19.9, 256 (4) 25.1 / 23.6, 512 29.2 / 24.4;  8, top-2 256 (2) 23.2 / 23.7, 384 (3) 24.9 / 24.6, 512 26.2 / 24.9
//   64, top-6           16 (1) 17.8 / 19.8, 32 (2) 19.8 / 19.5, 48 (3) 21.9 / 19.8, 80 (5) 25.9 / 19.7, 168 38.4 / 20.8
//   128, top-8 (two logits per lane)   16 (1) 22.6 / 22.3, 32 (2) 27.8 / 22.8, 127 57.5 / 24.5;  256 16 26.0 / 25.3, 64 48.9 / 29.5
// With several logits per lane (gated_blocked) there are fewer rounds, and at the line one launch is the clearly better one: 64 experts, top-6, 32 tokens
// 16.2 / 17.5, 32, top-4, 64 tokens 15.6 / 16.9.  The line is all the same that of one logit per lane, which weights that are not renormalised and
// unaligned logits still take: a further one would be 0.4 to 0.5 us better at 64 (128) tokens and worse from 96 (256) on (builds with the line
// moved there: 64 experts 64 tokens 17.8 / 18.2, 96 19.5 / 18.6, 160 21.9 / 18.5; 32 experts 128 16.8 / 17.3, 256 24.6 / 22.9).
// quant: the launch also quantises the token rows, which would be a third one; it then keeps all that one workgroup holds.
bool route_align_fits(int64_t M, int E, int topk, bool quant) {
  if (M < 1 || M * topk > kRouteAlignMaxN || !use_small_path(M * topk, E) || M * E > 16384 || topk > E) return false;
  int G = 1;
  while (G < E && G < 64) G *= 2;
  return quant || M * G <= 1024 * (E > 64 ? 1 : topk <= 2 ? 3 : 2);
}
int route_align_small(const void* logits, int logits_dtype, int64_t M, int E, int topk, int renorm, int block,
                      float* w, int32_t* ids, int32_t* sorted, int32_t* expert_ids, int32_t* npost,
                      const void* qx, int64_t qK, void* qq, float* qscale, hipStream_t st) {
  const int64_t sorted_len = M * topk + int64_t(E) * (block - 1);
  const RowQuant rq = {static_cast<const bf16_t*>(qx), static_cast<unsigned char*>(qq), qscale, static_cast<int>(qK)};
  switch (logits_dtype) {
    case FR_F32: dispatch_route_align<float>(logits, M, E, topk, renorm, block, sorted_len, w, ids, sorted, expert_ids, npost, rq, st); break;
    case FR_F16: dispatch_route_align<f16_t>(logits, M, E, topk, renorm, block, sorted_len, w, ids, sorted, expert_ids, npost, rq, st); break;
    case FR_BF16: dispatch_route_align<bf16_t>(logits, M, E, topk, renorm, block, sorted_len, w, ids, sorted, expert_ids, npost, rq, st); break;
    default: return fail(FR_E_DTYPE, "route_align_small: logits dtype %d not in {f32, f16, bf16}", logits_dtype);
  }
  return check_launch("route_align_small_kernel");
}

}  // namespace fr

extern "C" int64_t fr_moe_align_workspace_bytes(int64_t n, int E) {
  using namespace fr;
  if (n < 0 || E < 1 || E > kMaxE) return -1;
  if (use_small_path(n, E)) return 0;
  // two launches: the count workgroups' sums; three: [E][S] counts and E totals
  if (const int len = two_level_seg_len(n, E)) return static_cast<int64_t>(sizeof(int)) * E * two_level_groups(n, len);
  const int64_t S = n > 0 ? ceil_div(n, large_seg_len(n)) : 1;
  return static_cast<int64_t>(sizeof(int)) * E * (S + 1);
}

extern "C" int fr_moe_align(const void* topk_ids, int ids_dtype, int64_t n, int E, int block,
                            int32_t* sorted_token_ids, int32_t* expert_ids,
                            int32_t* num_tokens_post_pad, void* workspace, int64_t workspace_bytes,
                            void* stream) {
  using namespace fr;
  FR_REQUIRE(n >= 0 && n <= (int64_t(1) << 30), FR_E_SHAPE, "fr_moe_align: n=%lld outside [0, 2^30]", (long long)n);
  FR_REQUIRE(E >= 1 && E <= kMaxE, FR_E_SHAPE, "fr_moe_align: E=%d outside [1, %d]", E, kMaxE);
  FR_REQUIRE(block >= 1 && block <= 4096, FR_E_SHAPE, "fr_moe_align: block=%d outside [1, 4096]", block);
  FR_REQUIRE(n + int64_t(E) * block < (int64_t(1) << 31), FR_E_SHAPE, "fr_moe_align: padded length overflows int32");
  FR_REQUIRE(expert_ids && num_tokens_post_pad && (sorted_token_ids || n + int64_t(E) * (block - 1) == 0), FR_E_NULL, "fr_moe_align: null output pointer");
  FR_REQUIRE(n == 0 || topk_ids, FR_E_NULL, "fr_moe_align: null topk_ids");
  FR_REQUIRE(ids_dtype == FR_I32 || ids_dtype == FR_I64, FR_E_DTYPE, "fr_moe_align: ids dtype %d not in {i32, i64}", ids_dtype);
  const int64_t need = fr_moe_align_workspace_bytes(n, E);
  FR_REQUIRE(need == 0 || (workspace && workspace_bytes >= need), FR_E_WORKSPACE,
             "fr_moe_align: workspace %lld < %lld bytes", (long long)workspace_bytes, (long long)need);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (ids_dtype == FR_I32) return run<int32_t>(topk_ids, n, E, block, sorted_token_ids, expert_ids, num_tokens_post_pad, workspace, st);
  return run<int64_t>(topk_ids, n, E, block, sorted_token_ids, expert_ids, num_tokens_post_pad, workspace, st);
}
