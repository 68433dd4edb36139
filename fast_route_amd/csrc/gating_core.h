// Gating core shared by the gating kernels and the fused small-batch routing kernel:
// cross-lane reductions over a group of G lanes and gate_token(), the top-k gating of one
// token by one lane group.
#pragma once
#include "fr_common.h"

#include <float.h>
#include <limits.h>

#include <type_traits>

namespace fr {
namespace {

__device__ __forceinline__ bool better(float av, int ai, float bv, int bi) {
  return av > bv || (av == bv && ai < bi);
}

// max over the group, returned in every lane: DPP steps inside a row of 16 lanes,
// then the (uniform per row) row maxima are read out as scalars and combined
template <int G>
__device__ __forceinline__ float group_max(float v) {
  if constexpr (G > 1) v = fmaxf(v, partner_f32<1>(v));
  if constexpr (G > 2) v = fmaxf(v, partner_f32<2>(v));
  if constexpr (G > 4) v = fmaxf(v, partner_f32<4>(v));
  if constexpr (G > 8) v = fmaxf(v, partner_f32<8>(v));
  if constexpr (G > 16) {
    const int bits = __float_as_int(v);
    const float r0 = __int_as_float(__builtin_amdgcn_readlane(bits, 0));
    const float r1 = __int_as_float(__builtin_amdgcn_readlane(bits, 16));
    const float r2 = __int_as_float(__builtin_amdgcn_readlane(bits, 32));
    const float r3 = __int_as_float(__builtin_amdgcn_readlane(bits, 48));
    if constexpr (G == 32) v = (threadIdx.x & 32) ? fmaxf(r2, r3) : fmaxf(r0, r1);
    else v = fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
  }
  return v;
}

// sum over the group, same scheme (every lane adds the same numbers in the same order)
template <int G>
__device__ __forceinline__ float group_sum(float v) {
  if constexpr (G > 1) v += partner_f32<1>(v);
  if constexpr (G > 2) v += partner_f32<2>(v);
  if constexpr (G > 4) v += partner_f32<4>(v);
  if constexpr (G > 8) v += partner_f32<8>(v);
  if constexpr (G > 16) {
    const int bits = __float_as_int(v);
    const float r0 = __int_as_float(__builtin_amdgcn_readlane(bits, 0));
    const float r1 = __int_as_float(__builtin_amdgcn_readlane(bits, 16));
    const float r2 = __int_as_float(__builtin_amdgcn_readlane(bits, 32));
    const float r3 = __int_as_float(__builtin_amdgcn_readlane(bits, 48));
    if constexpr (G == 32) v = (threadIdx.x & 32) ? (r2 + r3) : (r0 + r1);
    else v = (r0 + r1) + (r2 + r3);
  }
  return v;
}

// Order-preserving map fp32 -> uint32 (larger float <=> larger key; every real value,
// -inf included, maps above 0, which serves as "not a candidate").
__device__ __forceinline__ unsigned float_key(float v) {
  const unsigned b = __float_as_uint(v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float key_float(unsigned k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}
// unsigned max over the group, in every lane (integer max needs no NaN canonicalisation,
// so the DPP moves fold into v_max_u32; rows are combined on the scalar unit)
template <int G>
__device__ __forceinline__ unsigned group_max_key(unsigned k) {
  if constexpr (G > 1) k = max(k, static_cast<unsigned>(partner_i32<1>(static_cast<int>(k))));
  if constexpr (G > 2) k = max(k, static_cast<unsigned>(partner_i32<2>(static_cast<int>(k))));
  if constexpr (G > 4) k = max(k, static_cast<unsigned>(partner_i32<4>(static_cast<int>(k))));
  if constexpr (G > 8) k = max(k, static_cast<unsigned>(partner_i32<8>(static_cast<int>(k))));
  if constexpr (G > 16) {
    const unsigned r0 = __builtin_amdgcn_readlane(static_cast<int>(k), 0);
    const unsigned r1 = __builtin_amdgcn_readlane(static_cast<int>(k), 16);
    const unsigned r2 = __builtin_amdgcn_readlane(static_cast<int>(k), 32);
    const unsigned r3 = __builtin_amdgcn_readlane(static_cast<int>(k), 48);
    if constexpr (G == 32) k = (threadIdx.x & 32) ? max(r2, r3) : max(r0, r1);
    else k = max(max(r0, r1), max(r2, r3));
  }
  return k;
}

// Cross-lane merge of per-lane online-softmax states (m = running max, s = sum of
// exp(x - m)): one max reduction, one rescale, one sum reduction.
template <int G>
__device__ __forceinline__ void group_online_softmax(float& m, float& s) {
  const float gm = group_max<G>(m);
  s = group_sum<G>((m == -INFINITY) ? 0.f : s * __expf(m - gm));
  m = gm;
}

template <int G>
__device__ __forceinline__ void group_argmax(float& v, int& i) {
  auto step = [&](auto tag) {
    constexpr int S = decltype(tag)::value;
    const float ov = partner_f32<S>(v);
    const int oi = partner_i32<S>(i);
    if (better(ov, oi, v, i)) {
      v = ov;
      i = oi;
    }
  };
  if constexpr (G > 1) step(std::integral_constant<int, 1>{});
  if constexpr (G > 2) step(std::integral_constant<int, 2>{});
  if constexpr (G > 4) step(std::integral_constant<int, 4>{});
  if constexpr (G > 8) step(std::integral_constant<int, 8>{});
  if constexpr (G > 16) step(std::integral_constant<int, 16>{});
  if constexpr (G > 32) step(std::integral_constant<int, 32>{});
}

constexpr int kGateThreads = 256;

// Gating of one token by a group of G lanes.  `load(e)` returns logit e as fp32;
// every lane of the wavefront must call this (dead groups pass live = false).
template <int G, int VPL, typename Load>
__device__ __forceinline__ void gate_token(Load load, bool live, int E, int topk, int renorm,
                                           float* __restrict__ w_row, int32_t* __restrict__ id_row) {
  const int g = threadIdx.x % G;
  float v[VPL];
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int e = g + i * G;
    v[i] = (live && e < E) ? load(e) : -INFINITY;
  }

  // online softmax over this lane's values (running max, rescaled running sum),
  // then merged across the group
  float m = v[0];
  float s = (v[0] == -INFINITY) ? 0.f : 1.f;
#pragma unroll
  for (int i = 1; i < VPL; ++i) {
    if (v[i] == -INFINITY) continue;
    const float mn = fmaxf(m, v[i]);
    s = (m == -INFINITY ? 0.f : s * __expf(m - mn)) + __expf(v[i] - mn);
    m = mn;
  }
  group_online_softmax<G>(m, s);

  float sel_v[VPL];
  int sel_i[VPL];
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    sel_v[i] = -INFINITY;
    sel_i[i] = 0;
  }
  unsigned taken = 0;
  float sel_sum = 0.f;
  const unsigned vkey = float_key(v[0] + 0.f);  // + 0.f: -0 and +0 are the same value
  for (int r = 0; r < topk; ++r) {
    float bv;
    int bi;
    if constexpr (VPL == 1) {
      // one logit per lane, lane order = expert order: the winner is the group max and,
      // among lanes holding it, the lowest lane (= lowest expert index) of a ballot
      const unsigned key = (g < E && !taken) ? vkey : 0u;
      const unsigned top = group_max_key<G>(key);
      bv = key_float(top);
      unsigned long long hit = __ballot(key == top);
      if constexpr (G < 64) hit = (hit >> (threadIdx.x & 63 & ~(G - 1))) & ((1ull << G) - 1ull);
      bi = __ffsll(hit) - 1;
      if (bi == g) taken = 1u;
    } else {
      bv = -INFINITY;
      bi = INT_MAX;
#pragma unroll
      for (int i = 0; i < VPL; ++i) {
        const int e = g + i * G;
        if (e < E && !((taken >> i) & 1u) && better(v[i], e, bv, bi)) {
          bv = v[i];
          bi = e;
        }
      }
      group_argmax<G>(bv, bi);
      if (bi % G == g) taken |= 1u << (bi / G);
    }
    sel_sum += __expf(bv - m);
#pragma unroll
    for (int sl = 0; sl < VPL; ++sl) {
      if (r == sl * G + g) {
        sel_v[sl] = bv;
        sel_i[sl] = bi;
      }
    }
  }

  const float denom = renorm ? sel_sum : s;
  if (live) {
#pragma unroll
    for (int sl = 0; sl < VPL; ++sl) {
      const int r = sl * G + g;
      if (r < topk) {
        w_row[r] = __expf(sel_v[sl] - m) / denom;
        id_row[r] = sel_i[sl];
      }
    }
  }
}

// 4 consecutive logits as fp32 from a 4-element-aligned address
template <typename T>
__device__ __forceinline__ f32x4 load4_as_float(const T* p) {
  if constexpr (sizeof(T) == 4) {
    return *reinterpret_cast<const f32x4*>(p);
  } else {
    typedef T vec4 __attribute__((ext_vector_type(4)));
    const vec4 t = *reinterpret_cast<const vec4*>(p);
    return f32x4{to_float(t[0]), to_float(t[1]), to_float(t[2]), to_float(t[3])};
  }
}

// Many experts: a group of only G lanes owns a token and every lane keeps NV vectors of 4
// consecutive logits, vector j of lane g holding experts 4*(G*j + g) .. 4*(G*j + g) + 3, so
// the G lanes read 4*G consecutive logits of the token per load and a wavefront gates 64/G
// tokens at once: the cross-lane rounds (the cost of the one-logit-per-lane form, a wavefront
// instruction per step per token) shrink to log2(G) steps shared by 64/G tokens.  Inside a
// lane expert indices rise with the slot number, across lanes ties go to the lower index,
// so the order is still (value descending, index ascending).  load4(e0) returns logits
// e0..e0+3, load1(e) logit e; E must be a multiple of 4.
//
// Bound by vector instructions (a lane looks at 4*NV logits in every round), so the selection runs on packed keys:
// the upper bits of a logit's order key over the complement of its expert index, which no two experts of a token
// share.  The largest key below the previous winner is the largest key minus the winner modulo 2^32 (keys above or
// equal wrap to small values, those below to large ones, nearest first): a subtraction and half a three-way maximum
// per logit and round where comparing exact keys and remembering the slot took five instructions.
// The packed order is the exact one unless two logits differ only in the bits the index displaced; that shows as two
// successive winners (one more than asked for is drawn) with equal upper bits while some logit of the token has a bit
// set down there.  A wavefront that sees it in any of its tokens puts these right: where the class of equal upper bits
// reaches beyond the last winner, the places it holds are filled again in the exact order of that class alone (its keys
// are the displaced bits over the index), then every winner's place is counted from the winners' own logits.  Logits that
// came from 16-bit values have no such bits.  (Sorting the winners by exchanges of neighbours took 15.1 us where the count
// takes 12.3, 64 experts, top-6, all in one class; 256 experts, top-32, it was 10 % faster.)
// Random fp32 logits, us, exact keys compared in every round / a whole second selection on exact keys after a collision /
// now: 65536 tokens, 64 experts, top-6 13.1 / 10.0 / 9.3; 16384 tokens, 256 experts, top-8 16.1 / 11.9 / 10.8, top-32 40.7 /
// 36.5 / 21.2.  A collision in every wavefront, 65536 tokens, 64 experts: 16-bit logits scaled in fp32 12.3 / 12.6 / 10.5,
// all but topk - 1 experts masked 11.5 / 12.7 / 9.9, all 64 logits within 70 units in the last place 12.5 / 12.5 / 12.3.
constexpr int kBlockedSlots = 4;  // result slots per lane: topk <= kBlockedSlots * G

// RANKED: renormalised weights from the largest logit and their sum in the order of rank, as gate_token takes them.
template <int G, int NV, bool RANKED = false, typename Load4, typename Load1>
__device__ __forceinline__ void gate_token_blocked(Load4 load4, Load1 load1, bool live, int E, int topk, int renorm,
                                                   float* __restrict__ w_row, int32_t* __restrict__ id_row) {
  constexpr int VPL = 4 * NV;
  static_assert(G <= 16, "the all-reduce uses the in-row DPP steps only");
  constexpr unsigned kIndexMask = G * VPL - 1;
  static_assert((G * VPL & (G * VPL - 1)) == 0, "expert indices fill whole bits");
  const int g = threadIdx.x % G;
  float v[VPL];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int e0 = 4 * (G * j + g);
    f32x4 t = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (live && e0 < E) t = load4(e0);
#pragma unroll
    for (int c = 0; c < 4; ++c) v[4 * j + c] = t[c];
  }

  // Packed keys of this lane's logits (0 = not a candidate); + 0.f: -0 and +0 are the same value.
  unsigned pk[VPL], low = 0u;
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int e = 4 * (G * (i / 4) + g) + (i % 4);
    const float x = v[i] + 0.f;
    if (live) low |= __float_as_uint(x);
    pk[i] = (e < E) ? (float_key(x) & ~kIndexMask) | (kIndexMask - static_cast<unsigned>(e)) : 0u;
  }
  int sel_i[kBlockedSlots];
#pragma unroll
  for (int i = 0; i < kBlockedSlots; ++i) sel_i[i] = 0;
  unsigned win = 0u, prev = 0u;  // this and the previous round's winner; with 0 the first round's difference is the key itself
  unsigned equal = 0u;  // the first winner with the upper bits of the one before it
  int top = 0;        // expert of the largest logit
  for (int r = 0; r <= topk; ++r) {
    unsigned best = 0u;
#pragma unroll
    for (int i = 0; i < VPL; ++i) best = max(best, pk[i] - win);
    if constexpr (G > 1) best = max(best, static_cast<unsigned>(partner_i32<1>(static_cast<int>(best))));
    if constexpr (G > 2) best = max(best, static_cast<unsigned>(partner_i32<2>(static_cast<int>(best))));
    if constexpr (G > 4) best = max(best, static_cast<unsigned>(partner_i32<4>(static_cast<int>(best))));
    if constexpr (G > 8) best = max(best, static_cast<unsigned>(partner_i32<8>(static_cast<int>(best))));
    const unsigned next = best + win;
    if (r > 0 && equal == 0u && ((next ^ win) & ~kIndexMask) == 0u) equal = next;
    prev = win;
    win = next;
    const int be = static_cast<int>(kIndexMask - (win & kIndexMask));
    if (r == 0) top = be;
    if (r < topk) {
#pragma unroll
      for (int sl = 0; sl < kBlockedSlots; ++sl)
        if (r == sl * G + g) sel_i[sl] = be;
    }
  }
  bool unsorted = false;  // winners whose order among themselves is in doubt
  if (__any(equal != 0u) && __any((low & kIndexMask) != 0u)) {
    // prev: the last winner, win: the one drawn beyond it
    int above = 0;  // logits of the token in higher classes than the last winner's
    unsigned ck[VPL];  // keys of that class, 0 for the rest
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int e = 4 * (G * (i / 4) + g) + (i % 4);
      above += pk[i] > (prev | kIndexMask) ? 1 : 0;
      ck[i] = (e < E && ((pk[i] ^ prev) & ~kIndexMask) == 0u)
                  ? (float_key(v[i] + 0.f) & kIndexMask) * (kIndexMask + 1) + (pk[i] & kIndexMask) + 1u : 0u;
    }
    if constexpr (G > 1) above += partner_i32<1>(above);
    if constexpr (G > 2) above += partner_i32<2>(above);
    if constexpr (G > 4) above += partner_i32<4>(above);
    if constexpr (G > 8) above += partner_i32<8>(above);
    const int places = (live && ((win ^ prev) & ~kIndexMask) == 0u) ? topk - above : 0;
    // a refilled class comes out in order: left to sort are higher classes, or one that ends with the last winner
    unsorted = live && equal != 0u && (places == 0 || equal > (prev | kIndexMask));
    unsigned cw = 0u;
    for (int q = 0; __any(q < places); ++q) {
      unsigned best = 0u;
#pragma unroll
      for (int i = 0; i < VPL; ++i) best = max(best, ck[i] - cw);
      if constexpr (G > 1) best = max(best, static_cast<unsigned>(partner_i32<1>(static_cast<int>(best))));
      if constexpr (G > 2) best = max(best, static_cast<unsigned>(partner_i32<2>(static_cast<int>(best))));
      if constexpr (G > 4) best = max(best, static_cast<unsigned>(partner_i32<4>(static_cast<int>(best))));
      if constexpr (G > 8) best = max(best, static_cast<unsigned>(partner_i32<8>(static_cast<int>(best))));
      cw += best;
      if (q < places) {
#pragma unroll
        for (int sl = 0; sl < kBlockedSlots; ++sl)
          if (above + q == sl * G + g) sel_i[sl] = static_cast<int>(kIndexMask - ((cw - 1u) & kIndexMask));
      }
    }
  }

  // The winners' logits again from the cache the row was just read through: they are spread over the lanes' registers.
  // Asked for together and unconditionally: slots that are not in use hold expert 0, groups without a token read token 0.
  float sel_v[kBlockedSlots], top_v = load1(top);
#pragma unroll
  for (int sl = 0; sl < kBlockedSlots; ++sl) sel_v[sl] = load1(sel_i[sl]);
  top_v += 0.f;
#pragma unroll
  for (int sl = 0; sl < kBlockedSlots; ++sl) sel_v[sl] = sl * G + g < topk ? sel_v[sl] + 0.f : -INFINITY;

  int place[kBlockedSlots];
#pragma unroll
  for (int sl = 0; sl < kBlockedSlots; ++sl) place[sl] = sl * G + g;
  if (__any(unsorted)) {
    // Every winner's place is the number of winners before it: the lanes' winners go round the group (Gray code over the
    // four exchanges), each compared with this lane's.  Slots that are not in use come after all others.
    unsigned key[kBlockedSlots], ok[kBlockedSlots];
    int oe[kBlockedSlots];
    unsigned top_key = 0u;
#pragma unroll
    for (int sl = 0; sl < kBlockedSlots; ++sl) {
      key[sl] = ok[sl] = sl * G + g < topk ? float_key(sel_v[sl]) : 0u;
      oe[sl] = sl * G + g < topk ? sel_i[sl] : INT_MAX;
      place[sl] = 0;
      top_key = max(top_key, key[sl]);
    }
#pragma unroll
    for (int step = 0; step < G; ++step) {
#pragma unroll
      for (int o = 0; o < kBlockedSlots; ++o) {
        if (o * G >= topk) continue;
        auto exchange = [&](auto tag) {
          constexpr int S = decltype(tag)::value;
          ok[o] = static_cast<unsigned>(partner_i32<S>(static_cast<int>(ok[o])));
          oe[o] = partner_i32<S>(oe[o]);
        };
        if (step & 1) exchange(std::integral_constant<int, 1>{});
        else if (step & 2) exchange(std::integral_constant<int, 2>{});
        else if (step & 4) exchange(std::integral_constant<int, 4>{});
        else if (step & 8) exchange(std::integral_constant<int, 8>{});
#pragma unroll
        for (int sl = 0; sl < kBlockedSlots; ++sl) {
          if (sl * G >= topk) continue;
          place[sl] += (ok[o] > key[sl] || (ok[o] == key[sl] && oe[o] < sel_i[sl])) ? 1 : 0;
        }
      }
    }
    if constexpr (G > 1) top_key = max(top_key, static_cast<unsigned>(partner_i32<1>(static_cast<int>(top_key))));
    if constexpr (G > 2) top_key = max(top_key, static_cast<unsigned>(partner_i32<2>(static_cast<int>(top_key))));
    if constexpr (G > 4) top_key = max(top_key, static_cast<unsigned>(partner_i32<4>(static_cast<int>(top_key))));
    if constexpr (G > 8) top_key = max(top_key, static_cast<unsigned>(partner_i32<8>(static_cast<int>(top_key))));
    top_v = key_float(top_key);
  }

  // top-1 first: with renormalised weights it is all the softmax statistics there are
  float m = top_v;
  float denom;
  if (RANKED && renorm) {
    float first = -INFINITY;  // (the first winner of a class refilled above is the packed order's, not always the largest)
#pragma unroll
    for (int sl = 0; sl < kBlockedSlots; ++sl)
      if (sl * G + g < topk && place[sl] == 0) first = sel_v[sl];
    m = group_max<G>(first);
    denom = 0.f;
    for (int r = 0; r < topk; ++r) {  // the one lane and slot that holds rank r adds it, the others zeros
      float term = 0.f;
#pragma unroll
      for (int sl = 0; sl < kBlockedSlots; ++sl)
        if (sl * G + g < topk && place[sl] == r) term = __expf(sel_v[sl] - m);
      denom += group_sum<G>(term);
    }
  } else if (renorm) {
    denom = 0.f;
#pragma unroll
    for (int sl = 0; sl < kBlockedSlots; ++sl)
      if (sl * G < topk) denom += group_sum<G>((live && sl * G + g < topk) ? __expf(sel_v[sl] - m) : 0.f);
  } else {
    m = v[0];
    float s = (v[0] == -INFINITY) ? 0.f : 1.f;
#pragma unroll
    for (int i = 1; i < VPL; ++i) {
      if (v[i] == -INFINITY) continue;
      const float mn = fmaxf(m, v[i]);
      s = (m == -INFINITY ? 0.f : s * __expf(m - mn)) + __expf(v[i] - mn);
      m = mn;
    }
    group_online_softmax<G>(m, s);
    denom = s;
  }
  if (live) {
#pragma unroll
    for (int sl = 0; sl < kBlockedSlots; ++sl) {
      const int r = sl * G + g;
      if (r < topk) {
        w_row[place[sl]] = __expf(sel_v[sl] - m) / denom;
        id_row[place[sl]] = sel_i[sl];
      }
    }
  }
}

}  // namespace
}  // namespace fr
