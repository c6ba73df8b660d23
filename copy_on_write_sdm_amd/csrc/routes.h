// Product-key route selection on the device: the producer of the decode
// step's write and read routes (copy_on_write_sdm/sdm.py:96-159).  Shared by
// routes.hip (cowsdm_product_key_routes) and controller.hip (the controller's
// prepare kernel selects its tokens' routes itself).
//
// One wave per route row.  A row holds 2*root scores (root = sqrt(N)); the
// two halves are shortlisted independently to their top `sub` = min(k, root)
// entries, the sub*sub pair sums are ranked, the best min(k, sub*sub) pairs
// become slots (first * root + second), sorted by slot, and their scores go
// through a softmax.
//
// Selection ranks every candidate at once: a candidate's key is its score in
// order-preserving bits above its inverted position, so keys are unique and
// "higher key" means "selected first" (higher score, then lower position;
// torch.topk leaves the order of equal scores open, and only a tie at the
// selection boundary can change which slot is selected).  Each lane counts
// the keys of the wave, broadcast one at a time with readlane, that beat its
// own; a candidate whose rank is below the count writes itself to LDS at its
// rank.  All inputs must be finite.

#pragma once

#include <algorithm>
#include <type_traits>

#include "common.h"

namespace cowsdm_impl {

constexpr int kRouteWaves = 4;                 // rows per workgroup
constexpr int kRouteMaxRoot = 1024;            // N <= 2^20
constexpr int kRouteMaxSelected = 32;          // pair-stage candidates <= 128

// -0.0 is added to +0.0 first so that equal scores get equal bits.
__device__ __forceinline__ uint64_t route_key(float v, int pos) {
  uint32_t bits = __float_as_uint(v + 0.0f);
  bits = (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
  return (static_cast<uint64_t>(bits) << 32) | static_cast<uint32_t>(~pos);
}

// rank[j] = number of keys in the wave (J per lane, absent ones 0) above key[j];
// lanes from LANES on hold absent keys only (every present key is above 0),
// so only the first LANES are broadcast
template <int J, int LANES = kWave>
__device__ __forceinline__ void wave_rank(const uint64_t (&key)[J], int (&rank)[J]) {
#pragma unroll
  for (int j = 0; j < J; ++j) rank[j] = 0;
#pragma unroll
  for (int j2 = 0; j2 < J; ++j2) {
    const uint32_t lo = static_cast<uint32_t>(key[j2]);
    const uint32_t hi = static_cast<uint32_t>(key[j2] >> 32);
    auto count = [&](int u) {
      const uint64_t other =
          (static_cast<uint64_t>(static_cast<uint32_t>(rl(static_cast<int>(hi), u))) << 32) |
          static_cast<uint32_t>(rl(static_cast<int>(lo), u));
#pragma unroll
      for (int j = 0; j < J; ++j) rank[j] += other > key[j] ? 1 : 0;
    };
    if constexpr (J <= 4) {
#pragma unroll
      for (int u = 0; u < LANES; ++u) count(u);   // lane selects as immediates
    } else {
      for (int u = 0; u < LANES; ++u) count(u);
    }
  }
}

// LDS written by lanes of one wave and read by others of the same wave
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Lane t < count ends with the t-th best (value, position) of the wave's
// candidates (pos < 0: absent).  stage_val/stage_pos hold kRouteMaxSelected
// entries of this wave.
template <int J, int LANES = kWave>
__device__ __forceinline__ void wave_top(const float (&val)[J], const int (&pos)[J], int count,
                                         int lane, float* stage_val, int* stage_pos,
                                         float& top_val, int& top_pos) {
  uint64_t key[J];
  int rank[J];
#pragma unroll
  for (int j = 0; j < J; ++j) key[j] = pos[j] >= 0 ? route_key(val[j], pos[j]) : 0;
  wave_rank<J, LANES>(key, rank);
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (pos[j] >= 0 && rank[j] < count) {
      stage_val[rank[j]] = val[j];
      stage_pos[rank[j]] = pos[j];
    }
  wave_lds_sync();
  top_val = lane < count ? stage_val[lane] : -__builtin_inff();
  top_pos = lane < count ? stage_pos[lane] : 0;
  wave_lds_sync();
}

// wave_top for J > 1 (root > 64, every lane holds at least one entry).  The
// count-th largest lane maximum T bounds the selection: count lane maxima
// are >= T, so an entry below T ranks at least count and is never selected.
// The entries >= T (about count + count/4 for random scores) are compacted
// into one per lane and ranked once; if more than 64 remain (many equal
// scores), every entry is ranked.
template <int J>
__device__ __forceinline__ void wave_top_pruned(const float (&val)[J], const int (&pos)[J],
                                                int count, int lane, float* stage_val,
                                                int* stage_pos, float* pool_val, int* pool_pos,
                                                float& top_val, int& top_pos) {
  uint64_t key[J];
  uint64_t best[1] = {0};
#pragma unroll
  for (int j = 0; j < J; ++j) {
    key[j] = pos[j] >= 0 ? route_key(val[j], pos[j]) : 0;
    best[0] = key[j] > best[0] ? key[j] : best[0];
  }
  int best_rank[1];
  wave_rank<1>(best, best_rank);   // 64 unique lane maxima: ranks 0..63
  const uint64_t at = __ballot(best_rank[0] == count - 1);
  const int holder = at ? __builtin_ctzll(at) : 0;
  const uint64_t bound =
      (static_cast<uint64_t>(static_cast<uint32_t>(rl(static_cast<int>(best[0] >> 32), holder)))
       << 32) |
      static_cast<uint32_t>(rl(static_cast<int>(static_cast<uint32_t>(best[0])), holder));
  uint64_t mask[J];
  int total = 0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    mask[j] = __ballot(pos[j] >= 0 && key[j] >= bound);
    total += __popcll(mask[j]);
  }
  if (total > kWave) {
    wave_top<J>(val, pos, count, lane, stage_val, stage_pos, top_val, top_pos);
    return;
  }
  const uint64_t below = (uint64_t{1} << lane) - 1;
  int base = 0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if ((mask[j] >> lane) & 1) {
      const int slot = base + __popcll(mask[j] & below);   // < total <= 64
      pool_val[slot] = val[j];
      pool_pos[slot] = pos[j];
    }
    base += __popcll(mask[j]);
  }
  wave_lds_sync();
  float one_val[1] = {lane < total ? pool_val[lane] : -__builtin_inff()};
  int one_pos[1] = {lane < total ? pool_pos[lane] : -1};
  wave_lds_sync();
  wave_top<1>(one_val, one_pos, count, lane, stage_val, stage_pos, top_val, top_pos);
}

// Row `row` of `projected` ([rows, 2 * root]) by the calling wave: its
// final_k routes (weights and slots, sorted by slot) at row * final_k.
// stage_val/stage_pos (kRouteMaxSelected entries) and pool_val/pool_pos
// (kWave entries) are this wave's LDS.
template <int J, int M>
__device__ __forceinline__ void product_key_route_row(
    const float* __restrict__ projected, int64_t row, int root, int sub, int final_k,
    float* __restrict__ weights, int64_t* __restrict__ indices, float* stage_val,
    int* stage_pos, float* pool_val, int* pool_pos) {
  const int lane = static_cast<int>(threadIdx.x) % kWave;
  const float* first = projected + row * 2 * root;
  const float* second = first + root;

  // 1. shortlist each half: entry e = lane + 64 j
  float fv[J], sv[J];
  int fp[J], sp[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int e = lane + kWave * j;
    const bool in = e < root;
    fv[j] = in ? first[e] : -__builtin_inff();
    sv[j] = in ? second[e] : -__builtin_inff();
    fp[j] = in ? e : -1;
    sp[j] = in ? e : -1;
  }
  float first_val, second_val;
  int first_idx, second_idx;
  if constexpr (J > 1) {
    wave_top_pruned<J>(fv, fp, sub, lane, stage_val, stage_pos, pool_val,
                       pool_pos, first_val, first_idx);
    wave_top_pruned<J>(sv, sp, sub, lane, stage_val, stage_pos, pool_val,
                       pool_pos, second_val, second_idx);
  } else if (root <= 16) {
    // root <= 64: entries only in lanes below root
    wave_top<J, 16>(fv, fp, sub, lane, stage_val, stage_pos, first_val, first_idx);
    wave_top<J, 16>(sv, sp, sub, lane, stage_val, stage_pos, second_val, second_idx);
  } else if (root <= 32) {
    wave_top<J, 32>(fv, fp, sub, lane, stage_val, stage_pos, first_val, first_idx);
    wave_top<J, 32>(sv, sp, sub, lane, stage_val, stage_pos, second_val, second_idx);
  } else {
    wave_top<J>(fv, fp, sub, lane, stage_val, stage_pos, first_val, first_idx);
    wave_top<J>(sv, sp, sub, lane, stage_val, stage_pos, second_val, second_idx);
  }

  // 2. pair c = a * sub + b scores first_val[a] + second_val[b].  Every pair
  // (a', b') <= (a, b) scores at least as high (float addition is monotone)
  // and has a lower position, so (a, b) ranks at least (a+1)(b+1) - 1 and can
  // be selected only if (a+1)(b+1) <= final_k: at most
  // sum_a min(sub, final_k / (a+1)) candidates, enumerated a-major.
  float cv[M];
  int cp[M];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    int rest = lane + kWave * m, a = -1, b = 0;
    for (int t = 0; t < sub; ++t) {
      const int per = min(sub, final_k / (t + 1));
      if (a < 0) {
        if (rest < per) { a = t; b = rest; } else { rest -= per; }
      }
    }
    const bool in = a >= 0;
    const float va = __shfl(first_val, in ? a : 0, kWave);
    const float vb = __shfl(second_val, b, kWave);
    cv[m] = in ? va + vb : -__builtin_inff();
    cp[m] = in ? a * sub + b : -1;
  }
  float score;
  int pair;
  wave_top<M>(cv, cp, final_k, lane, stage_val, stage_pos, score, pair);

  // 3. slot of each selected pair, its rank by slot, softmax of the scores
  const bool mine = lane < final_k;
  const int a = mine ? pair / sub : 0;
  const int b = mine ? pair - a * sub : 0;
  const int fa = __shfl(first_idx, a, kWave);
  const int sb = __shfl(second_idx, b, kWave);
  const int64_t slot = static_cast<int64_t>(fa) * root + sb;
  int rank = 0;
  for (int u = 0; u < final_k; ++u) {
    const int64_t other = static_cast<int64_t>(rl(static_cast<int>(slot), u));
    rank += other < slot ? 1 : 0;
  }
  float mx = mine ? score : -__builtin_inff();
  for (int o = kWave / 2; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
  const float e = mine ? expf(score - mx) : 0.0f;
  float total = e;
  for (int o = kWave / 2; o > 0; o >>= 1) total += __shfl_xor(total, o, kWave);
  if (mine) {
    weights[row * final_k + rank] = e / total;
    indices[row * final_k + rank] = slot;
  }
}

// ---- One lane per row (sqrt(N) <= 32) --------------------------------------
//
// The same selection with every row in one lane's registers: sorting
// networks over 64-bit keys, no cross-lane operation, no LDS.  What bounds
// the selection is its instructions, not bytes: at N = 256, K = 16 a wave
// per row issues 2,180 for one row, most of them to broadcast keys, a lane
// per row 2,300 for 64 rows.  A compare-exchange of two keys is one
// v_max_f64 and one v_min_f64, at the rate of 32-bit operations on this
// device, so keys are doubles.  131,072 rows (wave per row -> lane per row):
// N = 256 K = 16 166 -> 17 us, K = 4 127 -> 5.4; N = 1,024 K = 32
// 445 -> 30 us, K = 24 423 -> 69.

// A score as a positive finite double in route_key's order: the score's
// order-preserving bits below a fixed exponent bit (infinities and NaN
// patterns are ordered doubles like the others), with 29 bits left below
// them for `code`, which breaks ties.
__device__ __forceinline__ double route_pack(float v, uint32_t code) {
  const uint32_t bits = __float_as_uint(v);
  const uint32_t order = bits ^ (static_cast<uint32_t>(static_cast<int32_t>(bits) >> 31) |
                                 0x80000000u);
  return __hiloint2double(static_cast<int>((order >> 3) | 0x20000000u),
                          static_cast<int>((order << 29) | code));
}

__device__ __forceinline__ float route_score(double key) {
  const uint32_t order = (static_cast<uint32_t>(__double2hiint(key)) << 3) |
                         (static_cast<uint32_t>(__double2loint(key)) >> 29);
  return __uint_as_float(order ^ (~static_cast<uint32_t>(static_cast<int32_t>(order) >> 31) |
                                  0x80000000u));
}

__device__ __forceinline__ uint32_t route_code(double key) {
  return static_cast<uint32_t>(__double2loint(key)) & 0x1fffffffu;
}

constexpr double kRouteAbsent = 0.0;   // below every route_pack key

// v_max_f64 and v_min_f64 themselves: the keys are never NaN, and fmax would
// quiet each operand first.
__device__ __forceinline__ double key_max(double a, double b) {
#ifdef __HIP_DEVICE_COMPILE__
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
#else
  return a > b ? a : b;
#endif
}

__device__ __forceinline__ double key_min(double a, double b) {
#ifdef __HIP_DEVICE_COMPILE__
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
#else
  return a < b ? a : b;
#endif
}

__device__ __forceinline__ void sort_pair(double& high, double& low) {
  const double h = key_max(high, low);
  low = key_min(high, low);
  high = h;
}

// x, bitonic, into descending order
template <int N>
__device__ __forceinline__ void bitonic_clean(double* x) {
#pragma unroll
  for (int d = N / 2; d > 0; d /= 2) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if ((i & d) == 0) sort_pair(x[i], x[i + d]);
    }
  }
}

// Batcher's odd-even merge sort (K. E. Batcher, Sorting networks and their
// applications, 1968), descending
template <int N>
__device__ __forceinline__ void network_sort(double* x) {
#pragma unroll
  for (int p = 1; p < N; p *= 2) {
#pragma unroll
    for (int k = p; k >= 1; k /= 2) {
#pragma unroll
      for (int j = k % p; j + k < N; j += 2 * k) {
#pragma unroll
        for (int i = 0; i < k; ++i) {
          if (i + j + k < N && (i + j) / (2 * p) == (i + j + k) / (2 * p)) {
            sort_pair(x[i + j], x[i + j + k]);
          }
        }
      }
    }
  }
}

// top (descending) becomes the K highest of top and `other` (descending, of
// length M <= K), descending
template <int K, int M>
__device__ __forceinline__ void merge_top(double* top, const double* other) {
#pragma unroll
  for (int i = 0; i < M; ++i) top[K - 1 - i] = key_max(top[K - 1 - i], other[i]);
  bitonic_clean<K>(top);
}

// The K highest of x[0 .. N), descending, in x[0 .. K).
template <int N, int K>
__device__ __forceinline__ void network_top(double* x) {
  if constexpr (N <= K) {
    network_sort<N>(x);
  } else {
    network_top<N / 2, K>(x);
    network_top<N / 2, K>(x + N / 2);
    merge_top<K, K>(x, x + N / 2);
  }
}

constexpr int route_pow2(int n) {
  int p = 1;
  while (p < n) p *= 2;
  return p;
}

// Row `projected` ([2 * root], root <= NR) of the calling lane: its final_k
// <= KP routes at weights and indices (`on` false: read, not written).
// FULL: root == NR, sub == min(KP, NR), final_k == KP, and `projected` is
// 16-byte aligned.
template <int NR, int KP, bool FULL>
__device__ __forceinline__ void product_key_route_lane(bool on,
                                                       const float* __restrict__ projected,
                                                       int root, int sub, int final_k,
                                                       float* __restrict__ weights,
                                                       int64_t* __restrict__ indices) {
  constexpr int KL = KP < NR ? KP : NR;   // entries of a shortlist
  if constexpr (FULL) {
    root = NR;
    sub = KL;
    final_k = KP;
  }
  // 1. shortlists: score and index of the sub best of each half; the codes
  // of lower positions are higher
  float fv[KL], sv[KL];
  uint32_t fi[KL], si[KL];
  auto shortlist = [&](const float* half, float (&val)[KL], uint32_t (&idx)[KL])
      __attribute__((always_inline)) {
    float v[NR];
    double x[NR];
    if constexpr (FULL) {
#pragma unroll
      for (int e = 0; e < NR; e += 4) {
        const float4 q = *reinterpret_cast<const float4*>(half + e);
        v[e] = q.x;
        v[e + 1] = q.y;
        v[e + 2] = q.z;
        v[e + 3] = q.w;
      }
    } else {
#pragma unroll
      for (int e = 0; e < NR; ++e) v[e] = half[e < root ? e : 0];
    }
#pragma unroll
    for (int e = 0; e < NR; ++e) {
      // -0.0 + 0.0 is +0.0: equal scores get equal keys
      x[e] = route_pack(v[e] + 0.0f, static_cast<uint32_t>(NR - 1 - e));
      if (!FULL && e >= root) x[e] = kRouteAbsent;
    }
    network_top<NR, KL>(x);
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      val[i] = route_score(x[i]);
      idx[i] = NR - 1 - route_code(x[i]);
    }
  };
  shortlist(projected, fv, fi);
  shortlist(projected + root, sv, si);
#pragma unroll
  for (int i = 0; i < KL; ++i) fi[i] *= static_cast<uint32_t>(root);   // its first slot

  // 2. the pairs with (a+1)(b+1) <= KP hold the KP best (see
  // product_key_route_row).  Along a row or a column of them the keys
  // descend, so they are merged as sorted lists, row r from (r, r) on and
  // column r from (r + 1, r) on; what lies at r >= 2 is sorted at once.  A
  // key's code: its position, first a, then b, inverted; below it the slot.
  // A sum of two of these scores is never -0.0.
  auto pair = [&](int a, int b) __attribute__((always_inline)) {
    const uint32_t code = (static_cast<uint32_t>(KL * KL - 1 - (a * KL + b)) << 12) |
                          (fi[a] + si[b]);
    const double key = route_pack(fv[a] + sv[b], code);
    return FULL || (a < sub && b < sub) ? key : kRouteAbsent;
  };
  double top[KP];
#pragma unroll
  for (int b = 0; b < KP; ++b) top[b] = b < KL ? pair(0, b) : kRouteAbsent;
  auto merge_line = [&](auto row, auto by_row) __attribute__((always_inline)) {
    constexpr int r = decltype(row)::value;
    constexpr bool R = decltype(by_row)::value;
    constexpr int first = R ? r : r + 1;
    constexpr int end = KP / (r + 1) < KL ? KP / (r + 1) : KL;
    if constexpr (end > first) {
      double list[end - first];
#pragma unroll
      for (int i = first; i < end; ++i) list[i - first] = R ? pair(r, i) : pair(i, r);
      merge_top<KP, end - first>(top, list);
    }
  };
  using std::integral_constant;
  merge_line(integral_constant<int, 0>{}, std::false_type{});
  merge_line(integral_constant<int, 1>{}, std::true_type{});
  merge_line(integral_constant<int, 1>{}, std::false_type{});
  constexpr int tail = [] {
    int n = 0;
    for (int a = 2; a < KL; ++a) {
      for (int b = 2; b < KL; ++b) n += (a + 1) * (b + 1) <= KP ? 1 : 0;
    }
    return n;
  }();
  if constexpr (tail > 0) {
    constexpr int TP = route_pow2(tail);
    double rest[TP];
#pragma unroll
    for (int i = tail; i < TP; ++i) rest[i] = kRouteAbsent;
    int n = 0;
#pragma unroll
    for (int a = 2; a < KL; ++a) {
#pragma unroll
      for (int b = 2; b < KL; ++b) {
        if ((a + 1) * (b + 1) <= KP) rest[n++] = pair(a, b);
      }
    }
    network_sort<TP>(rest);
    merge_top<KP, TP>(top, rest);
  }

  // 3. softmax of the final_k best, summed in product_key_route_row's order
  // (lane i there with lanes i ^ 16, i ^ 8, ...), then sorted by slot
  const float mx = route_score(top[0]);
  constexpr int EP = KP < 2 ? 2 : KP;
  float e[EP], part[EP];
#pragma unroll
  for (int i = 0; i < KP; ++i) {
    e[i] = FULL || i < final_k ? expf(route_score(top[i]) - mx) : 0.0f;
    part[i] = e[i];
  }
#pragma unroll
  for (int d = KP / 2; d > 0; d /= 2) {
#pragma unroll
    for (int i = 0; i < d; ++i) part[i] = part[i] + part[i + d];
  }
  const float total = part[0];
#pragma unroll
  for (int i = 0; i < KP; ++i) {
    // ascending slots from the highest key down, routes past final_k last
    const uint32_t slot = route_code(top[i]) & 0xfffu;
    top[i] = __hiloint2double(
        static_cast<int>(0x20000fffu - (FULL || i < final_k ? slot : 0x1000u)),
        __float_as_int(e[i] / total));
  }
  network_sort<KP>(top);
  if (on) {
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      if (FULL || i < final_k) {
        weights[i] = __int_as_float(__double2loint(top[i]));
        indices[i] = 0x20000fffu - static_cast<uint32_t>(__double2hiint(top[i]));
      }
    }
  }
}

constexpr int kRouteLaneRoot = 32;
constexpr int kRouteLaneRows = 4096;   // see cowsdm_product_key_routes

// ---- One wave per row, few routes (sqrt(N) <= 32, K <= 16) ------------------
//
// product_key_route_row for a decode step's few rows, where the latency of
// one row is what counts: the same keys and the same pairs as the lane form,
// sorted across lanes.  A step of a bitonic sort is a DPP move of the key and
// a v_max_f64 / v_min_f64 (only the three moves between rows of 16 lanes go
// through ds_bpermute), so the selection is about 400 instructions without
// LDS staging, against about 900 and a dozen waits on LDS.
// 64 rows, launch included: N = 256 K = 16 6.2 -> 3.5 us, K = 4 4.4 -> 3.4,
// N = 1,024 K = 16 6.3 -> 3.3, N = 400 K = 8 5.2 -> 3.4.

// The key of lane ^ 1, ^ 2, ^ 4, ^ 8 (STEP 1, 2, 4, 8) or of the mirrored lane
// of 4, 8 or 16 (STEP 3, 7, 15).
template <int STEP>
__device__ __forceinline__ int lane_partner(int x) {
  if constexpr (STEP == 4) {
    // lanes 0-3 and 8-11 of a row from four above, the others from four below
    const int up = __builtin_amdgcn_update_dpp(0, x, 0x104, 0xf, 0x5, true);
    return __builtin_amdgcn_update_dpp(up, x, 0x114, 0xf, 0xa, false);
  } else {
    constexpr int ctrl = STEP == 1    ? 0xB1    // quad_perm [1,0,3,2]
                         : STEP == 2  ? 0x4E    // quad_perm [2,3,0,1]
                         : STEP == 3  ? 0x1B    // quad_perm [3,2,1,0]
                         : STEP == 7  ? 0x141   // row_half_mirror
                         : STEP == 8  ? 0x128   // row_ror:8
                                      : 0x140;  // row_mirror
    return __builtin_amdgcn_update_dpp(0, x, ctrl, 0xf, 0xf, true);
  }
}

// One step of a descending sort within rows of 16 lanes: the lane whose
// highest bit of STEP is 0 keeps the higher key.
template <int STEP>
__device__ __forceinline__ double row_step(double key, int lane) {
  constexpr int bit = STEP == 3 ? 2 : STEP == 7 ? 4 : STEP == 15 ? 8 : STEP;
  const double other = __hiloint2double(lane_partner<STEP>(__double2hiint(key)),
                                        lane_partner<STEP>(__double2loint(key)));
  const double high = key_max(key, other), low = key_min(key, other);
  return (lane & bit) == 0 ? high : low;
}

// a bitonic row into descending order
__device__ __forceinline__ double row_clean(double key, int lane) {
  key = row_step<8>(key, lane);
  key = row_step<4>(key, lane);
  key = row_step<2>(key, lane);
  return row_step<1>(key, lane);
}

__device__ __forceinline__ double row_sort(double key, int lane) {
  key = row_step<1>(key, lane);
  key = row_step<3>(key, lane);
  key = row_step<1>(key, lane);
  key = row_step<7>(key, lane);
  key = row_step<2>(key, lane);
  key = row_step<1>(key, lane);
  key = row_step<15>(key, lane);
  key = row_step<4>(key, lane);
  key = row_step<2>(key, lane);
  return row_step<1>(key, lane);
}

__device__ __forceinline__ double lane_key(double key, int lane) {
  return __hiloint2double(__builtin_amdgcn_ds_bpermute(4 * lane, __double2hiint(key)),
                          __builtin_amdgcn_ds_bpermute(4 * lane, __double2loint(key)));
}

// Two descending rows, `flip` ^ lane apart (31 or 63: the mirrored lanes of
// neighbouring rows or pairs of rows), into the 16 highest of both,
// descending, in either.
__device__ __forceinline__ double row_merge(double key, int lane, int flip) {
  return row_clean(key_max(key, lane_key(key, lane ^ flip)), lane);
}

// Row `row` of `projected` by the calling wave; root <= 32, final_k <= 16.
__device__ __forceinline__ void product_key_route_row_sorted(
    const float* __restrict__ projected, int64_t row, int root, int sub, int final_k,
    float* __restrict__ weights, int64_t* __restrict__ indices) {
  const int lane = static_cast<int>(threadIdx.x) % kWave;
  const float* const first = projected + row * 2 * root;
  // 1. the halves' shortlists: sqrt(N) <= 16 the first half in the lanes of
  // row 0 and the second in those of row 1, above that two rows each
  const bool wide = root > 16;
  const int per = wide ? 32 : 16;          // lanes of a half
  const int e = lane % per, half = lane / per;
  const bool in = half < 2 && e < root;
  const float v = first[in ? half * root + e : 0];
  double key = in ? route_pack(v + 0.0f, static_cast<uint32_t>(31 - e)) : kRouteAbsent;
  key = row_sort(key, lane);
  if (wide) key = row_merge(key, lane, 31);

  // 2. the pairs with (a+1)(b+1) <= 16, a row or a column of them to a row
  // of lanes where it fills one: (0, b); (a, 0); (1, b) and (a, 1); the rest
  const int i = lane % 16;
  int a = 0, b = i;
  if (lane >= 48) {
    a = i < 3 ? 2 : i == 4 ? 4 : 3;        // (2,2) (2,3) (2,4) (3,2) (4,2) (3,3)
    b = i < 3 ? i + 2 : i == 5 ? 3 : 2;
    if (i > 5) b = 16;
  } else if (lane >= 32) {
    a = i < 7 ? 1 : i - 5;                 // (1,1) .. (1,7), (2,1) .. (7,1)
    b = i < 7 ? i + 1 : 1;
    if (i > 12) b = 16;
  } else if (lane >= 16) {
    a = i + 1;                             // (1,0) .. (15,0)
    b = 0;
  }
  const double fk = lane_key(key, a % 16), sk = lane_key(key, per + b % 16);
  const uint32_t slot = (31 - route_code(fk)) * static_cast<uint32_t>(root) +
                        (31 - route_code(sk));
  const uint32_t code = (static_cast<uint32_t>(255 - (a * 16 + b)) << 12) | slot;
  double top = a < sub && b < sub ? route_pack(route_score(fk) + route_score(sk), code)
                                  : kRouteAbsent;
  top = row_merge(row_merge(row_sort(top, lane), lane, 31), lane, 63);

  // 3. every row of lanes holds the 16 best: softmax of the first final_k,
  // summed in product_key_route_row's order, then each one's place by slot
  const float score = route_score(top);
  const float mx = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(score)));
  const bool mine = i < final_k;
  const float ex = mine ? expf(score - mx) : 0.0f;
  float total = ex;
  total += __int_as_float(lane_partner<8>(__float_as_int(total)));
  total += __int_as_float(lane_partner<4>(__float_as_int(total)));
  total += __int_as_float(lane_partner<2>(__float_as_int(total)));
  total += __int_as_float(lane_partner<1>(__float_as_int(total)));
  const int own = mine ? static_cast<int>(route_code(top) & 0xfffu) : 0x1000 + i;
  int rank = 0;
#define COWSDM_ROUTE_RANK(r) \
  rank += __builtin_amdgcn_update_dpp(0, own, 0x120 + r, 0xf, 0xf, true) < own ? 1 : 0
  COWSDM_ROUTE_RANK(1);
  COWSDM_ROUTE_RANK(2);
  COWSDM_ROUTE_RANK(3);
  COWSDM_ROUTE_RANK(4);
  COWSDM_ROUTE_RANK(5);
  COWSDM_ROUTE_RANK(6);
  COWSDM_ROUTE_RANK(7);
  COWSDM_ROUTE_RANK(8);
  COWSDM_ROUTE_RANK(9);
  COWSDM_ROUTE_RANK(10);
  COWSDM_ROUTE_RANK(11);
  COWSDM_ROUTE_RANK(12);
  COWSDM_ROUTE_RANK(13);
  COWSDM_ROUTE_RANK(14);
  COWSDM_ROUTE_RANK(15);
#undef COWSDM_ROUTE_RANK
  if (lane < 16 && mine) {
    weights[row * final_k + rank] = ex / total;
    indices[row * final_k + rank] = own;
  }
}

// Whether a row's routes are selected by product_key_route_row_sorted when a
// wave has the row (the pairs' rows of lanes hold 16 of a shortlist).
inline bool route_row_sorted(int root, int final_k) { return root <= 32 && final_k <= 16; }

// The selection's shape for N slots and `selected` routes a row: root =
// sqrt(N), sub = min(selected, root) entries shortlisted per half, final_k =
// min(selected, sub * sub) routes; 0, or the error of
// cowsdm_product_key_routes (recorded by fail()).
inline int32_t route_geometry(int64_t slots, int64_t selected, int& root_out, int& sub_out,
                              int& final_out) {
  int64_t root = 0;
  while ((root + 1) * (root + 1) <= slots) ++root;
  if (slots < 1 || root * root != slots)
    return fail(-1, "slot count and product-key projection do not match");
  if (selected < 1 || selected > slots)
    return fail(-1, "selected product keys must be between one and slots");
  if (root > kRouteMaxRoot)
    return fail(-2, "product_key_routes: sqrt(slots) <= %d on the HIP path (got %lld)",
                kRouteMaxRoot, static_cast<long long>(root));
  const int64_t sub = selected < root ? selected : root;
  if (sub > kRouteMaxSelected)
    return fail(-2, "product_key_routes: min(selected, sqrt(slots)) <= %d on the HIP path "
                "(got %lld)", kRouteMaxSelected, static_cast<long long>(sub));
  const int64_t final_k = selected < sub * sub ? selected : sub * sub;
  if (final_k > kRouteMaxSelected)
    return fail(-2, "product_key_routes: at most %d routes per row on the HIP path (got %lld)",
                kRouteMaxSelected, static_cast<long long>(final_k));
  root_out = static_cast<int>(root);
  sub_out = static_cast<int>(sub);
  final_out = static_cast<int>(final_k);
  return 0;
}

// Candidates of the pair stage over 64: the selection's M (1 or 2).
inline int route_pair_m(int sub, int final_k) {
  int pairs = 0;   // at most 119 for final_k <= 32
  for (int t = 0; t < sub; ++t) pairs += std::min(sub, final_k / (t + 1));
  return pairs <= kWave ? 1 : 2;
}

}  // namespace cowsdm_impl
