// The token-serial SDM recurrence over sparse routes: a layer's prefill
// (copy_on_write_sdm/sdm.py:464-529 as SparseDeltaMemory.forward runs it,
// sdm.py:1136-1262) straight from the controller's outputs, token-major rows
// (b * T + t) * H + h, without the dense route vectors that recurrence.hip
// takes.
//
// Bound: the serial chain of a token, not bytes (per token and bank 2W + R
// rows of D floats, all in LDS): the load of the written rows, decay, the
// retrieval's sum over the write routes, delta, update, store.  So the whole
// table of a (bank, 32 columns) stays in LDS for the sequence and the chain
// is kept short:
// * a wave owns 8 columns and 8 lanes share a column: lane g of a column
//   takes the write routes g, g + 8, ... and the read routes likewise, so a
//   token is one LDS load per lane for W <= 8 and two for R <= 16, and both
//   sums are three DPP adds within the 8 lanes;
// * LDS operations of one wave complete in order, so the loads of the next
//   token's rows are issued right behind this token's store, without a wait
//   or a barrier, and the reading of a token is summed while the next
//   token's rows are on their way;
// * routes, gates and values of a chunk of tokens are staged in LDS by four
//   producer waves, one chunk ahead and loaded two ahead: route entries as
//   (byte offset of the row, weight), exp(forget) taken there, so the chain
//   holds no conversion and waits on no global load.
// A bank's column blocks go to one XCD (its L2 then serves the staging of
// all of them).
//
// At B = 64, T = 2,048, N = 256, D = 128, W = 4, R = 16 (131,072 tokens):
// 207 us, 0.10 us per token of a bank, where the dense route vectors and the
// dense-route kernel took 445 + 1,858 us; one bank alone takes 193 us.
//
// Values that are not finite spread as in the dense sums, where a zero route
// times such a row, or times such a delta, is NaN.  Every lane keeps 0 * (each
// row it wrote), 0 or NaN, and starts its partial sums from it, which marks
// the columns that met one; at the end of the sequence a wave takes its marked
// columns again from the first token on, one token after the other with all
// rows looked over, until everything in them is NaN (exact_columns).

#include <type_traits>

#include "lds_recurrence.h"

namespace cowsdm_impl {

constexpr int kRrMaxRoutes = 32;

struct RrParams {
  int64_t banks, time, heads;
  int slots, width, writes, reads, blocks;   // blocks: column blocks per bank
  int chunk_shift;                           // log2 of the tokens per chunk
  const float* m0;              // [H, N, D]
  const int64_t* write_idx;     // [B * T * H, W]
  const float* write_w;
  const float* values;          // [B * T * H, D]
  const float* gate;            // [B * T * H]: input gate, also the erase gate
  const float* forget;          // [B * T * H]
  const int64_t* read_idx;      // [B * T * H, R]
  const float* read_w;
  float* readings;              // [B * T * H, D]
  float* final_memory;          // [B * H, N, D]
};

// A wave's columns (of `bad`: the same in a column's lanes) of a bank's table
// and readings in the dense sums' own terms, from the initial memory `m0` on:
// as the kernel below computes them, but the rows that a sum has no route for,
// or a zero one, are looked over for values that are not finite.  Tokens are
// taken until every row of these columns is NaN: what follows is NaN, and
// marked columns already read so.  `mine`: the column's table.
template <int WPL, int RPL>
__device__ __forceinline__ void exact_columns(const RrParams& P, char* mine, int64_t b, int64_t h,
                                              int d, int g, bool bad) {
  const int N = P.slots, D = P.width;
  const bool in = d < D;
  const float* const m0 = P.m0 + h * N * static_cast<int64_t>(D);
  auto row = [&](int n) __attribute__((always_inline)) {
    return reinterpret_cast<float*>(mine + n * kRrRowBytes);
  };
  for (int n = g; n <= N; n += kRrGroups) {
    if (bad) *row(n) = in && n < N ? m0[static_cast<int64_t>(n) * D + d] : 0.0f;
  }
  // 0, or NaN if a row of the column is not finite
  auto look_over = [&]() __attribute__((always_inline)) {
    float z = 0.0f;
#pragma unroll 4
    for (int n = g; n < N; n += kRrGroups) z = __builtin_fmaf(*row(n), 0.0f, z);
    return z;
  };
  for (int64_t t = 0; t < P.time; ++t) {
    const int64_t at = (b * P.time + t) * P.heads + h;
    // the lane's routes; none, or one past the table, has weight 0 and row N
    auto route = [&](const int64_t* idx, const float* w, int k, int i, float& weight)
        __attribute__((always_inline)) {
      const int j = g + kRrGroups * i;
      const int64_t n = j < k ? idx[at * k + j] : -1;
      const bool on = n >= 0 && n < N;
      weight = on ? w[at * k + j] : 0.0f;
      return row(on ? static_cast<int>(n) : N);
    };
    const float alpha = expf(P.forget[at]), gate = P.gate[at];
    const float gv = gate * (in ? P.values[at * D + d] : 0.0f);
    float* to[WPL];
    float ww[WPL], cur[WPL];
#pragma unroll
    for (int i = 0; i < WPL; ++i) {
      to[i] = route(P.write_idx, P.write_w, P.writes, i, ww[i]);
      cur[i] = *to[i] * alpha;
    }
#pragma unroll
    for (int i = 0; i < WPL; ++i) {
      if (bad && ww[i] != 0.0f) *to[i] = 0.0f;   // out of the others' sight
    }
    float part = look_over();
#pragma unroll
    for (int i = 0; i < WPL; ++i) {
      if (ww[i] != 0.0f) part = __builtin_fmaf(ww[i], cur[i], part);
    }
    const float delta = __builtin_fmaf(-gate, column_sum8(part), gv);
    if (bad && !(delta * 0.0f == 0.0f)) {
      for (int n = g; n < N; n += kRrGroups) *row(n) = __builtin_nanf("");
    }
#pragma unroll
    for (int i = 0; i < WPL; ++i) {
      if (bad && ww[i] != 0.0f) *to[i] = __builtin_fmaf(ww[i], delta, cur[i]);
    }
    float* from[RPL];
    float rw[RPL], val[RPL];
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      from[i] = route(P.read_idx, P.read_w, P.reads, i, rw[i]);
      val[i] = *from[i];
    }
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      if (bad && rw[i] != 0.0f) *from[i] = 0.0f;
    }
    float sum = look_over();
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      if (rw[i] != 0.0f) sum = __builtin_fmaf(rw[i], val[i], sum);
      if (bad && rw[i] != 0.0f) *from[i] = val[i];
    }
    const float reading = column_sum8(sum);
    if (bad && g == 0) P.readings[at * D + d] = reading;
    if (__ballot(bad && delta == delta) == 0) break;
  }
}

// WPL, RPL: write and read routes per lane (W <= 8 * WPL, R <= 8 * RPL).
// V: floats per access to the initial and final memory, 4 when D % 4 == 0 and
// both are 16-byte aligned.
template <int WPL, int RPL, int V>
__global__ __launch_bounds__(kRrThreads, 4) void route_recurrence_kernel(RrParams P) {
  using Rec = RrRecord<WPL, RPL>;
  extern __shared__ char lds[];
  // bank and column block: the blocks of one bank on one XCD (workgroups
  // take the XCDs in turn)
  const int64_t local = blockIdx.x / kXcds;
  const int64_t bank = blockIdx.x % kXcds + kXcds * (local / P.blocks);
  if (bank >= P.banks) return;   // the whole workgroup
  const int block = static_cast<int>(local % P.blocks);
  const int nw = (static_cast<int>(blockDim.x) - kRrProducers) / kWave;   // compute waves
  const int cols = nw * kRrCols;
  const int N = P.slots, D = P.width, CH = 1 << P.chunk_shift;
  const int64_t T = P.time, H = P.heads;
  const int64_t b = bank / H, h = bank % H;
  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int table_bytes = (N + 1) * kRrRowBytes;   // a wave's table, row N unused by routes
  char* const stage = lds + nw * table_bytes;
  float* const poison = reinterpret_cast<float*>(
      stage + 2 * (CH + kRrPad) * Rec::kBytes);   // [cols]
  const int d0 = block * cols;
  const float* const m0 = P.m0 + h * N * static_cast<int64_t>(D);
  // the workgroup's columns of a table, `V` floats a thread, kRrRowsAhead
  // rows a thread in flight: f(row, first column, its V values)
  const int per_row = cols / V;
  const int rows_at_once = static_cast<int>(blockDim.x) / per_row;
  const int tn = tid / per_row, tc = (tid - tn * per_row) * V;
  const bool tcol = tn < rows_at_once && d0 + tc < D;   // V == 4: D % 4 == 0
  using Vec = typename std::conditional<V == 4, float4, float>::type;
  auto table_at = [&](int n, int c) __attribute__((always_inline)) {
    return reinterpret_cast<Vec*>(lds + (c / kRrCols) * table_bytes + n * kRrRowBytes +
                                  (c % kRrCols) * 4);
  };

  // 0 or NaN per column: whether the initial memory holds a non-finite value
  if (tid < cols) poison[tid] = 0.0f;
  __syncthreads();
  for (int n0 = tn; n0 < N + 1; n0 += kRrRowsAhead * rows_at_once) {
    Vec v[kRrRowsAhead] = {};
#pragma unroll
    for (int q = 0; q < kRrRowsAhead; ++q) {
      const int n = n0 + q * rows_at_once;
      if (tcol && n < N) {
        v[q] = *reinterpret_cast<const Vec*>(m0 + static_cast<int64_t>(n) * D + d0 + tc);
      }
    }
#pragma unroll
    for (int q = 0; q < kRrRowsAhead; ++q) {
      const int n = n0 + q * rows_at_once;
      if (tn < rows_at_once && n < N + 1) *table_at(n, tc) = v[q];
      const float* const e = reinterpret_cast<const float*>(&v[q]);
#pragma unroll
      for (int k = 0; k < V; ++k) {
        // any thread's NaN will do
        if (!(e[k] * 0.0f == 0.0f)) poison[tc + k] = __builtin_nanf("");
      }
    }
  }

  // compute waves and producers each run a loop of their own over the chunks,
  // meeting at one barrier before the first and one after every chunk
  const int64_t chunks = (T + CH - 1) >> P.chunk_shift;
  const int col = lane / kRrGroups, g = lane % kRrGroups;
  if (wave >= nw) {
    // A producer's share of a chunk on its way from memory to the stage: the
    // loads of a chunk are issued a whole chunk before they are stored.
    constexpr int kPerW = kRrGroups * WPL, kPerR = kRrGroups * RPL;   // entries a token
    constexpr int kPassW = kRrMaxChunk * kPerW / kRrProducers;
    constexpr int kPassR = kRrMaxChunk * kPerR / kRrProducers;
    constexpr int kPassV = kRrMaxChunk * kRrCols * kRrWaves / kRrProducers;
    const int p = tid - nw * kWave;   // producer thread
    const uint32_t hstride = static_cast<uint32_t>(H);
    int64_t widx[kPassW], ridx[kPassR];
    float wwt[kPassW], rwt[kPassR], vals[kPassV], forget = 0.0f, gate = 0.0f;
    auto tokens_in = [&](int64_t c) __attribute__((always_inline)) {
      const int64_t left = T - (c << P.chunk_shift);
      return static_cast<int>(left < CH ? left : CH);
    };
    auto load = [&](int64_t c) __attribute__((always_inline)) {
      const int in = tokens_in(c);
      const int64_t row0 = (b * T + (c << P.chunk_shift)) * H + h;
      // token e / per, clamped to the chunk's last one, entry e % per likewise;
      // offsets within the chunk fit in 32 bits
      auto entries = [&](int64_t* idx, float* w, const int64_t* from, const float* weights, int k,
                         int per, int passes) __attribute__((always_inline)) {
        from += row0 * k;
        weights += row0 * k;
#pragma unroll
        for (int q = 0; q < passes; ++q) {
          const int e = q * kRrProducers + p;
          const uint32_t at = static_cast<uint32_t>(min(e / per, in - 1)) * hstride * k +
                              static_cast<uint32_t>(min(e % per, k - 1));
          idx[q] = from[at];
          w[q] = weights[at];
        }
      };
      entries(ridx, rwt, P.read_idx, P.read_w, P.reads, kPerR, kPassR);
      entries(widx, wwt, P.write_idx, P.write_w, P.writes, kPerW, kPassW);
      const float* const from = P.values + row0 * D;
#pragma unroll
      for (int q = 0; q < kPassV; ++q) {
        const int e = q * kRrProducers + p;
        vals[q] = from[static_cast<uint32_t>(min(e / (kRrCols * kRrWaves), in - 1)) * hstride * D +
                       static_cast<uint32_t>(min(d0 + e % (kRrCols * kRrWaves), D - 1))];
      }
      const uint32_t r = static_cast<uint32_t>(min(p, in - 1)) * hstride;
      forget = (P.forget + row0)[r];
      gate = (P.gate + row0)[r];
    };
    // tokens past T and routes past W or R point at row N with weight 0,
    // gates (1, 0): they change nothing
    auto store = [&](int64_t c) __attribute__((always_inline)) {
      const int in = tokens_in(c);
      char* const base = stage + (c & 1) * (CH + kRrPad) * Rec::kBytes;
      auto entries = [&](const int64_t* idx, const float* w, int k, int offset, int per,
                         int passes) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < passes; ++q) {
          const int e = q * kRrProducers + p;
          const int j = e / per, i = e % per;
          const bool on = j < in && i < k && idx[q] >= 0 && idx[q] < N;
          if (j < CH) {
            *reinterpret_cast<uint2*>(base + j * Rec::kBytes + offset + 8 * i) =
                make_uint2(static_cast<uint32_t>(on ? idx[q] : N) * kRrRowBytes,
                           on ? __float_as_uint(w[q]) : 0u);
          }
        }
      };
      entries(ridx, rwt, P.reads, Rec::kRead, kPerR, kPassR);
      entries(widx, wwt, P.writes, Rec::kWrite, kPerW, kPassW);
#pragma unroll
      for (int q = 0; q < kPassV; ++q) {
        const int e = q * kRrProducers + p;
        const int j = e / (kRrCols * kRrWaves), v = e % (kRrCols * kRrWaves);
        if (j < CH) {
          *reinterpret_cast<float*>(base + j * Rec::kBytes + Rec::kValue + 4 * v) =
              j < in && d0 + v < D ? vals[q] : 0.0f;
        }
      }
      if (p < CH) {
        *reinterpret_cast<float2*>(base + p * Rec::kBytes + Rec::kGates) =
            p < in ? make_float2(expf(forget), gate) : make_float2(1.0f, 0.0f);
      }
    };

    load(0);
    // the records after each stage's chunk
    for (int e = p; e < 2 * kRrPad * Rec::kBytes / 8; e += kRrProducers) {
      const int rec = e / (Rec::kBytes / 8), at = 8 * (e % (Rec::kBytes / 8));
      uint2 v = make_uint2(0u, 0u);
      if (at < Rec::kGates) v.x = static_cast<uint32_t>(N) * kRrRowBytes;
      if (at == Rec::kGates) v.x = __float_as_uint(1.0f);
      *reinterpret_cast<uint2*>(stage + ((rec / kRrPad) * (CH + kRrPad) + CH + rec % kRrPad) *
                                            Rec::kBytes + at) = v;
    }
    store(0);
    if (chunks > 1) load(1);
    __syncthreads();
    for (int64_t c = 0; c < chunks; ++c) {
      // the other stage was read out before the barrier that ended chunk c - 1
      if (c + 1 < chunks) store(c + 1);
      if (c + 2 < chunks) load(c + 2);
      __syncthreads();
    }
  } else {
    __syncthreads();
    char* const mine = lds + wave * table_bytes + col * 4;   // this column's table
    const int d = d0 + wave * kRrCols + col;
    float pz = poison[wave * kRrCols + col];   // 0, or NaN once a row was not finite
    for (int64_t c = 0; c < chunks; ++c) {
      const char* base = stage + (c & 1) * (CH + kRrPad) * Rec::kBytes;
      const char* pw = base + Rec::kWrite + 8 * g;
      const char* pr = base + Rec::kRead + 8 * g;
      const char* pg = base + Rec::kGates;
      const char* pv = base + Rec::kValue + 4 * (wave * kRrCols + col);
      char* at[WPL];               // this token's written rows: address, weight,
      float ww[WPL], wa[WPL];      // exp(forget) where the weight is not 0,
      float cur[WPL];              // value before the token
      float old_rw[RPL], old_row[RPL];   // the token before: read weights and rows
      float old_pz = pz, keep = 0.0f;
      float2 gates = *reinterpret_cast<const float2*>(pg);
      float gv = gates.y * *reinterpret_cast<const float*>(pv);
#pragma unroll
      for (int i = 0; i < WPL; ++i) {
        const uint2 e = *reinterpret_cast<const uint2*>(pw + 8 * kRrGroups * i);
        at[i] = mine + e.x;
        ww[i] = __uint_as_float(e.y);
        wa[i] = ww[i] != 0.0f ? gates.x : 1.0f;
        cur[i] = *reinterpret_cast<float*>(at[i]);
      }
#pragma unroll
      for (int i = 0; i < RPL; ++i) old_rw[i] = old_row[i] = 0.0f;
      // ahead of their use: token j's read entries, token j + 1's write
      // entries, gates and value
      struct Ahead {
        uint2 write[WPL], read[RPL];
        float2 gates;
        float value;
      };
      auto ahead = [&](Ahead& a, int u) __attribute__((always_inline)) {   // iteration u of 8
#pragma unroll
        for (int i = 0; i < RPL; ++i) {
          a.read[i] = *reinterpret_cast<const uint2*>(pr + u * Rec::kBytes + 8 * kRrGroups * i);
        }
#pragma unroll
        for (int i = 0; i < WPL; ++i) {
          a.write[i] = *reinterpret_cast<const uint2*>(pw + (u + 1) * Rec::kBytes +
                                                       8 * kRrGroups * i);
        }
        a.gates = *reinterpret_cast<const float2*>(pg + (u + 1) * Rec::kBytes);
        a.value = *reinterpret_cast<const float*>(pv + (u + 1) * Rec::kBytes);
      };
      Ahead now_a, next_a;
      ahead(now_a, 0);
      // iteration j updates with token j, then sums the reading of token
      // j - 1 while token j + 1's written rows load; lane g keeps the reading
      // of token 8k + g, stored every 8 tokens
      int64_t t = (c << P.chunk_shift) - kRrGroups + g;
      float* out = P.readings + ((b * T + t) * H + h) * D + d;
      for (int j0 = 0; j0 < CH; j0 += kRrGroups) {
#pragma unroll
        for (int u = 0; u < kRrGroups; ++u) {
          ahead(next_a, u + 1);
          __builtin_amdgcn_sched_barrier(0);
          float part = pz;
#pragma unroll
          for (int i = 0; i < WPL; ++i) {
            cur[i] = cur[i] * wa[i];
            part = __builtin_fmaf(ww[i], cur[i], part);
          }
          const float delta = __builtin_fmaf(-gates.y, column_sum8(part), gv);
#pragma unroll
          for (int i = 0; i < WPL; ++i) {
            const float now = __builtin_fmaf(ww[i], delta, cur[i]);
            *reinterpret_cast<float*>(at[i]) = now;
            pz = __builtin_fmaf(now, 0.0f, pz);
          }
#pragma unroll
          for (int i = 0; i < WPL; ++i) {
            at[i] = mine + now_a.write[i].x;
            ww[i] = __uint_as_float(now_a.write[i].y);
            wa[i] = ww[i] != 0.0f ? now_a.gates.x : 1.0f;
            cur[i] = *reinterpret_cast<float*>(at[i]);
          }
          float rw[RPL], row[RPL];
#pragma unroll
          for (int i = 0; i < RPL; ++i) {
            rw[i] = __uint_as_float(now_a.read[i].y);
            row[i] = *reinterpret_cast<float*>(mine + now_a.read[i].x);
          }
          // the store, then these loads, leave first: what follows covers
          // their latency
          __builtin_amdgcn_sched_barrier(0);
          gates = now_a.gates;
          gv = now_a.gates.y * now_a.value;
          now_a = next_a;
          float sum = old_pz;
#pragma unroll
          for (int i = 0; i < RPL; ++i) sum = __builtin_fmaf(old_rw[i], old_row[i], sum);
          const float reading = column_sum8(sum);
          keep = g == (u + kRrGroups - 1) % kRrGroups ? reading : keep;
          if (u == 0 && j0 > 0 && t < T && d < D) *out = keep;
#pragma unroll
          for (int i = 0; i < RPL; ++i) {
            old_rw[i] = rw[i];
            old_row[i] = row[i];
          }
          old_pz = pz;
          __builtin_amdgcn_sched_barrier(0);
        }
        pw += kRrGroups * Rec::kBytes;
        pr += kRrGroups * Rec::kBytes;
        pg += kRrGroups * Rec::kBytes;
        pv += kRrGroups * Rec::kBytes;
        t += kRrGroups;
        out += kRrGroups * H * D;
      }
      // the chunk's last reading and its last store
      float sum = old_pz;
#pragma unroll
      for (int i = 0; i < RPL; ++i) sum = __builtin_fmaf(old_rw[i], old_row[i], sum);
      const float reading = column_sum8(sum);
      keep = g == kRrGroups - 1 ? reading : keep;
      if (t < T && d < D) *out = keep;
      __syncthreads();
    }
    const bool bad = d < D && !(column_sum8(pz) == 0.0f);
    if (__ballot(bad)) exact_columns<WPL, RPL>(P, mine, b, h, d, g, bad);
  }
  __syncthreads();
  float* const out = P.final_memory + bank * N * static_cast<int64_t>(D) + d0 + tc;
  if (!tcol) return;
#pragma unroll 4
  for (int n = tn; n < N; n += rows_at_once) {
    *reinterpret_cast<Vec*>(out + static_cast<int64_t>(n) * D) = *table_at(n, tc);
  }
}

template <int WPL, int RPL>
int32_t launch_route_recurrence(RrParams& P, hipStream_t s) {
  // the waves that D fills, fewer where the tables and the smallest stage
  // would not fit in LDS; then the longest chunk (up to 64 tokens) that fits
  auto bytes = [&](int nw, int shift) {
    return nw * (P.slots + 1) * kRrRowBytes +
           2 * ((1 << shift) + kRrPad) * RrRecord<WPL, RPL>::kBytes + 4 * nw * kRrCols;
  };
  int nw = (P.width + kRrCols - 1) / kRrCols;
  nw = nw > kRrWaves ? kRrWaves : nw;
  while (nw > 1 && bytes(nw, 4) > kRrLds) --nw;
  int shift = 6;
  while (shift > 4 && bytes(nw, shift) > kRrLds) --shift;
  const int lds = bytes(nw, shift);
  P.chunk_shift = shift;
  P.blocks = (P.width + nw * kRrCols - 1) / (nw * kRrCols);
  const int64_t grid = kXcds * ((P.banks + kXcds - 1) / kXcds) * P.blocks;
  if (grid > (int64_t{1} << 31) - 1) return fail(COWSDM_ELIMIT, "route recurrence: batch too large");
  const uintptr_t align = reinterpret_cast<uintptr_t>(P.m0) |
                          reinterpret_cast<uintptr_t>(P.final_memory);
  const bool v4 = P.width % 4 == 0 && align % 16 == 0;
  auto* const kernel = v4 ? &route_recurrence_kernel<WPL, RPL, 4>
                          : &route_recurrence_kernel<WPL, RPL, 1>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
      return fail(static_cast<int32_t>(e), "route recurrence: %d bytes of LDS", lds);
    }
  }
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)),
                     dim3(nw * kWave + kRrProducers), lds, s, P);
  return launch_status("route recurrence");
}

template <int WPL>
int32_t launch_route_recurrence_reads(RrParams& P, hipStream_t s) {
  if (P.reads <= kRrGroups) return launch_route_recurrence<WPL, 1>(P, s);
  if (P.reads <= 2 * kRrGroups) return launch_route_recurrence<WPL, 2>(P, s);
  return launch_route_recurrence<WPL, 4>(P, s);
}

}  // namespace cowsdm_impl

using namespace cowsdm_impl;

extern "C" int32_t cowsdm_route_recurrence_forward(const cowsdm_route_recurrence_t* r,
                                                   void* stream) {
  if (!r) return fail(COWSDM_EARG, "route recurrence: null argument");
  if (r->batch < 0 || r->time <= 0 || r->heads <= 0 || r->slots <= 0 || r->width <= 0 ||
      r->writes <= 0 || r->reads <= 0) {
    return fail(COWSDM_EARG, "route recurrence: invalid sizes");
  }
  if (r->slots > kRrMaxSlots) {
    return fail(COWSDM_ELIMIT, "route recurrence: at most %d slots", kRrMaxSlots);
  }
  if (r->writes > kRrMaxRoutes || r->reads > kRrMaxRoutes) {
    return fail(COWSDM_ELIMIT, "route recurrence: at most %d routes per token", kRrMaxRoutes);
  }
  // offsets within a chunk of tokens stay below 2^31
  if (r->width > (int64_t{1} << 24) || r->heads > (int64_t{1} << 24) ||
      r->heads * (r->width + kRrMaxRoutes) * kRrMaxChunk >= (int64_t{1} << 31)) {
    return fail(COWSDM_ELIMIT, "route recurrence: width too large");
  }
  if (r->batch == 0) return 0;
  if (!r->initial_memory || !r->write_indices || !r->write_weights || !r->values ||
      !r->input_gate || !r->forget_log_gate || !r->read_indices || !r->read_weights ||
      !r->readings || !r->final_memory) {
    return fail(COWSDM_EARG, "route recurrence: null pointer argument");
  }
  RrParams P{};
  P.banks = r->batch * r->heads;
  P.time = r->time;
  P.heads = r->heads;
  P.slots = static_cast<int>(r->slots);
  P.width = static_cast<int>(r->width);
  P.writes = static_cast<int>(r->writes);
  P.reads = static_cast<int>(r->reads);
  P.m0 = r->initial_memory;
  P.write_idx = r->write_indices;
  P.write_w = r->write_weights;
  P.values = r->values;
  P.gate = r->input_gate;
  P.forget = r->forget_log_gate;
  P.read_idx = r->read_indices;
  P.read_w = r->read_weights;
  P.readings = r->readings;
  P.final_memory = r->final_memory;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (P.writes <= kRrGroups) return launch_route_recurrence_reads<1>(P, s);
  if (P.writes <= 2 * kRrGroups) return launch_route_recurrence_reads<2>(P, s);
  return launch_route_recurrence_reads<4>(P, s);
}
