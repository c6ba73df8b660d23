// The token-serial SDM recurrence over dense route vectors: the forward
// recurrence of training and prefill (copy_on_write_sdm/sdm.py:534-607,
// _native_sdm_forward_kernel, launched at sdm.py:829-861), and the scatter
// of sparse routes into dense route vectors (sdm.py:162-172).
//
// Per batch row b and token t, over the whole [N, D] memory:
//   memory[n]  *= exp(forget_log_gate[b, t])   where write_routes[b, t, n] != 0
//   retrieved   = sum_n write_routes[b, t, n] * memory[n]
//   delta       = input_gate[b, t] * values[b, t] - erase_gate[b, t] * retrieved
//   memory[n]  += write_routes[b, t, n] * delta
//   readings[b, t] = sum_n read_routes[b, t, n] * memory[n]
//
// The route vectors come from product keys: a few of their N entries are not
// zero.  Producer waves compact every vector to its nonzero entries while the
// tokens before it run, and the recurrence then touches only those rows, as
// in route_recurrence.hip (the table of 32 columns in LDS, 8 lanes to a
// column, the same pipeline).  A token with more than 8 nonzero write or 32
// nonzero read routes is a dense one, and from its first dense token on a
// sequence is left to a kernel that holds the memory in registers and sums
// over every row (below), launched behind this one: it goes on from the memory
// that this one leaves before that token, whose number it finds in the place of
// the sequence's last reading (handed_over).  A token's arithmetic depends on the
// vectors up to its own, so later tokens never change earlier results.  (With
// up to 64 slots it also depends on whether batch x width is below 4,096, see
// the rule in cowsdm_recurrence_forward: there a batch row's results
// differ in rounding between a small batch and a large one.)
//
// A zero route times a row, or a delta, that is not finite is NaN in the dense
// sums.  Every lane starts its sums from 0 * the rows it wrote, so a column
// that met one reads NaN from that token to the last; at the end its wave
// takes it again with sums over every row, and stores what follows the first
// reading that is not finite.
//
// A dense token costs 0.8 us there (N = 256) and 3.9 here with every row in
// LDS, so one is enough to hand a sequence over: 128 tokens of 16 writes behind
// a first token without any, B = 16, D = 128, 508 -> 114 us, 716 -> 291 with the
// per-token memories.
//
// Per-token memories (the backward's input) are 4 N D bytes a token, written
// by four waves of their own from LDS, 16 bytes a lane and a table row's 32
// columns (128 bytes) together, between two barriers of the token; the
// compute waves load the next token's rows and sum the reading meanwhile.
// (From the compute waves, each storing its 8 columns, 64 batch rows of 64
// tokens took 210 us against 112: half-written 64-byte requests.)
//
// Measured at T = 128, N = 256, D = 128, 4 writes, 16 reads, before (every
// row of every token in registers) and after, time of the call: with the
// per-token memories B = 16 275 -> 88 us (269 MB: 3.1 TB/s; what bounds it is
// the token's two barriers, 0.6 us a token, the bytes alone are 40 us), B = 64
// and T = 64 338 -> 112 us (537 MB, 4.8 TB/s: the bytes); without them 101 ->
// 30 us (the token's serial chain and the host's part of the call).  The
// second launch, where it has nothing to do, takes 4.7 us of them at B = 16.

#include <type_traits>

#include "lds_recurrence.h"

namespace cowsdm_impl {

constexpr int kDrWrites = kRrGroups;         // nonzero write routes of a sparse token
constexpr int kDrReads = 4 * kRrGroups;      // nonzero read routes
constexpr int kDrStoreThreads = 4 * kWave;   // waves that write the per-token memories
constexpr int kDrProducers = 8 * kWave;      // threads that compact the tokens
constexpr int kDrThreads = kRrWaves * kWave + kDrProducers;
constexpr int kDrShift = 4, kDrChunk = 1 << kDrShift;   // tokens staged at a time
constexpr int kDrCopy = 8;                   // rows of a memory such a thread has in flight
constexpr int kDrSegments = kRrMaxSlots / kWave;
constexpr int kCus = 256;

struct RecParams {
  int64_t batch, time;
  int slots, width;
  int blocks;            // column blocks per batch row
  bool all_dense;        // every sequence is taken as one of dense tokens
  const float* m0;       // [B, N, D]
  const float* wr;       // [B, T, N]
  const float* values;   // [B, T, D]
  const float* ig;       // [B, T]
  const float* eg;       // [B, T]
  const float* flg;      // [B, T]
  const float* rr;       // [B, T, N]
  float* readings;       // [B, T, D]
  float* states;         // [B, T, N, D] or null
  float* final_memory;   // [B, N, D] or null
};

// A sequence that is handed over at token `stop` holds these bits in the place
// of its last token's reading, which is still to come, in every column: a NaN
// that no sequence that is done leaves there (done_reading).
constexpr uint32_t kDrNan = 0x7fc00000u;
constexpr int64_t kDrMaxTime = int64_t{1} << 22;

__device__ __forceinline__ float handed_over(int64_t stop) {
  return __uint_as_float(kDrNan | static_cast<uint32_t>(stop + 1));   // stop + 1 < 2^22
}

__device__ __forceinline__ float done_reading(float x) {
  return x != x ? __uint_as_float(kDrNan) : x;
}

// The token that the sequence of this last reading is handed over at, or -1.
__device__ __forceinline__ int64_t handed_over_at(float last) {
  const uint32_t bits = __float_as_uint(last);
  return bits > kDrNan && bits < kDrNan + kDrMaxTime ? static_cast<int64_t>(bits - kDrNan) - 1
                                                     : -1;
}

// Whether a token is not a dense one (the same in every wave that asks).
__device__ __forceinline__ bool sparse_token(const float* w, const float* r, int N) {
  const int lane = static_cast<int>(threadIdx.x) % kWave;
  int writes = 0, reads = 0;
#pragma unroll 4
  for (int n = lane; n < ((N + kWave - 1) & -kWave); n += kWave) {
    const int at = n < N ? n : 0;
    const float x = w[at], y = r[at];
    writes += __popcll(__ballot(n < N && x != 0.0f));
    reads += __popcll(__ballot(n < N && y != 0.0f));
  }
  return writes <= kDrWrites && reads <= kDrReads;
}

// A barrier of the workgroup that orders LDS only: global loads and stores
// stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// A wave's columns that are `bad` (the same in a column's lanes), `end` tokens
// from the initial memory on with sums over every row: the table (`mine`: the
// column's) is left as the memory behind them (before token T and without
// per-token memories it also goes to where the next kernel looks for it), and
// readings and per-token memories are stored from the first reading that is
// not finite.
template <bool STATES>
__device__ __forceinline__ void redo_columns(const RecParams& P, char* mine, int64_t b, int d,
                                             int g, int64_t end, bool bad) {
  const int N = P.slots, D = P.width;
  const int64_t T = P.time;
  float* const readings = P.readings + b * T * D + (bad ? d : 0);
  auto finite = [](float x) __attribute__((always_inline)) { return x * 0.0f == 0.0f; };
  auto row = [&](int n) __attribute__((always_inline)) {
    return reinterpret_cast<float*>(mine + n * kRrRowBytes);
  };
  __threadfence();   // the wave's own readings, by other lanes of it
  int64_t from = end;
  for (int64_t t = g; bad && t < from; t += kRrGroups) {
    if (!finite(readings[t * D])) from = t;
  }
#pragma unroll
  for (int o = kRrGroups / 2; o > 0; o >>= 1) {
    const int64_t other = __shfl_xor(from, o, kWave);
    from = other < from ? other : from;
  }
  for (int n = g; n < N; n += kRrGroups) {
    if (bad) *row(n) = P.m0[(b * N + n) * static_cast<int64_t>(D) + d];
  }
  for (int64_t t = 0; t < end; ++t) {
    const int64_t bt = b * T + t;
    const float* const wt = P.wr + bt * N;
    const float* const rt = P.rr + bt * N;
    const float alpha = expf(P.flg[bt]);
    float part = 0.0f;
#pragma unroll 8
    for (int n = g; n < N; n += kRrGroups) {
      const float w = wt[n], m = *row(n);
      part = __builtin_fmaf(w, w != 0.0f ? m * alpha : m, part);
    }
    const float gv = P.ig[bt] * (bad ? P.values[bt * D + d] : 0.0f);
    const float delta = __builtin_fmaf(-P.eg[bt], column_sum8(part), gv);
    float sum = 0.0f;
#pragma unroll 8
    for (int n = g; n < N; n += kRrGroups) {
      const float w = wt[n], m = *row(n);
      const float now = __builtin_fmaf(w, delta, w != 0.0f ? m * alpha : m);
      if (bad) *row(n) = now;
      sum = __builtin_fmaf(rt[n], now, sum);
    }
    const float reading = column_sum8(sum);
    if (bad && t >= from) {
      if (g == 0) readings[t * D] = done_reading(reading);
      if (STATES) {
        for (int n = g; n < N; n += kRrGroups) {
          P.states[(bt * N + n) * static_cast<int64_t>(D) + d] = *row(n);
        }
      }
    }
    // once every row of these columns is NaN, so is what follows; their
    // readings are already
    if (__ballot(bad && delta == delta) == 0) {
      float* to = P.states + (bt + 1) * N * static_cast<int64_t>(D) + d;
      for (int64_t n = g; STATES && bad && n < (end - 1 - t) * N; n += kRrGroups) {
        to[n * D] = __builtin_nanf("");
      }
      break;
    }
  }
  if (!STATES && end < T) {
    for (int n = g; n < N; n += kRrGroups) {
      if (bad) P.final_memory[(b * N + n) * static_cast<int64_t>(D) + d] = *row(n);
    }
  }
}

// V: floats per access to the memories, 4 when D % 4 == 0 and they are
// 16-byte aligned.  SEG: 64-slot segments of a route vector, at most.
template <int V, int SEG, bool STATES>
__global__ __launch_bounds__(kDrThreads + (STATES ? kDrStoreThreads : 0)) void recurrence_kernel(RecParams P) {
  using Rec = RrRecord<1, 4>;
  using Vec = typename std::conditional<V == 4, float4, float>::type;
  extern __shared__ char lds[];
  const int64_t local = blockIdx.x / kXcds;
  const int64_t b = blockIdx.x % kXcds + kXcds * (local / P.blocks);
  if (b >= P.batch) return;   // the whole workgroup
  const int block = static_cast<int>(local % P.blocks);
  const int nw = (static_cast<int>(blockDim.x) - kDrProducers -
                  (STATES ? kDrStoreThreads : 0)) / kWave;   // compute waves
  const int cols = nw * kRrCols;
  const int N = P.slots, D = P.width, CH = kDrChunk;
  const int64_t T = P.time;
  const int tid = static_cast<int>(threadIdx.x);
  // the whole workgroup again: every wave counts the same vectors
  float* const last_reading_out = P.readings + (b * T + T - 1) * D + block * cols + tid;
  if (T > 0 && !sparse_token(P.wr + b * T * N, P.rr + b * T * N, N)) {
    if (tid < cols && block * cols + tid < D) *last_reading_out = handed_over(0);
    return;
  }
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int table_bytes = (N + 1) * kRrRowBytes;   // a wave's table, row N unused by routes
  char* const stage = lds + nw * table_bytes;
  float* const poison = reinterpret_cast<float*>(stage + 2 * (CH + kRrPad) * Rec::kBytes);
  const int d0 = block * cols;

  // the workgroup's columns of a [N, D] memory: V floats a thread
  const int per_row = cols / V;
  auto table_at = [&](int n, int c) __attribute__((always_inline)) {
    return reinterpret_cast<Vec*>(lds + (c / kRrCols) * table_bytes + n * kRrRowBytes +
                                  (c % kRrCols) * 4);
  };
  // `poison`, 0 or NaN per column: whether the initial memory holds a value
  // that is not finite.  `stop`: the sequence's first dense token, set by the
  // compute waves in its chunk (all the same value), for all others at the end
  // of that chunk.  `redo`: whether some columns are taken again.
  int64_t* const stop = reinterpret_cast<int64_t*>(poison + cols);
  int* const redo = reinterpret_cast<int*>(stop + 1);
  if (tid < cols) poison[tid] = 0.0f;
  if (tid == 0) {
    *stop = INT64_MAX;
    *redo = 0;
  }
  __syncthreads();
  {
    const float* const m0 = P.m0 + b * N * static_cast<int64_t>(D);
    const int at_once = static_cast<int>(blockDim.x) / per_row;
    const int tn = tid / per_row, tc = (tid - tn * per_row) * V;
    for (int n0 = tn; n0 < N + 1; n0 += kRrRowsAhead * at_once) {
      Vec v[kRrRowsAhead] = {};
#pragma unroll
      for (int q = 0; q < kRrRowsAhead; ++q) {
        const int n = n0 + q * at_once;
        if (tn < at_once && d0 + tc < D && n < N) {
          v[q] = *reinterpret_cast<const Vec*>(m0 + static_cast<int64_t>(n) * D + d0 + tc);
        }
      }
#pragma unroll
      for (int q = 0; q < kRrRowsAhead; ++q) {
        const int n = n0 + q * at_once;
        if (tn < at_once && n < N + 1) *table_at(n, tc) = v[q];
        const float* const e = reinterpret_cast<const float*>(&v[q]);
#pragma unroll
        for (int k = 0; k < V; ++k) {
          if (!(e[k] * 0.0f == 0.0f)) poison[tc + k] = __builtin_nanf("");
        }
      }
    }
  }

  const int64_t chunks = (T + CH - 1) >> kDrShift;
  const int col = lane / kRrGroups, g = lane % kRrGroups;
  float pz = 0.0f;   // compute waves: NaN once a row was not finite
  // Whether the sequence ends in chunk c.  A wave asks after the chunk's last
  // barrier, and what a faster one may have set by then is a later chunk's.
  // (A relaxed load: a volatile one waits for the wave's stores.  Once a chunk:
  // asked for every token by the store waves it took 10 us of 98 at B = 16,
  // T = 128, N = 256, D = 128.)
  auto stops_in = [&](int64_t c) __attribute__((always_inline)) {
    return (__hip_atomic_load(stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >> kDrShift) <=
           c;
  };
  if (wave >= nw && wave < nw + kDrProducers / kWave) {
    // ---- producers: wave pw takes the tokens pw, pw + 8, ..., kAhead of them
    // loaded before they are needed.  A token is compacted in parts, one
    // beside each of eight tokens, so that none is long beside a token.
    const int pw = wave - nw;
    constexpr int kEach = kDrProducers / kWave, kParts = 8;
    constexpr int kAhead = SEG <= 4 ? 2 : 1;   // divides the tokens of a wave in a chunk
    float w[kAhead][SEG], r[kAhead][SEG];
    float value[kAhead] = {}, gate[kAhead] = {}, erase[kAhead] = {}, forget[kAhead] = {};
    auto load = [&](int i, int64_t t) __attribute__((always_inline)) {
      if (t >= T) return;
      const float* const wt = P.wr + (b * T + t) * N;
      const float* const rt = P.rr + (b * T + t) * N;
#pragma unroll
      for (int q = 0; q < SEG; ++q) {
        const int n = q * kWave + lane;
        w[i][q] = n < N ? wt[n] : 0.0f;
        r[i][q] = n < N ? rt[n] : 0.0f;
      }
      const int64_t at = b * T + t;
      value[i] = lane < cols && d0 + lane < D ? P.values[at * D + d0 + lane] : 0.0f;
      gate[i] = P.ig[at];
      erase[i] = P.eg[at];
      forget[i] = P.flg[at];
    };
    const uint64_t below = (uint64_t{1} << lane) - 1;
    char* rec = nullptr;
    int writes = 0, reads = 0;
    auto blank = [&]() __attribute__((always_inline)) {   // row N with weight 0 changes nothing
      if (lane < kDrWrites + kDrReads) {
        *reinterpret_cast<uint2*>(rec + 8 * lane) =
            make_uint2(static_cast<uint32_t>(N) * kRrRowBytes, 0u);
      }
    };
    auto compact = [&](float x, int n, int offset, int most, int& count)
        __attribute__((always_inline)) {
      const uint64_t some = __ballot(x != 0.0f);
      const int at = count + __popcll(some & below);
      if (x != 0.0f && at < most) {
        *reinterpret_cast<uint2*>(rec + offset + 8 * at) =
            make_uint2(static_cast<uint32_t>(n) * kRrRowBytes, __float_as_uint(x));
      }
      count += __popcll(some);
    };
    // part p of token t in slot i: its entries, in order of their rows, over
    // blank ones; then its gates and value, and the loads of token t + 8 kAhead
    auto produce = [&](int i, int p, int64_t t) __attribute__((always_inline)) {
      if (p == 0) {
        rec = stage + (((t >> kDrShift) & 1) * (CH + kRrPad) + (t & (CH - 1))) * Rec::kBytes;
        blank();
        writes = reads = 0;
      }
      const bool in = t < T;
      if (in) {
#pragma unroll
        for (int e = p * 2 * SEG / kParts; e < (p + 1) * 2 * SEG / kParts; ++e) {
          const int q = e / 2;
          if (e % 2 == 0) {
            compact(w[i][q], q * kWave + lane, Rec::kWrite, kDrWrites, writes);
          } else {
            compact(r[i][q], q * kWave + lane, Rec::kRead, kDrReads, reads);
          }
        }
      }
      if (p < kParts - 1) return;
      const float flag = writes > kDrWrites || reads > kDrReads ? 1.0f : 0.0f;
      if (lane == 0) {
        *reinterpret_cast<float4*>(rec + Rec::kGates) =
            in ? make_float4(expf(forget[i]), gate[i], erase[i], flag)
               : make_float4(1.0f, 0.0f, 0.0f, 0.0f);
      }
      if (lane < kRrCols * kRrWaves) {
        *reinterpret_cast<float*>(rec + Rec::kValue + 4 * lane) = in ? value[i] : 0.0f;
      }
      load(i, t + kAhead * kEach);
    };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) load(i, pw + i * kEach);
    for (int q = pw; q < 2 * kRrPad; q += kEach) {   // the records after each stage's chunk
      rec = stage + ((q / kRrPad) * (CH + kRrPad) + CH + q % kRrPad) * Rec::kBytes;
      blank();
      if (lane == 0) {
        *reinterpret_cast<float4*>(rec + Rec::kGates) = make_float4(1.0f, 0.0f, 0.0f, 0.0f);
      }
      if (lane < kRrCols * kRrWaves) *reinterpret_cast<float*>(rec + Rec::kValue + 4 * lane) = 0.0f;
    }
    // chunk c of `chunks`, beside chunk c - 1 (whose stage is the other one)
    auto chunk = [&](int64_t c, bool paced) __attribute__((always_inline)) {
      for (int j = pw; j < CH; j += kAhead * kEach) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
#pragma unroll
          for (int p = 0; p < kParts; ++p) {
            if (c < chunks || !paced) produce(i, p, (c << kDrShift) + j + i * kEach);
            if (paced) {
              lds_barrier();
              lds_barrier();
            }
          }
        }
      }
    };
    chunk(0, false);
    __syncthreads();
    for (int64_t c = 1; c <= chunks; ++c) {
      if constexpr (STATES) {
        chunk(c, true);
      } else {
        if (c < chunks) chunk(c, false);
        __syncthreads();
      }
      if (stops_in(c - 1)) break;
    }
  } else if (STATES && wave >= nw) {
    // ---- the per-token memories: the table as it is between a token's barriers
    const int p = tid - nw * kWave - kDrProducers;
    const int copiers = kDrStoreThreads / per_row;   // rows at once
    const int n0 = p / per_row, cc = (p - n0 * per_row) * V;
    const bool on = n0 < copiers && d0 + cc < D;
    const int rows = kDrCopy * copiers;
    typedef float Copy __attribute__((ext_vector_type(V)));
    float* out = P.states + (b * T * N + n0) * static_cast<int64_t>(D) + d0 + cc;
    __syncthreads();
    // (every lane takes part in the barriers, so the loops are the same in all)
    for (int64_t c = 0; c < chunks; ++c) {
      const int64_t left = T - (c << kDrShift);
      const int in = static_cast<int>(left < CH ? left : CH);   // tokens of the chunk
      for (int j = 0; j < CH; ++j, out += static_cast<int64_t>(N) * D) {
        lds_barrier();
        float* to = out;
        for (int first = 0; first < N; first += rows) {
          Copy v[kDrCopy];
#pragma unroll
          for (int q = 0; q < kDrCopy; ++q) {
            const int n = first + n0 + q * copiers;
            v[q] = *reinterpret_cast<const Copy*>(table_at(n < N ? n : N, cc));
          }
          if (first + rows >= N) lds_barrier();   // the last rows are in registers
#pragma unroll
          for (int q = 0; q < kDrCopy; ++q) {
            if (on && j < in && first + n0 + q * copiers < N) *reinterpret_cast<Copy*>(to) = v[q];
            to += static_cast<int64_t>(copiers) * D;
          }
        }
      }
      if (stops_in(c)) break;
    }
  } else {
    // ---- compute waves
    __syncthreads();
    char* const mine = lds + wave * table_bytes + col * 4;   // this column's table
    const int d = d0 + wave * kRrCols + col;
    pz = poison[wave * kRrCols + col];
    bool stopped = false;   // at a dense token, with pz before it
    float pz_before = 0.0f;
    // a token's two barriers: its update is done; its memory has been read out
    auto updated = [&]() __attribute__((always_inline)) { if (STATES) lds_barrier(); };
    auto copied = [&]() __attribute__((always_inline)) { if (STATES) lds_barrier(); };
    auto entry = [&](const char* p) __attribute__((always_inline)) {
      return *reinterpret_cast<const uint2*>(p);
    };
    auto at_row = [&](uint32_t offset) __attribute__((always_inline)) {
      return reinterpret_cast<float*>(mine + offset);
    };
    for (int64_t c = 0; c < chunks; ++c) {
      const char* base = stage + (c & 1) * (CH + kRrPad) * Rec::kBytes;
      const char* pw = base + Rec::kWrite + 8 * g;
      const char* pr = base + Rec::kRead + 8 * g;
      const char* pg = base + Rec::kGates;
      const char* pv = base + Rec::kValue + 4 * (wave * kRrCols + col);
      // the pipeline: token j's written row, its weight, its decay and its
      // value before the token; its gates; its read entries; token j - 1's
      // read weights and rows
      float* at;
      float ww, wa, cur, gv;
      float4 gates;
      float old_rw[4], old_row[4], old_pz = pz, keep = 0.0f;
      struct Ahead {
        uint2 write, read[4];
        float4 gates;
        float value;
      };
      auto ahead = [&](Ahead& a, int u) __attribute__((always_inline)) {   // iteration u of 8
#pragma unroll
        for (int i = 0; i < 4; ++i) a.read[i] = entry(pr + u * Rec::kBytes + 8 * kRrGroups * i);
        a.write = entry(pw + (u + 1) * Rec::kBytes);
        a.gates = *reinterpret_cast<const float4*>(pg + (u + 1) * Rec::kBytes);
        a.value = *reinterpret_cast<const float*>(pv + (u + 1) * Rec::kBytes);
      };
      Ahead now_a, next_a;
      auto begin = [&](int u) __attribute__((always_inline)) {   // token u of the group at p*
        const uint2 e = entry(pw + u * Rec::kBytes);
        gates = *reinterpret_cast<const float4*>(pg + u * Rec::kBytes);
        gv = gates.y * *reinterpret_cast<const float*>(pv + u * Rec::kBytes);
        at = at_row(e.x);
        ww = __uint_as_float(e.y);
        wa = ww != 0.0f ? gates.x : 1.0f;
        cur = *at;
#pragma unroll
        for (int i = 0; i < 4; ++i) old_rw[i] = old_row[i] = 0.0f;
        ahead(now_a, u);
      };
      begin(0);
      int64_t t = (c << kDrShift) - kRrGroups + g;
      float* out = P.readings + (b * T + t) * D + d;
      auto last_reading = [&]() __attribute__((always_inline)) {
        float sum = old_pz;
#pragma unroll
        for (int i = 0; i < 4; ++i) sum = __builtin_fmaf(old_rw[i], old_row[i], sum);
        return column_sum8(sum);
      };
      for (int j0 = 0; j0 < CH; j0 += kRrGroups) {
        // lane g: whether token g of these 8 is a dense one
        const float flag = *reinterpret_cast<const float*>(pg + g * Rec::kBytes + 12);
        const uint32_t dense = static_cast<uint32_t>(__ballot(flag != 0.0f)) & 0xffu;
        if (dense == 0) {
#pragma unroll
          for (int u = 0; u < kRrGroups; ++u) {
            ahead(next_a, u + 1);
            __builtin_amdgcn_sched_barrier(0);
            cur = cur * wa;
            const float delta = __builtin_fmaf(-gates.z, column_sum8(__builtin_fmaf(ww, cur, pz)),
                                               gv);
            const float now = __builtin_fmaf(ww, delta, cur);
            *at = now;
            pz = __builtin_fmaf(now, 0.0f, pz);
            updated();
            at = at_row(now_a.write.x);
            ww = __uint_as_float(now_a.write.y);
            wa = ww != 0.0f ? now_a.gates.x : 1.0f;
            cur = *at;
            float rw[4], row[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              rw[i] = __uint_as_float(now_a.read[i].y);
              row[i] = *at_row(now_a.read[i].x);
            }
            __builtin_amdgcn_sched_barrier(0);
            gates = now_a.gates;
            gv = now_a.gates.y * now_a.value;
            now_a = next_a;
            const float reading = last_reading();
            keep = g == (u + kRrGroups - 1) % kRrGroups ? reading : keep;
            if (u == 0 && j0 > 0 && t < T && d < D) *out = done_reading(keep);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              old_rw[i] = rw[i];
              old_row[i] = row[i];
            }
            old_pz = pz;
            copied();
            __builtin_amdgcn_sched_barrier(0);
          }
        } else {
          // one token after the other, in the arithmetic above, up to the
          // first dense one; what follows only keeps the barriers, and its
          // results are the next kernel's
          const float before = last_reading();
          keep = g == kRrGroups - 1 ? before : keep;
          if (j0 > 0 && t < T && d < D) *out = done_reading(keep);
          const int first = stopped ? 0 : __builtin_ctz(dense);
          for (int u = 0; u < first; ++u) {
            const uint2 e = entry(pw + u * Rec::kBytes);
            gates = *reinterpret_cast<const float4*>(pg + u * Rec::kBytes);
            gv = gates.y * *reinterpret_cast<const float*>(pv + u * Rec::kBytes);
            float* const p = at_row(e.x);
            const float w = __uint_as_float(e.y);
            const float m = *p * (w != 0.0f ? gates.x : 1.0f);
            const float delta = __builtin_fmaf(-gates.z, column_sum8(__builtin_fmaf(w, m, pz)),
                                               gv);
            const float now = __builtin_fmaf(w, delta, m);
            *p = now;
            pz = __builtin_fmaf(now, 0.0f, pz);
            updated();
            float sum = pz;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const uint2 q = entry(pr + u * Rec::kBytes + 8 * kRrGroups * i);
              sum = __builtin_fmaf(__uint_as_float(q.y), *at_row(q.x), sum);
            }
            const float reading = column_sum8(sum);
            keep = g == u ? reading : keep;
            copied();
          }
          if (!stopped) {
            stopped = true;
            pz_before = pz;
            if (lane == 0) *stop = (c << kDrShift) + j0 + first;
            if (!STATES && d < D && column_sum8(pz) == 0.0f) {   // others: redo_columns
              // the memory before the dense token, where the next kernel
              // looks for it (else it is the last per-token memory)
              for (int n = g; n < N; n += kRrGroups) {
                P.final_memory[(b * N + n) * static_cast<int64_t>(D) + d] =
                    *at_row(n * kRrRowBytes);
              }
            }
          }
          for (int u = first; u < kRrGroups; ++u) {
            updated();
            copied();
          }
          begin(kRrGroups);
          old_pz = 0.0f;
        }
        pw += kRrGroups * Rec::kBytes;
        pr += kRrGroups * Rec::kBytes;
        pg += kRrGroups * Rec::kBytes;
        pv += kRrGroups * Rec::kBytes;
        t += kRrGroups;
        out += kRrGroups * D;
      }
      // the chunk's last reading and its last store
      const float reading = last_reading();
      keep = g == kRrGroups - 1 ? reading : keep;
      if (t < T && d < D) *out = done_reading(keep);
      if (!STATES) __syncthreads();
      if (stopped) break;
    }
    if (stopped) pz = pz_before;
  }
  // a column that was never other than finite keeps pz 0
  const bool bad = wave < nw && T > 0 && d0 + wave * kRrCols + col < D &&
                   !(column_sum8(pz) == 0.0f);
  if (bad) *redo = 1;
  __syncthreads();   // what the store waves wrote is out, too
  const int64_t end = *stop < T ? *stop : T;
  if (*redo) {
    if (__ballot(bad)) {
      redo_columns<STATES>(P, lds + wave * table_bytes + col * 4, b, d0 + wave * kRrCols + col, g,
                           end, bad);
    }
    __syncthreads();
  }
  if (end < T) {
    if (tid < cols && d0 + tid < D) *last_reading_out = handed_over(end);
    return;
  }
  if (!P.final_memory) return;
  float* const out = P.final_memory + b * N * static_cast<int64_t>(D);
  const int at_once = static_cast<int>(blockDim.x) / per_row;
  const int tn = tid / per_row, tc = (tid - tn * per_row) * V;
  if (tn >= at_once || d0 + tc >= D) return;
#pragma unroll 4
  for (int n = tn; n < N; n += at_once) {
    *reinterpret_cast<Vec*>(out + static_cast<int64_t>(n) * D + d0 + tc) = *table_at(n, tc);
  }
}

// ---- sequences from their first dense token on
//
// A wave owns 4 columns of one batch row's memory for the whole sequence,
// in registers: lane = 16 * column + row group, and row group g holds rows
// g * RPL .. g * RPL + RPL - 1 (RPL rows per lane, N <= 16 * RPL).  A
// column's 16 row groups are one DPP row of the wave, so both sums over N
// are in-register: each lane's partial sum over its rows, a DPP prefix
// within the row (lane 15 ends with the column's total) and a readlane per
// column, which gives every row of a column the same value.  The tokens of
// a sequence are serial; batch rows and column blocks are independent
// waves.  The inputs of the next tokens are in flight while a token
// computes (route vectors and values up to 8 tokens ahead, as many as 64
// registers hold; the gates of 64 tokens a lane each, a chunk ahead), and
// every load is a vector load whose value is first used tokens later.

constexpr int kRecCols = 4;                  // columns per wave
constexpr int kRecGroups = kWave / kRecCols; // row groups per column: one DPP row
constexpr int kRecWaves = 4;                 // waves per workgroup
constexpr int kRecThreads = kRecWaves * kWave;

// Sum of v over the 16 lanes of each DPP row, the same value in every lane
// of the row: an inclusive DPP prefix within the row (row_shr 1, 2, 4, 8;
// lanes shifted in from outside the row add 0), lane 15 of each row read
// back, the row's value selected by the lane's column.
__device__ __forceinline__ float column_sum(float v, int col) {
  int x = __float_as_int(v);
  x = __float_as_int(__int_as_float(x) +
                     __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false)));
  x = __float_as_int(__int_as_float(x) +
                     __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false)));
  x = __float_as_int(__int_as_float(x) +
                     __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false)));
  x = __float_as_int(__int_as_float(x) +
                     __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false)));
  const float s0 = __int_as_float(__builtin_amdgcn_readlane(x, 15));
  const float s1 = __int_as_float(__builtin_amdgcn_readlane(x, 31));
  const float s2 = __int_as_float(__builtin_amdgcn_readlane(x, 47));
  const float s3 = __int_as_float(__builtin_amdgcn_readlane(x, 63));
  return col == 0 ? s0 : (col == 1 ? s1 : (col == 2 ? s2 : s3));
}

// RPL rows of one route vector (`row`, the same in every lane) from row n0
// on.  Rows at or above N are loaded from row 0 instead and must be masked
// where they are used (a select right after the load would wait for it).
// V4: N % 4 == 0, 16-byte aligned vectors and RPL % 4 == 0.
template <int RPL, bool V4>
__device__ __forceinline__ void load_rows(const float* row, int n0, int N, float (&w)[RPL]) {
  if constexpr (V4) {
#pragma unroll
    for (int j = 0; j < RPL; j += 4) {
      const uint32_t off = n0 + j < N ? static_cast<uint32_t>(n0 + j) : 0u;
      const float4 q = *reinterpret_cast<const float4*>(row + off);
      w[j] = q.x;
      w[j + 1] = q.y;
      w[j + 2] = q.z;
      w[j + 3] = q.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < RPL; ++j) w[j] = row[n0 + j < N ? static_cast<uint32_t>(n0 + j) : 0u];
  }
}

// The RPL rows of a lane's column to or from a [N, D] block (`base`, the
// same in every lane; lane offset n0 * D + d, row stride D): one branch when
// all of them are below N, a check per row otherwise.
template <int RPL>
__device__ __forceinline__ void store_rows(float* base, uint32_t off, uint32_t D, int n0, int N,
                                           const float (&m)[RPL]) {
  if (n0 + RPL <= N) {
#pragma unroll
    for (int i = 0; i < RPL; ++i) base[off + static_cast<uint32_t>(i) * D] = m[i];
  } else {
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      if (n0 + i < N) base[off + static_cast<uint32_t>(i) * D] = m[i];
    }
  }
}

// Tokens whose route vectors are in flight at once: as many as fit in 64
// registers (two vectors of RPL rows each), at most 8 (more spills
// registers and halves the waves a SIMD holds).
template <int RPL>
constexpr int rec_ahead() {
  return 32 / RPL < 1 ? 1 : (32 / RPL > 8 ? 8 : 32 / RPL);
}

// EXACT: N == 16 * RPL, every lane's rows are below N (no masks).
template <int RPL, bool V4, bool EXACT>
__global__ __launch_bounds__(kRecThreads) void dense_recurrence_kernel(RecParams P) {
  constexpr int PF = rec_ahead<RPL>();
  const int lane = static_cast<int>(threadIdx.x) % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int64_t item = static_cast<int64_t>(blockIdx.x) * kRecWaves + wave;
  if (item >= P.batch * P.blocks) return;
  const int64_t b = item / P.blocks;
  const int cb = static_cast<int>(item - b * P.blocks);
  const int col = lane / kRecGroups;
  const int g = lane % kRecGroups;
  const int N = P.slots, D = P.width;
  // its columns hold the same number; the same in every lane of the wave
  const int64_t start =
      P.all_dense ? 0
                  : handed_over_at(P.readings[((b + 1) * P.time - 1) * D + cb * kRecCols]);
  if (start < 0) return;
  const int64_t T = P.time - start;
  const int64_t first = b * P.time + start;   // of the tokens, over the batch
  const int d = cb * kRecCols + col;
  const bool col_ok = d < D;
  const int n0 = g * RPL;

  // the lane's rows in a [N, D] block: offset n0 * D + d, stride D (the
  // host keeps N * D below 2^31)
  const uint32_t off = static_cast<uint32_t>(n0) * static_cast<uint32_t>(D) +
                       static_cast<uint32_t>(col_ok ? d : 0);
  float m[RPL];
  {
    // the memory before token `start` (recurrence_kernel's)
    const float* src = start == 0 ? P.m0 + b * N * static_cast<int64_t>(D)
                       : P.states ? P.states + (first - 1) * N * static_cast<int64_t>(D)
                                  : P.final_memory + b * N * static_cast<int64_t>(D);
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      const bool in = col_ok && n0 + i < N;
      const float v = src[in ? off + static_cast<uint32_t>(i * D) : 0u];
      m[i] = in ? v : 0.0f;
    }
  }
  const float* const wr_b = P.wr + first * N;
  const float* const rr_b = P.rr + first * N;
  // ring of PF tokens' route vectors and values: slot j holds token t0 + j
  // of the current round, and is refilled with token t + PF as soon as
  // token t is done.  Every load is a vector load, so a wait for the oldest
  // one does not wait for the newer ones.
  float w[PF][RPL], r[PF][RPL], val[PF];
  auto fetch = [&](int j, int64_t t) __attribute__((always_inline)) {
    load_rows<RPL, V4>(wr_b + t * N, n0, N, w[j]);
    load_rows<RPL, V4>(rr_b + t * N, n0, N, r[j]);
    // a lane past the width computes on column 0's values and stores nothing
    val[j] = P.values[(first + t) * D + (col_ok ? d : 0)];
  };
  // the gates of 64 tokens, lane k holding token 64c + k's, a chunk ahead
  float gates[2][3];
  auto fetch_gates = [&](int slot, int64_t c) __attribute__((always_inline)) {
    const int64_t t = c * kWave + lane;
    const int64_t bt = first + (t < T ? t : 0);
    gates[slot][0] = P.flg[bt];
    gates[slot][1] = P.ig[bt];
    gates[slot][2] = P.eg[bt];
  };
  if (T > 0) fetch_gates(0, 0);
  if (T > kWave) fetch_gates(1, 1);
  if (T > 0) {
#pragma unroll
    for (int j = 0; j < PF; ++j) fetch(j, j < T ? j : T - 1);
  }
  for (int64_t t0 = 0; t0 < T; t0 += PF) {
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int64_t t = t0 + j;
      if (t >= T) break;
      const int64_t bt = first + t;
      const int k = static_cast<int>(t % kWave);
      const int slot = static_cast<int>((t / kWave) & 1);
      float fg, in_g, er_g;
      if (slot == 0) {
        fg = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gates[0][0]), k));
        in_g = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gates[0][1]), k));
        er_g = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gates[0][2]), k));
      } else {
        fg = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gates[1][0]), k));
        in_g = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gates[1][1]), k));
        er_g = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gates[1][2]), k));
      }
      if (k == kWave - 1 && (t / kWave) + 2 < (T + kWave - 1) / kWave) {
        // chunk t / 64 is done: its slot takes the chunk after next
        if (slot == 0) fetch_gates(0, t / kWave + 2); else fetch_gates(1, t / kWave + 2);
      }
      const float alpha = expf(fg);
      float wj[RPL], rj[RPL];
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        wj[i] = EXACT || n0 + i < N ? w[j][i] : 0.0f;
        rj[i] = EXACT || n0 + i < N ? r[j][i] : 0.0f;
      }
      float part = 0.0f;
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        m[i] = wj[i] != 0.0f ? m[i] * alpha : m[i];
        part = __builtin_fmaf(wj[i], m[i], part);
      }
      const float retrieved = column_sum(part, col);
      const float delta = in_g * val[j] - er_g * retrieved;
      float rp = 0.0f;
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        m[i] = __builtin_fmaf(wj[i], delta, m[i]);
        if (!EXACT && n0 + i >= N) m[i] = 0.0f;   // 0 * a delta that is not finite
        rp = __builtin_fmaf(rj[i], m[i], rp);
      }
      // the slot takes token t + PF (the last token again near the end, so
      // that every round loads the same registers)
      fetch(j, t + PF < T ? t + PF : T - 1);
      const float reading = column_sum(rp, col);
      if (g == 0 && col_ok) P.readings[bt * D + d] = reading;
      if (P.states && col_ok) {
        store_rows<RPL>(P.states + bt * N * static_cast<int64_t>(D), off, D, n0, N, m);
      }
    }
  }
  if (P.final_memory && col_ok) {
    store_rows<RPL>(P.final_memory + b * N * static_cast<int64_t>(D), off, D, n0, N, m);
  }
}

// Dense route vectors: out[row, n] = the weight of the last k with
// indices[row, k] == n, else 0; an index outside [0, N) sets bit 0x1 of
// *bad.  Thread = (row, n); a row's K indices are read by each of its N
// threads (from cache).
template <typename IDX>
__global__ __launch_bounds__(256) void dense_routes_kernel(const float* weights, const IDX* indices,
                                                           int64_t rows, int k, int slots,
                                                           float* out, int32_t* bad) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= rows * slots) return;
  const int64_t row = e / slots;
  const int n = static_cast<int>(e - row * slots);
  float v = 0.0f;
  bool outside = false;
  for (int j = 0; j < k; ++j) {
    const int64_t x = static_cast<int64_t>(indices[row * k + j]);
    if (x == n) v = weights[row * k + j];
    outside |= (n == 0) && (x < 0 || x >= slots);
  }
  out[e] = v;
  if (outside && bad) atomicOr(bad, 1);
}

template <int RPL>
void launch_dense_recurrence(const RecParams& P, bool v4, unsigned grid, hipStream_t s) {
  const bool exact = P.slots == kRecGroups * RPL;
  if constexpr (RPL >= 4) {
    if (v4 && exact) {
      hipLaunchKernelGGL((dense_recurrence_kernel<RPL, true, true>), dim3(grid), dim3(kRecThreads), 0,
                         s, P);
      return;
    }
    if (v4) {
      hipLaunchKernelGGL((dense_recurrence_kernel<RPL, true, false>), dim3(grid), dim3(kRecThreads), 0,
                         s, P);
      return;
    }
  }
  if (exact) {
    hipLaunchKernelGGL((dense_recurrence_kernel<RPL, false, true>), dim3(grid), dim3(kRecThreads), 0,
                       s, P);
  } else {
    hipLaunchKernelGGL((dense_recurrence_kernel<RPL, false, false>), dim3(grid), dim3(kRecThreads), 0,
                       s, P);
  }
}

int32_t launch_dense_sequences(RecParams P, hipStream_t s) {
  P.blocks = (P.width + kRecCols - 1) / kRecCols;
  const int64_t waves = P.batch * P.blocks;
  const int64_t grid = (waves + kRecWaves - 1) / kRecWaves;
  if (grid > (int64_t{1} << 31) - 1) return fail(COWSDM_ELIMIT, "recurrence: batch too large");
  const int groups_rows = (P.slots + kRecGroups - 1) / kRecGroups;   // rows per lane needed
  const uintptr_t align = reinterpret_cast<uintptr_t>(P.wr) | reinterpret_cast<uintptr_t>(P.rr);
  const bool v4 = P.slots % 4 == 0 && align % 16 == 0;
  const unsigned g = static_cast<unsigned>(grid);
  if (groups_rows <= 1) {
    launch_dense_recurrence<1>(P, v4, g, s);
  } else if (groups_rows <= 2) {
    launch_dense_recurrence<2>(P, v4, g, s);
  } else if (groups_rows <= 4) {
    launch_dense_recurrence<4>(P, v4, g, s);
  } else if (groups_rows <= 8) {
    launch_dense_recurrence<8>(P, v4, g, s);
  } else if (groups_rows <= 16) {
    launch_dense_recurrence<16>(P, v4, g, s);
  } else if (groups_rows <= 32) {
    launch_dense_recurrence<32>(P, v4, g, s);
  } else {
    launch_dense_recurrence<64>(P, v4, g, s);
  }
  return launch_status("recurrence");
}

template <int V, int SEG, bool STATES>
int32_t launch_recurrence(RecParams& P, hipStream_t s) {
  auto bytes = [&](int nw) {
    return nw * (P.slots + 1) * kRrRowBytes + 2 * (kDrChunk + kRrPad) * RrRecord<1, 4>::kBytes +
           4 * nw * kRrCols + 16;
  };
  // the waves that D fills, fewer where the tables and the stage would not
  // fit in LDS
  int nw = (P.width + kRrCols - 1) / kRrCols;
  nw = nw > kRrWaves ? kRrWaves : nw;
  // with per-token memories two waves where four would leave CUs idle, for a
  // CU writes 64 bytes a cycle: 87 us against 102 at B = 16, T = 128, N = 256,
  // D = 128; where four fill the chip their 128-byte rows are the better ones
  // (241 us against 266 at B = 64, T = 16, N = 1024, D = 256)
  if (STATES && nw > 2 && P.batch * ((P.width + nw * kRrCols - 1) / (nw * kRrCols)) < kCus) nw = 2;
  while (nw > 1 && bytes(nw) > kRrLds) --nw;
  const int lds = bytes(nw);
  P.blocks = (P.width + nw * kRrCols - 1) / (nw * kRrCols);
  const int64_t grid = kXcds * ((P.batch + kXcds - 1) / kXcds) * P.blocks;
  if (grid > (int64_t{1} << 31) - 1) return fail(COWSDM_ELIMIT, "recurrence: batch too large");
  auto* const kernel = &recurrence_kernel<V, SEG, STATES>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return fail(static_cast<int32_t>(e), "recurrence: %d bytes of LDS", lds);
  }
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)),
                     dim3(nw * kWave + kDrProducers + (STATES ? kDrStoreThreads : 0)), lds, s, P);
  return launch_status("recurrence");
}

template <int V, bool STATES>
int32_t launch_recurrence_slots(RecParams& P, hipStream_t s) {
  if (P.slots <= 4 * kWave) return launch_recurrence<V, 4, STATES>(P, s);
  return launch_recurrence<V, kDrSegments, STATES>(P, s);
}

}  // namespace cowsdm_impl

using namespace cowsdm_impl;

extern "C" int32_t cowsdm_recurrence_forward(const cowsdm_recurrence_t* r, void* stream) {
  if (!r) return fail(COWSDM_EARG, "recurrence: null argument");
  if (r->batch < 0 || r->time < 0 || r->slots <= 0 || r->width <= 0) {
    return fail(COWSDM_EARG, "recurrence: invalid sizes");
  }
  if (r->slots > kRrMaxSlots) {
    return fail(COWSDM_ELIMIT, "recurrence: at most %d slots", kRrMaxSlots);
  }
  if (r->width > (int64_t{1} << 24) || r->slots * r->width >= (int64_t{1} << 31)) {
    return fail(COWSDM_ELIMIT, "recurrence: width too large");
  }
  if (r->batch == 0) return 0;
  if (!r->initial_memory || (!r->readings && r->time > 0)) {
    return fail(COWSDM_EARG, "recurrence: null pointer argument");
  }
  if (r->time > 0 && (!r->write_routes || !r->values || !r->input_gate || !r->erase_gate ||
                      !r->forget_log_gate || !r->read_routes)) {
    return fail(COWSDM_EARG, "recurrence: null pointer argument");
  }
  RecParams P{};
  P.batch = r->batch;
  P.time = r->time;
  P.slots = static_cast<int>(r->slots);
  P.width = static_cast<int>(r->width);
  P.m0 = r->initial_memory;
  P.wr = r->write_routes;
  P.values = r->values;
  P.ig = r->input_gate;
  P.eg = r->erase_gate;
  P.flg = r->forget_log_gate;
  P.rr = r->read_routes;
  P.readings = r->readings;
  P.states = r->states;
  P.final_memory = r->final_memory;
  const uintptr_t align = reinterpret_cast<uintptr_t>(P.m0) |
                          reinterpret_cast<uintptr_t>(P.states) |
                          reinterpret_cast<uintptr_t>(P.final_memory);
  const bool v4 = P.width % 4 == 0 && align % 16 == 0;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  // up to 64 slots and few columns the memory in registers is the faster one
  // with per-token memories (T = 128, D = 64: 56 us against 74 at B = 1, N = 32,
  // 70 against 75 at N = 64; with B = 64, D = 128 98 against 79 and 185 against
  // 87); without them it is not (50 to 54 us against 27 to 30), but both calls
  // have to give the same readings.  The line cannot lie at N or D alone: with
  // either kernel for all of N <= 64 one of these sides loses a third or more.
  // And the sparse sequences' launch, at most 16 waves to 16 columns, has to
  // stay below 2^32 threads.
  // A sequence is handed over with its memory in one of the outputs and the
  // token's number in the low bits of a float.
  P.all_dense = (!P.states && !P.final_memory) || P.time >= kDrMaxTime ||
                (P.slots <= kWave && P.batch * P.width < 4096) ||
                (P.batch + kXcds - 1) * ((P.width + 15) / 16) >= (int64_t{1} << 22);
  if (P.all_dense) return launch_dense_sequences(P, s);
  RecParams sparse = P;
  const int32_t rc =
      P.states ? (v4 ? launch_recurrence_slots<4, true>(sparse, s)
                     : launch_recurrence_slots<1, true>(sparse, s))
               : (v4 ? launch_recurrence_slots<4, false>(sparse, s)
                     : launch_recurrence_slots<1, false>(sparse, s));
  // behind it, from each sequence's first dense token on
  return rc || P.time == 0 ? rc : launch_dense_sequences(P, s);
}

extern "C" int32_t cowsdm_dense_routes(const float* weights, const void* indices,
                                       int32_t index_dtype, int64_t rows, int64_t per_row,
                                       int64_t slots, float* dense, int32_t* bad, void* stream) {
  if (rows < 0 || per_row < 0 || slots <= 0) return fail(COWSDM_EARG, "dense routes: invalid sizes");
  if (per_row > 1024 || slots > (int64_t{1} << 30)) {
    return fail(COWSDM_ELIMIT, "dense routes: shape outside the supported range");
  }
  if (index_dtype != COWSDM_INDEX_INT32 && index_dtype != COWSDM_INDEX_INT64) {
    return fail(COWSDM_EARG, "dense routes: unknown index dtype");
  }
  if (rows == 0) return 0;
  if (!dense || (per_row > 0 && (!weights || !indices))) {
    return fail(COWSDM_EARG, "dense routes: null pointer argument");
  }
  const int64_t total = rows * slots;
  const int64_t grid = (total + 255) / 256;
  if (grid > (int64_t{1} << 31) - 1) return fail(COWSDM_ELIMIT, "dense routes: too many rows");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (index_dtype == COWSDM_INDEX_INT32) {
    hipLaunchKernelGGL(dense_routes_kernel<int32_t>, dim3(static_cast<unsigned>(grid)), dim3(256),
                       0, s, weights, static_cast<const int32_t*>(indices), rows,
                       static_cast<int>(per_row), static_cast<int>(slots), dense, bad);
  } else {
    hipLaunchKernelGGL(dense_routes_kernel<int64_t>, dim3(static_cast<unsigned>(grid)), dim3(256),
                       0, s, weights, static_cast<const int64_t*>(indices), rows,
                       static_cast<int>(per_row), static_cast<int>(slots), dense, bad);
  }
  return launch_status("dense routes");
}
