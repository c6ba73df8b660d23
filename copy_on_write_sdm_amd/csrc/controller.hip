// The SDM controller's per-token work around the copy-on-write step
// (copy_on_write_sdm/inference.py:459-535): before the step, the input
// LayerNorm, the read / write key, value, forget and input projections and
// the gates; after it, the readings LayerNorm, the sigmoid output gate and
// the output projection.  Routes are selected from the keys by
// cowsdm_product_key_routes (routes.hip), or, where that is faster
// (prepare_selects), by the prepare kernel itself once its tokens' keys are
// out (one wave per route row, routes.h): cowsdm_controller_prepare_routes;
// with nothing between two layers, one layer's finish and the next one's
// prepare and routes then share a launch too
// (cowsdm_controller_finish_prepare_routes).
//
// The projections are products [tokens, width] x [width, rows] in float32 on
// the matrix cores (v_mfma_f32_16x16x4_f32): a wave computes tiles of 16 MT
// tokens by 16 NT rows, the normalised tokens in LDS, the weights ([width,
// rows], so 16 NT rows of one input are consecutive) from L2 straight to
// registers.  Inputs are taken 16 at a time, lanes 16 q .. 16 q + 15 holding
// inputs 4 q .. 4 q + 3, one of the four per MFMA; the first and third of
// them sum into one accumulator and the others into a second, so that
// consecutive MFMAs do not wait for each other, and the two are added at the
// end.  Every kernel sums in this order, whatever its tile: a token's outputs
// do not depend on the batch it is in.
//
// Few tokens are bound by the latency of a chain of dependent loads, not by
// arithmetic: there a workgroup takes one token (16 at most), the tile's
// other rows repeating it, so that all of a batch's tokens are in flight at
// once, and every wave loads the weights of its first tile before it waits
// for its tokens.  Many tokens are bound by the matrix cores and by bytes
// about alike: there a workgroup is one or a few waves, so that those of a
// compute unit are at different stages, loading, multiplying and storing at
// once (131,072 tokens at width 128, N = 256: prepare with 13 waves in step
// 233 us, with one 138).  What is left of them is the matrix cores' own time
// (49 and 56 us) and the vector instructions of the norms, gates and stores,
// which 32-bit MFMAs do not run beside.
//
// 131,072 tokens: prepare 490 -> 138 us, finish 330 -> 114; 2,331 tokens of
// width 400, 4 heads, N = 1,024: 96 -> 36 and 86 -> 39; 64 tokens: 9.0 -> 6.8
// and 8.2 -> 6.7 us, each against the half-wave dot products before.

#include "common.h"
#include "routes.h"

namespace cowsdm_impl {

constexpr int kCtlMaxWidth = 1024;    // LDS: 2 x 16 tokens x width floats
constexpr int kCtlTile = 16;          // tokens and rows of an MFMA tile
constexpr int kCtlGroup = 16;         // inputs of one load per lane (4 MFMAs)
// groups of weights a wave has in flight: a projection of 128 inputs whole
// where one tile waits for them, 32 or 64 MFMAs ahead otherwise
template <int MT, int NT>
constexpr int ctl_chunk() {
  return MT * NT == 1 ? 8 : 4;
}
constexpr int kCtlMaxWaves = 16;
constexpr int kCtlThreads = kCtlMaxWaves * kWave;
constexpr int kCtlManyThreads = 4 * kWave;   // workgroups of many tokens
constexpr int kCtlPad = 4;            // floats after a token's row in LDS
constexpr int kCtlPrepareWaves = 1;   // a prepare's of many tokens
constexpr int kCtlFewTokens = 512;    // one row a lane up to here
constexpr int kCtlUnits = 256;        // workgroups that fill the device's compute units

struct CtlParams {
  cowsdm_controller_t c;
  int64_t batch;
  const float* tokens;        // prepare: [batch, width]
  const float* normalized;    // finish: [batch, width]
  const float* reading;       // finish: [batch * heads, head_width]
  float* out_normalized;      // prepare
  float* read_keys;           // prepare: [batch * heads, key_width]
  float* write_keys;
  float* values;              // prepare: [batch * heads, head_width]
  float* input_gate;          // prepare: [batch * heads]
  float* forget_log_gate;
  float* out;                 // finish: [batch, width]
  const float* residual;      // finish: [batch, width] or null
  float* out_sum;             // finish: residual + out, when residual is set
  int width, heads, head_width, key_width, rows;
  int tokens_per_group;       // tokens of a workgroup, at most 16 * MT
  int ld;                     // floats from one token's row in LDS to the next
};

// The routes the prepare kernel selects itself (prepare_selects): every
// token's read and write route rows, one wave per row.
struct CtlRoutes {
  int root, read_sub, read_k, write_sub, write_k;
  float* read_weights;        // [batch * heads, read_k]
  int64_t* read_indices;
  float* write_weights;       // [batch * heads, write_k]
  int64_t* write_indices;
};

// Sum over the 16 lanes of a DPP row, the same in all of them: neighbours,
// pairs, quads (row_half_mirror), eights (row_mirror).
__device__ __forceinline__ float row_sum(float v) {
#define COWSDM_ROW_ADD(ctrl)                                                     \
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true))
  COWSDM_ROW_ADD(0xB1);
  COWSDM_ROW_ADD(0x4E);
  COWSDM_ROW_ADD(0x141);
  COWSDM_ROW_ADD(0x140);
#undef COWSDM_ROW_ADD
  return v;
}

// LayerNorm of n floats by 16 lanes, as torch's layer_norm: the mean, the
// biased variance, then (x - mean) / sqrt(var + eps) * w + b, into dst (LDS;
// src may be dst) and, when it is set, copy.  V floats a lane at a time: 4
// when n and the offsets into the rows are multiples of 4.
template <int V>
__device__ __forceinline__ void row_layer_norm_v(const float* src, float* dst, float* copy, int n,
                                                 const float* w, const float* b, float eps) {
  using Vec = __attribute__((ext_vector_type(V))) float;
  const int lane = static_cast<int>(threadIdx.x) % kCtlTile * V;
  float s = 0.0f;
#pragma unroll 2
  for (int i = lane; i < n; i += kCtlTile * V) {
    const Vec x = *reinterpret_cast<const Vec*>(src + i);
    *reinterpret_cast<Vec*>(dst + i) = x;
#pragma unroll
    for (int k = 0; k < V; ++k) s += x[k];
  }
  const float mean = row_sum(s) / static_cast<float>(n);
  float v = 0.0f;
#pragma unroll 2
  for (int i = lane; i < n; i += kCtlTile * V) {
    const Vec x = *reinterpret_cast<const Vec*>(dst + i);
#pragma unroll
    for (int k = 0; k < V; ++k) v = __builtin_fmaf(x[k] - mean, x[k] - mean, v);
  }
  const float var = row_sum(v) / static_cast<float>(n);
  const float rstd = 1.0f / sqrtf(var + eps);
#pragma unroll 2
  for (int i = lane; i < n; i += kCtlTile * V) {
    const Vec x = *reinterpret_cast<const Vec*>(dst + i);
    const Vec wv = *reinterpret_cast<const Vec*>(w + i);
    const Vec bv = *reinterpret_cast<const Vec*>(b + i);
    Vec y;
#pragma unroll
    for (int k = 0; k < V; ++k) y[k] = (x[k] - mean) * rstd * wv[k] + bv[k];
    *reinterpret_cast<Vec*>(dst + i) = y;
    if (copy) *reinterpret_cast<Vec*>(copy + i) = y;
  }
}

__device__ __forceinline__ void row_layer_norm(const float* src, float* dst, float* copy, int n,
                                               const float* w, const float* b, float eps) {
  if (n % 4 == 0) {
    row_layer_norm_v<4>(src, dst, copy, n, w, b, eps);
  } else {
    row_layer_norm_v<1>(src, dst, copy, n, w, b, eps);
  }
}

// torch.nn.functional.softplus with beta 1 and threshold 20
__device__ __forceinline__ float softplus(float x) { return x > 20.0f ? x : log1pf(expf(x)); }
__device__ __forceinline__ float sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }

using v4f = __attribute__((ext_vector_type(4))) float;

// A wave's weights of C groups of inputs for 16 NT rows: lane 16 q + n holds
// input 16 g + 4 q + s of row j0 + NT n + u at [(4 g + s) NT + u].  NT == 2:
// the number of rows is even.
template <int NT, int C>
struct CtlWeights {
  float w[4 * C * NT];
};

// The lane's first row; rows past the last ones repeat those, unused.
template <int NT>
__device__ __forceinline__ int ctl_row(int j0, int rows) {
  const int j = j0 + NT * (static_cast<int>(threadIdx.x) % kCtlTile);
  return j < rows ? j : rows - NT;
}

// Where the lane's weights of a group are in wt [width, rows], in bytes (rows
// stay below 2^24).
template <int NT>
__device__ __forceinline__ uint32_t ctl_lane_offset(int j0, int rows) {
  const int q = (static_cast<int>(threadIdx.x) % kWave) / kCtlTile;
  return 4 * (static_cast<uint32_t>(4 * q) * rows + ctl_row<NT>(j0, rows));
}

// Group `group` (whole groups only: the last one again past it, unused) of wt
// into f's place g.
template <int NT, int C>
__device__ __forceinline__ void load_group(CtlWeights<NT, C>& f, int g, const float* wt,
                                           int width, int rows, uint32_t at, int group) {
  using Vec = __attribute__((ext_vector_type(NT))) float;
  const int k0 = min(group, width / kCtlGroup - 1) * kCtlGroup;
  const char* const base = reinterpret_cast<const char*>(wt + static_cast<int64_t>(k0) * rows);
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const Vec v = *reinterpret_cast<const Vec*>(base + (at + static_cast<uint32_t>(4 * s) * rows));
#pragma unroll
    for (int u = 0; u < NT; ++u) f.w[(4 * g + s) * NT + u] = v[u];
  }
}

// The first C groups.
template <int NT, int C>
__device__ __forceinline__ void load_weights(CtlWeights<NT, C>& f, const float* wt, int width,
                                             int rows, int j0) {
  if (width < kCtlGroup) return;
  const uint32_t at = ctl_lane_offset<NT>(j0, rows);
#pragma unroll
  for (int g = 0; g < C; ++g) {
    load_group(f, g, wt, width, rows, at, g);
    __builtin_amdgcn_sched_barrier(0);   // in the order of their use
  }
}

// acc[m][u]: lane 16 q + n's tokens 16 m + 4 q + i (i = 0 .. 3) of row
// j0 + NT n + u, from the tokens in LDS (x, stride ld, inputs up to a
// multiple of 16) and wt; f holds the weights of the first chunk.
// Tokens from `tokens` on repeat the last one.
template <int MT, int NT>
__device__ __forceinline__ void project_tile(const float* x, int ld, int tokens, const float* wt,
                                             int width, int rows, int j0,
                                             CtlWeights<NT, ctl_chunk<MT, NT>()>& f,
                                             v4f (&acc)[MT][NT]) {
  constexpr int C = ctl_chunk<MT, NT>();
  const int lane = static_cast<int>(threadIdx.x) % kWave;
  const float* row[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int t = m * kCtlTile + lane % kCtlTile;
    row[m] = x + (t < tokens ? t : tokens - 1) * ld + 4 * (lane / kCtlTile);
  }
  v4f sum[2][MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
#pragma unroll
    for (int u = 0; u < NT; ++u) sum[0][m][u] = sum[1][m][u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  }
  auto inputs = [&](v4f (&a)[MT], int g) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < MT; ++m) a[m] = *reinterpret_cast<const v4f*>(row[m] + g * kCtlGroup);
  };
  auto multiply = [&](const v4f (&a)[MT], const float* w) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
#pragma unroll
        for (int u = 0; u < NT; ++u) {
          sum[s & 1][m][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(
              a[m][s], w[s * NT + u], sum[s & 1][m][u], 0, 0, 0);
        }
      }
    }
  };
  // all chunks but the last one load the next one as they go, each group into
  // the registers it has just used, on no condition: how many loads are
  // behind a group's is then known, and its wait leaves them in flight
  const int whole = width / kCtlGroup;
  const uint32_t at = ctl_lane_offset<NT>(j0, rows);
  v4f a[MT], next_a[MT];
  inputs(a, 0);
  int g0 = 0;
  for (; g0 + C < whole; g0 += C) {
#pragma unroll
    for (int g = 0; g < C; ++g) {
      inputs(next_a, g0 + g + 1);
      __builtin_amdgcn_sched_barrier(0);   // the next inputs leave before this group's MFMAs
      multiply(a, f.w + 4 * g * NT);
      load_group(f, g, wt, width, rows, at, g0 + g + C);
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m] = next_a[m];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int g = 0; g < C; ++g) {
    if (g0 + g < whole) {
      inputs(next_a, min(g0 + g + 1, whole - 1));
      __builtin_amdgcn_sched_barrier(0);
      multiply(a, f.w + 4 * g * NT);
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m] = next_a[m];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (width % kCtlGroup) {
    // the tokens' inputs past the width are 0; so are these weights, which
    // need not be finite past the end of a row
    float w[4 * NT];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = whole * kCtlGroup + 4 * (lane / kCtlTile) + s;
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        w[s * NT + u] =
            k < width ? wt[static_cast<int64_t>(k) * rows + ctl_row<NT>(j0, rows) + u] : 0.0f;
      }
    }
    inputs(a, whole);
    multiply(a, w);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) {
#pragma unroll
    for (int u = 0; u < NT; ++u) acc[m][u] = sum[0][m][u] + sum[1][m][u];
  }
}

__device__ __forceinline__ int group_tokens(const CtlParams& P, int64_t b0) {
  return static_cast<int>(P.batch - b0 < P.tokens_per_group ? P.batch - b0 : P.tokens_per_group);
}

// inputs from the width up to a multiple of 16 of `tokens` rows in LDS
__device__ __forceinline__ void zero_tail(float* x, int ld, int tokens, int width) {
  const int to = (width + kCtlGroup - 1) / kCtlGroup * kCtlGroup;
  for (int t = static_cast<int>(threadIdx.x) / kCtlTile; t < tokens;
       t += static_cast<int>(blockDim.x) / kCtlTile) {
    const int i = width + static_cast<int>(threadIdx.x) % kCtlTile;
    if (i < to) x[t * ld + i] = 0.0f;
  }
}

// f(token, its values + their biases) for a tile's values of this lane
template <int MT, int NT, class F>
__device__ __forceinline__ void each_value(const v4f (&acc)[MT][NT], const float* bias, int j,
                                           int tokens, F f) {
  const int q = (static_cast<int>(threadIdx.x) % kWave) / kCtlTile;
  float b[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) b[u] = bias[j + u];
  auto all = [&](auto whole) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = m * kCtlTile + 4 * q + i;
        if (decltype(whole)::value || t < tokens) {
          float y[NT];
#pragma unroll
          for (int u = 0; u < NT; ++u) y[u] = acc[m][u][i] + b[u];
          f(t, y);
        }
      }
    }
  };
  // without a test per value where every token is there (one tile's are few)
  if (MT > 1 && tokens == MT * kCtlTile) {
    all(std::true_type{});
  } else {
    all(std::false_type{});
  }
}

// prepare of the workgroup's tokens for the row tiles (16 NT rows each)
// first_tile + wave, + waves, ... below end_tile; x: their rows in LDS, with
// FROM_LDS already holding the tokens (the previous layer's finish put them
// there); `weights`: the first chunk of the wave's first tile.  With
// `store_norm` the normalised tokens are stored.
template <int MT, int NT, bool FROM_LDS>
__device__ __forceinline__ void controller_prepare_body(
    const CtlParams& P, float* x, CtlWeights<NT, ctl_chunk<MT, NT>()>& weights, int first_tile,
    int end_tile, bool store_norm) {
  using Vec = __attribute__((ext_vector_type(NT))) float;
  const int W = P.width, H = P.heads, KW = P.key_width;
  const int64_t b0 = static_cast<int64_t>(blockIdx.x) * P.tokens_per_group;
  const int T = group_tokens(P, b0);
  const int tid = static_cast<int>(threadIdx.x);
  const int waves = static_cast<int>(blockDim.x) / kWave;
  for (int t = tid / kCtlTile; t < T; t += static_cast<int>(blockDim.x) / kCtlTile) {
    row_layer_norm(FROM_LDS ? x + t * P.ld : P.tokens + (b0 + t) * W, x + t * P.ld,
                   store_norm ? P.out_normalized + (b0 + t) * W : nullptr, W, P.c.norm_weight,
                   P.c.norm_bias, P.c.norm_eps);
  }
  zero_tail(x, P.ld, T, W);
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  // rows: read keys (H x KW), write keys (H x KW), values (W), forget (H),
  // input (H); a token's keys, values and gates of all heads are consecutive.
  // With NT == 2 (even W) the first three begin and end at even rows.
  for (int tile = first_tile + wave; tile < end_tile; tile += waves) {
    const int j0 = tile * kCtlTile * NT;
    if (tile >= first_tile + waves) load_weights(weights, P.c.proj_weight_t, W, P.rows, j0);
    v4f acc[MT][NT];
    project_tile<MT, NT>(x, P.ld, T, P.c.proj_weight_t, W, P.rows, j0, weights, acc);
    const int j = j0 + NT * (tid % kCtlTile);
    if (j >= P.rows) continue;
    const int keys = H * KW;
    int r = j;
    if (r < 2 * keys + W) {
      float* to = P.read_keys;
      int stride = keys;
      if (r >= 2 * keys) {
        r -= 2 * keys;
        to = P.values;
        stride = W;
      } else if (r >= keys) {
        r -= keys;
        to = P.write_keys;
      }
      to += b0 * stride + r;
      each_value<MT, NT>(acc, P.c.proj_bias, j, T, [&](int t, const float (&y)[NT])
          __attribute__((always_inline)) {
        Vec v;
#pragma unroll
        for (int u = 0; u < NT; ++u) v[u] = y[u];
        *reinterpret_cast<Vec*>(to + static_cast<uint32_t>(t * stride)) = v;
      });
      continue;
    }
    r -= 2 * keys + W;
    each_value<MT, NT>(acc, P.c.proj_bias, j, T, [&](int t, const float (&y)[NT])
        __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < NT; ++u) {
        const int h = r + u;
        if (h < H) {
          P.forget_log_gate[(b0 + t) * H + h] =
              -expf(P.c.a_log[h]) * softplus(y[u] + P.c.dt_bias[h]);
        } else {
          P.input_gate[(b0 + t) * H + h - H] = sigmoid(y[u]);
        }
      }
    });
  }
}

// blockIdx.y: the share of the row tiles
template <int MT, int NT>
__global__ __launch_bounds__(MT == 1 ? kCtlThreads : kCtlManyThreads, MT == 1 ? 4 : 3) void
controller_prepare_kernel(CtlParams P, int tiles_each) {
  extern __shared__ float lds[];
  const int tiles = (P.rows + kCtlTile * NT - 1) / (kCtlTile * NT);
  const int first = static_cast<int>(blockIdx.y) * tiles_each;
  const int end = first + tiles_each < tiles ? first + tiles_each : tiles;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  CtlWeights<NT, ctl_chunk<MT, NT>()> weights;
  if (first + wave < end) {
    load_weights(weights, P.c.proj_weight_t, P.width, P.rows, (first + wave) * kCtlTile * NT);
  }
  controller_prepare_body<MT, NT, false>(P, lds, weights, first, end, blockIdx.y == 0);
}

// The read and write routes of the workgroup's tokens from the keys its
// threads stored (visible to the whole workgroup after a barrier), one wave
// per route row.
struct RouteStage {
  float val[kCtlMaxWaves][kRouteMaxSelected];
  int pos[kCtlMaxWaves][kRouteMaxSelected];
  float pool_val[kCtlMaxWaves][kWave];
  int pool_pos[kCtlMaxWaves][kWave];
};

// M: how a row's routes are selected, 0 sorted across lanes (then the stage
// is not used), else product_key_route_row's M
template <int M>
__device__ __forceinline__ void controller_route_row(const float* keys, int64_t row, int root,
                                                     int sub, int k, float* weights,
                                                     int64_t* indices, RouteStage* st,
                                                     int wave) {
  if constexpr (M == 0) {
    product_key_route_row_sorted(keys, row, root, sub, k, weights, indices);
  } else {
    product_key_route_row<1, M>(keys, row, root, sub, k, weights, indices, st->val[wave],
                                st->pos[wave], st->pool_val[wave], st->pool_pos[wave]);
  }
}

template <int MR, int MW>
__device__ __forceinline__ void controller_routes_part(const CtlParams& P, const CtlRoutes& R) {
  RouteStage* stage = nullptr;
  if constexpr (MR + MW > 0) {
    __shared__ RouteStage shared;
    stage = &shared;
  }
  const int64_t b0 = static_cast<int64_t>(blockIdx.x) * P.tokens_per_group;
  const int rows = group_tokens(P, b0) * P.heads;
  const int wave = static_cast<int>(threadIdx.x) / kWave;
  for (int task = wave; task < 2 * rows; task += static_cast<int>(blockDim.x) / kWave) {
    if (task < rows) {
      controller_route_row<MR>(P.read_keys, b0 * P.heads + task, R.root, R.read_sub, R.read_k,
                               R.read_weights, R.read_indices, stage, wave);
    } else {
      controller_route_row<MW>(P.write_keys, b0 * P.heads + task - rows, R.root, R.write_sub,
                               R.write_k, R.write_weights, R.write_indices, stage, wave);
    }
  }
}

// prepare, then the routes of the workgroup's tokens
template <int MR, int MW>
__global__ __launch_bounds__(kCtlThreads) void controller_prepare_routes_kernel(CtlParams P,
                                                                                CtlRoutes R) {
  extern __shared__ float lds[];
  const int tiles = (P.rows + kCtlTile - 1) / kCtlTile;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  CtlWeights<1, ctl_chunk<1, 1>()> weights;
  if (wave < tiles) {
    load_weights(weights, P.c.proj_weight_t, P.width, P.rows, wave * kCtlTile);
  }
  controller_prepare_body<1, 1, false>(P, lds, weights, 0, tiles, true);
  __syncthreads();
  controller_routes_part<MR, MW>(P, R);
}

// finish of the workgroup's tokens.  lds: the normalised inputs, then the
// normalised readings, which become gate * normalised readings; with TO_LDS
// the residual sums (the next layer's inputs) end up in the first of the two,
// its inputs being dead once the gate is applied.  `weights`: the first chunk
// of the wave's first tile, of the gate's for the waves below `split` and of
// the output projection's for the rest.  The gate's tiles go to the waves
// below `split` and the output projection's to the waves from `split` on
// (both to all waves when split is 0: then the weights are the gate's).
template <int MT, int NT, bool TO_LDS>
__device__ __forceinline__ void controller_finish_body(
    const CtlParams& P, float* lds, int split, CtlWeights<NT, ctl_chunk<MT, NT>()>& weights) {
  using Vec = __attribute__((ext_vector_type(NT))) float;
  const int W = P.width, HW = P.head_width;
  float* const nrm = lds;
  float* const rd = lds + P.tokens_per_group * P.ld;
  const int64_t b0 = static_cast<int64_t>(blockIdx.x) * P.tokens_per_group;
  const int T = group_tokens(P, b0);
  const int tid = static_cast<int>(threadIdx.x);
  const int rows = static_cast<int>(blockDim.x) / kCtlTile;   // 16-lane rows
  // a token's readings [heads, head_width] are its `width` contiguous floats
  for (int g = tid / kCtlTile; g < T * P.heads; g += rows) {
    const int t = g / P.heads, h = g - t * P.heads;
    row_layer_norm(P.reading + (b0 + t) * W + h * HW, rd + t * P.ld + h * HW, nullptr, HW,
                   P.c.read_norm_weight, P.c.read_norm_bias, P.c.read_norm_eps);
  }
  if (W % 4 == 0) {
    for (int t = tid / kCtlTile; t < T; t += rows) {
#pragma unroll 2
      for (int i = tid % kCtlTile * 4; i < W; i += kCtlTile * 4) {
        *reinterpret_cast<v4f*>(nrm + t * P.ld + i) =
            *reinterpret_cast<const v4f*>(P.normalized + (b0 + t) * W + i);
      }
    }
  } else {
    for (int t = tid / kCtlTile; t < T; t += rows) {
      for (int i = tid % kCtlTile; i < W; i += kCtlTile) {
        nrm[t * P.ld + i] = P.normalized[(b0 + t) * W + i];
      }
    }
  }
  zero_tail(nrm, P.ld, T, W);
  zero_tail(rd, P.ld, T, W);
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int waves = static_cast<int>(blockDim.x) / kWave;
  const int tiles = (W + kCtlTile * NT - 1) / (kCtlTile * NT);
  const int gate_waves = split ? split : waves, out_waves = split ? waves - split : waves;
  for (int tile = wave; wave < gate_waves && tile < tiles; tile += gate_waves) {
    const int j0 = tile * kCtlTile * NT;
    if (tile >= gate_waves) load_weights(weights, P.c.gate_weight_t, W, W, j0);
    v4f acc[MT][NT];
    project_tile<MT, NT>(nrm, P.ld, T, P.c.gate_weight_t, W, W, j0, weights, acc);
    const int j = j0 + NT * (tid % kCtlTile);
    if (j >= W) continue;
    each_value<MT, NT>(acc, P.c.gate_bias, j, T, [&](int t, const float (&y)[NT])
        __attribute__((always_inline)) {
      Vec* const at = reinterpret_cast<Vec*>(rd + t * P.ld + j);
      Vec v = *at;
#pragma unroll
      for (int u = 0; u < NT; ++u) v[u] = sigmoid(y[u]) * v[u];
      *at = v;
    });
  }
  const int out_wave = wave - split;
  if (!split && wave < tiles) {
    load_weights(weights, P.c.out_weight_t, W, W, wave * kCtlTile * NT);
  }
  __syncthreads();
  for (int tile = out_wave; out_wave >= 0 && tile < tiles; tile += out_waves) {
    const int j0 = tile * kCtlTile * NT;
    if (tile >= out_waves) load_weights(weights, P.c.out_weight_t, W, W, j0);
    v4f acc[MT][NT];
    project_tile<MT, NT>(rd, P.ld, T, P.c.out_weight_t, W, W, j0, weights, acc);
    const int j = j0 + NT * (tid % kCtlTile);
    if (j >= W) continue;
    each_value<MT, NT>(acc, P.c.out_bias, j, T, [&](int t, const float (&y)[NT])
        __attribute__((always_inline)) {
      const uint32_t at = static_cast<uint32_t>(t * W + j);
      Vec v;
#pragma unroll
      for (int u = 0; u < NT; ++u) v[u] = y[u];
      *reinterpret_cast<Vec*>(P.out + b0 * W + at) = v;
      if (P.residual) {
        Vec next = *reinterpret_cast<const Vec*>(P.residual + b0 * W + at);
#pragma unroll
        for (int u = 0; u < NT; ++u) next[u] = next[u] + y[u];
        *reinterpret_cast<Vec*>(P.out_sum + b0 * W + at) = next;
        if constexpr (TO_LDS) *reinterpret_cast<Vec*>(nrm + t * P.ld + j) = next;
      }
    });
  }
}

// The first chunk of the wave's first tile in a finish (see there).
template <int NT, int C>
__device__ __forceinline__ void load_finish_weights(CtlWeights<NT, C>& weights,
                                                    const CtlParams& P, int split) {
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int tiles = (P.width + kCtlTile * NT - 1) / (kCtlTile * NT);
  const bool gate = split == 0 || wave < split;
  const int tile = gate ? wave : wave - split;
  if (tile < tiles) {
    load_weights(weights, gate ? P.c.gate_weight_t : P.c.out_weight_t, P.width, P.width,
                 tile * kCtlTile * NT);
  }
}

template <int MT, int NT>
__global__ __launch_bounds__(MT == 1 ? kCtlThreads : kCtlManyThreads, 4) void
controller_finish_kernel(CtlParams P, int split) {
  extern __shared__ float lds[];
  CtlWeights<NT, ctl_chunk<MT, NT>()> weights;
  load_finish_weights(weights, P, split);
  controller_finish_body<MT, NT, false>(P, lds, split, weights);
}

// one layer's finish with the residual add, then the next layer's prepare
// and routes on the same tokens, whose inputs the finish left in LDS
template <int MR, int MW>
__global__ __launch_bounds__(kCtlThreads) void controller_finish_prepare_routes_kernel(
    CtlParams F, CtlParams P, CtlRoutes R, int split) {
  extern __shared__ float lds[];
  const int tiles = (P.rows + kCtlTile - 1) / kCtlTile;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  CtlWeights<1, ctl_chunk<1, 1>()> finish, weights;
  load_finish_weights(finish, F, split);
  if (wave < tiles) {
    load_weights(weights, P.c.proj_weight_t, P.width, P.rows, wave * kCtlTile);
  }
  controller_finish_body<1, 1, true>(F, lds, split, finish);
  __syncthreads();
  controller_prepare_body<1, 1, true>(P, lds, weights, 0, tiles, true);
  __syncthreads();
  controller_routes_part<MR, MW>(P, R);
}

namespace {

int32_t check_controller(const cowsdm_controller_t* c, int64_t batch, CtlParams& P) {
  if (!c) return fail(COWSDM_EARG, "controller: null controller");
  if (batch < 0) return fail(COWSDM_EARG, "controller: negative batch");
  if (c->width <= 0 || c->heads <= 0 || c->width % c->heads != 0) {
    return fail(COWSDM_EARG, "width must be divisible by memory_heads");
  }
  if (c->width > kCtlMaxWidth) {
    return fail(COWSDM_ELIMIT, "controller: width <= %d on the HIP path (got %lld)",
                kCtlMaxWidth, static_cast<long long>(c->width));
  }
  int64_t root = 0;
  while ((root + 1) * (root + 1) <= c->slots) ++root;
  if (c->slots < 1 || root * root != c->slots) {
    return fail(COWSDM_EARG, "faithful SDM slots must be a perfect square");
  }
  P.c = *c;
  P.batch = batch;
  P.width = static_cast<int>(c->width);
  P.heads = static_cast<int>(c->heads);
  P.head_width = static_cast<int>(c->width / c->heads);
  P.key_width = static_cast<int>(2 * root);
  const int64_t rows = 2 * c->heads * 2 * root + c->width + 2 * c->heads;
  if (rows > (int64_t{1} << 24)) return fail(COWSDM_ELIMIT, "controller: too many projection rows");
  P.rows = static_cast<int>(rows);
  P.ld = (P.width + kCtlGroup - 1) / kCtlGroup * kCtlGroup + kCtlPad;
  return 0;
}

// Few tokens: one per workgroup until the workgroups fill the device, at
// most a tile's 16.
int few_tokens(int64_t batch) {
  const int64_t each = (batch + kCtlUnits - 1) / kCtlUnits;
  return static_cast<int>(each > kCtlTile ? kCtlTile : each);
}

// Waves for `tiles` row tiles: as few rounds as 16 waves take, evenly.
int tile_waves(int tiles) {
  const int rounds = (tiles + kCtlMaxWaves - 1) / kCtlMaxWaves;
  return (tiles + rounds - 1) / rounds;
}

// Whether `batch` tokens fill the device 32 to a workgroup, with at most
// 40 KiB of LDS for its `rows` rows a token (four workgroups to a compute
// unit): every weight is then used for two tiles of tokens.
bool many_tokens(const CtlParams& P, int rows) {
  return P.batch >= 2 * kCtlTile * kCtlUnits && rows * 2 * kCtlTile * P.ld * 4 <= 40 * 1024;
}

int64_t token_groups(const CtlParams& P) {
  return (P.batch + P.tokens_per_group - 1) / P.tokens_per_group;
}

// `rows` rows a token of dynamic LDS
size_t token_lds(const CtlParams& P, int rows) {
  return sizeof(float) * rows * P.tokens_per_group * P.ld;
}

// Past 64 KiB a kernel's dynamic LDS has to be asked for.
int32_t allow_lds(const void* kernel, size_t lds) {
  if (lds <= 64 * 1024) return 0;
  const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           static_cast<int>(lds));
  return e == hipSuccess ? 0 : fail(static_cast<int32_t>(e), "controller: %zu bytes of LDS", lds);
}

}  // namespace
}  // namespace cowsdm_impl

using namespace cowsdm_impl;

extern "C" int64_t cowsdm_controller_rows(int64_t width, int64_t heads, int64_t slots) {
  int64_t root = 0;
  while ((root + 1) * (root + 1) <= slots) ++root;
  if (width <= 0 || heads <= 0 || slots < 1 || root * root != slots) return -1;
  return 2 * heads * 2 * root + width + 2 * heads;
}

namespace {

int32_t prepare_params(const cowsdm_controller_t* c, const float* tokens, int64_t batch,
                       float* normalized, float* read_keys, float* write_keys, float* values,
                       float* input_gate, float* forget_log_gate, CtlParams& P) {
  if (int32_t e = check_controller(c, batch, P)) return e;
  if (batch == 0) return 0;
  if (!tokens || !normalized || !read_keys || !write_keys || !values || !input_gate ||
      !forget_log_gate || !c->norm_weight || !c->norm_bias || !c->proj_weight_t ||
      !c->proj_bias || !c->a_log || !c->dt_bias) {
    return fail(COWSDM_EARG, "controller prepare: null pointer argument");
  }
  P.tokens = tokens;
  P.out_normalized = normalized;
  P.read_keys = read_keys;
  P.write_keys = write_keys;
  P.values = values;
  P.input_gate = input_gate;
  P.forget_log_gate = forget_log_gate;
  if (batch > (int64_t{1} << 31) - 1) {
    return fail(COWSDM_ELIMIT, "controller: batch too large");
  }
  return 0;
}

template <int MR, int MW>
int32_t launch_prepare_routes(CtlParams P, const CtlRoutes& R, hipStream_t s) {
  P.tokens_per_group = few_tokens(P.batch);
  const size_t lds = token_lds(P, 1);   // at most 256 inputs a token (prepare_selects)
  auto* const kernel = &controller_prepare_routes_kernel<MR, MW>;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(token_groups(P))), dim3(kCtlThreads),
                     lds, s, P, R);
  return launch_status("controller prepare routes");
}

template <int MR, int MW>
int32_t launch_finish_prepare_routes(CtlParams F, CtlParams P, const CtlRoutes& R,
                                     hipStream_t s) {
  F.tokens_per_group = P.tokens_per_group = few_tokens(P.batch);
  const size_t lds = token_lds(P, 2);
  auto* const kernel = &controller_finish_prepare_routes_kernel<MR, MW>;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(token_groups(P))), dim3(kCtlThreads),
                     lds, s, F, P, R, kCtlMaxWaves / 2);
  return launch_status("controller finish and prepare");
}

template <int MT, int NT>
int32_t launch_prepare(CtlParams P, hipStream_t s) {
  P.tokens_per_group = MT * kCtlTile;
  const int64_t groups = token_groups(P);
  const int tiles = (P.rows + kCtlTile * NT - 1) / (kCtlTile * NT);
  // few groups of tokens: their row tiles are shared out, at least 4 each, to
  // about four workgroups a compute unit (2,331 tokens of width 400, 920
  // rows: one 48 us, two 39, four 36)
  int64_t shares = std::min<int64_t>((tiles + 3) / 4,
                                     std::max<int64_t>(1, 4 * kCtlUnits / groups));
  const int each = static_cast<int>((tiles + shares - 1) / shares);
  shares = (tiles + each - 1) / each;
  const int waves = MT > 1 ? kCtlPrepareWaves : std::max(4, (tile_waves(each) + 1) / 2);
  const size_t lds = token_lds(P, 1);
  auto* const kernel = &controller_prepare_kernel<MT, NT>;
  if (int32_t e = allow_lds(reinterpret_cast<const void*>(kernel), lds)) return e;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(groups), static_cast<unsigned>(shares)),
                     dim3(waves * kWave), lds, s, P, each);
  return launch_status("controller prepare");
}

template <int MT, int NT>
int32_t launch_finish(CtlParams P, hipStream_t s) {
  P.tokens_per_group = MT > 1 ? MT * kCtlTile : few_tokens(P.batch);
  const int tiles = (P.width + kCtlTile * NT - 1) / (kCtlTile * NT);
  // up to 8 tiles each, the gate and the output projection have waves of
  // their own, so that both have their weights before the tokens arrive;
  // not for many tokens, where the idle half would be missed
  const int split = MT == 1 && NT == 1 && tiles <= kCtlMaxWaves / 2 ? tiles : 0;
  const int waves = MT > 1 ? std::min(tiles, kCtlManyThreads / kWave)
                    : split ? 2 * split
                            : tile_waves(tiles);
  const size_t lds = token_lds(P, 2);
  auto* const kernel = &controller_finish_kernel<MT, NT>;
  if (int32_t e = allow_lds(reinterpret_cast<const void*>(kernel), lds)) return e;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(token_groups(P))), dim3(waves * kWave),
                     lds, s, P, split);
  return launch_status("controller finish");
}

// Two rows a lane (NT == 2: half the loads and stores, twice the bytes of
// each) where the rows are even and there is work enough that a tile's time
// does not matter: not for the few tokens of a decode step.
template <class One, class Two, class Many>
int32_t by_tokens(const CtlParams& P, int lds_rows, One one, Two two, Many many) {
  const bool even = P.width % 2 == 0;
  if (even && many_tokens(P, lds_rows)) return many();
  return even && P.batch > kCtlFewTokens ? two() : one();
}

// How a wave selects its rows' routes (controller_route_row's M).
int route_m(const CtlRoutes& R, int sub, int k) {
  return route_row_sorted(R.root, k) ? 0 : route_pair_m(sub, k);
}

// Whether a prepare selects its routes itself, in workgroups of 16 waves that
// project every row of their tokens: `rows` route rows (of a read or write
// route each) and P's projection.  Its row tiles then take a round of the
// waves each 16, and a round about as long as its chunks of 128 inputs, where
// the separate prepare shares the tiles out to more workgroups.  The two more
// launches take 4 us where the kernels are short and 6 us of the host
// (prepare_sdm_step 22 us against 28), so the line lies where the fused kernel
// passes that.  16 tokens, rounds x chunks: 1 (width 128, N = 256, 1 head)
// 8.7 us against 13.0, 3 (4 heads of N = 1,024) 14.0 against 12.6, 4 (width
// 256, 2 heads) 16.8 against 13.3, 5 (width 128, 8 heads of N = 1,024) 20
// against 12.5, 8 (width 256, 4 heads of N = 1,024) 26 against 14, 16 (width
// 400, 4 heads of N = 1,024) 45 against 16, 72 (width 1,024, 8 heads) 218
// against 21.  And from more tokens than one workgroup of 16 each on every
// compute unit on, a second one waits: 4,096 rows of 1 head 15.8 against 17.5,
// 6,000 28 against 20; of 4 heads 17.9 against 17.4, 22.9 against 20.6 at 8,192.
bool prepare_selects(const CtlParams& P, int root, int64_t rows) {
  const int rounds = (P.rows + kCtlTile * kCtlMaxWaves - 1) / (kCtlTile * kCtlMaxWaves);
  const int chunk = kCtlGroup * ctl_chunk<1, 1>();
  return root <= kWave && rounds * ((P.width + chunk - 1) / chunk) <= 5 &&
         rows <= kCtlTile * kCtlUnits;
}

// The route geometry of `reads` and `writes` selections over c's slots and
// the four output pointers (checked once batch > 0).
int32_t route_params(const cowsdm_controller_t* c, int64_t batch, int64_t reads, int64_t writes,
                     float* read_weights, int64_t* read_indices, float* write_weights,
                     int64_t* write_indices, CtlRoutes& R) {
  if (int32_t e = route_geometry(c->slots, reads, R.root, R.read_sub, R.read_k)) return e;
  if (int32_t e = route_geometry(c->slots, writes, R.root, R.write_sub, R.write_k)) return e;
  if (batch == 0) return 0;
  if (!read_weights || !read_indices || !write_weights || !write_indices) {
    return fail(COWSDM_EARG, "controller prepare: null route pointer");
  }
  R.read_weights = read_weights;
  R.read_indices = read_indices;
  R.write_weights = write_weights;
  R.write_indices = write_indices;
  return 0;
}

int32_t finish_params(const cowsdm_controller_t* c, const float* normalized,
                      const float* reading, int64_t batch, float* out, const float* residual,
                      float* out_sum, CtlParams& P) {
  if (residual && !out_sum) return fail(COWSDM_EARG, "controller finish: null residual sum");
  P.residual = residual;
  P.out_sum = out_sum;
  if (int32_t e = check_controller(c, batch, P)) return e;
  if (batch == 0) return 0;
  if (!normalized || !reading || !out || !c->gate_weight_t || !c->gate_bias ||
      !c->out_weight_t || !c->out_bias || !c->read_norm_weight || !c->read_norm_bias) {
    return fail(COWSDM_EARG, "controller finish: null pointer argument");
  }
  P.normalized = normalized;
  P.reading = reading;
  P.out = out;
  if (batch > (int64_t{1} << 31) - 1) {
    return fail(COWSDM_ELIMIT, "controller: batch too large");
  }
  return 0;
}

}  // namespace

extern "C" int32_t cowsdm_controller_prepare(const cowsdm_controller_t* c, const float* tokens,
                                             int64_t batch, float* normalized, float* read_keys,
                                             float* write_keys, float* values, float* input_gate,
                                             float* forget_log_gate, void* stream) {
  CtlParams P{};
  if (int32_t e = prepare_params(c, tokens, batch, normalized, read_keys, write_keys, values,
                                 input_gate, forget_log_gate, P)) {
    return e;
  }
  if (batch == 0) return 0;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  return by_tokens(P, 1, [&] { return launch_prepare<1, 1>(P, s); },
                   [&] { return launch_prepare<1, 2>(P, s); },
                   [&] { return launch_prepare<2, 2>(P, s); });
}

extern "C" int32_t cowsdm_product_key_routes(const float* projected, int64_t rows,
                                             int64_t slots, int64_t selected,
                                             float* weights, int64_t* indices, void* stream);

extern "C" int32_t cowsdm_controller_prepare_routes(
    const cowsdm_controller_t* c, const float* tokens, int64_t batch, float* normalized,
    float* read_keys, float* write_keys, float* values, float* input_gate,
    float* forget_log_gate, int64_t reads, int64_t writes, float* read_weights,
    int64_t* read_indices, float* write_weights, int64_t* write_indices, void* stream) {
  CtlParams P{};
  if (int32_t e = prepare_params(c, tokens, batch, normalized, read_keys, write_keys, values,
                                 input_gate, forget_log_gate, P)) {
    return e;
  }
  CtlRoutes R{};
  if (int32_t e = route_params(c, batch, reads, writes, read_weights, read_indices,
                               write_weights, write_indices, R)) {
    return e;
  }
  if (batch == 0) return 0;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (!prepare_selects(P, R.root, batch * c->heads)) {
    if (int32_t e = cowsdm_controller_prepare(c, tokens, batch, normalized, read_keys,
                                              write_keys, values, input_gate, forget_log_gate,
                                              stream)) {
      return e;
    }
    const int64_t rows = batch * c->heads;
    if (int32_t e = cowsdm_product_key_routes(read_keys, rows, c->slots, reads, read_weights,
                                              read_indices, stream)) {
      return e;
    }
    return cowsdm_product_key_routes(write_keys, rows, c->slots, writes, write_weights,
                                     write_indices, stream);
  }
  const int mr = route_m(R, R.read_sub, R.read_k), mw = route_m(R, R.write_sub, R.write_k);
  if (mr == 0 && mw == 0) return launch_prepare_routes<0, 0>(P, R, s);
  if (mr == 0) return mw == 1 ? launch_prepare_routes<0, 1>(P, R, s) : launch_prepare_routes<0, 2>(P, R, s);
  if (mw == 0) return mr == 1 ? launch_prepare_routes<1, 0>(P, R, s) : launch_prepare_routes<2, 0>(P, R, s);
  if (mr == 1) return mw == 1 ? launch_prepare_routes<1, 1>(P, R, s) : launch_prepare_routes<1, 2>(P, R, s);
  return mw == 1 ? launch_prepare_routes<2, 1>(P, R, s) : launch_prepare_routes<2, 2>(P, R, s);
}

extern "C" int32_t cowsdm_controller_finish_residual(const cowsdm_controller_t* c,
                                                     const float* normalized,
                                                     const float* reading, int64_t batch,
                                                     float* out, const float* residual,
                                                     float* out_sum, void* stream) {
  CtlParams P{};
  if (int32_t e = finish_params(c, normalized, reading, batch, out, residual, out_sum, P)) {
    return e;
  }
  if (batch == 0) return 0;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  return by_tokens(P, 2, [&] { return launch_finish<1, 1>(P, s); },
                   [&] { return launch_finish<1, 2>(P, s); },
                   [&] { return launch_finish<2, 2>(P, s); });
}

extern "C" int32_t cowsdm_controller_finish(const cowsdm_controller_t* c,
                                            const float* normalized, const float* reading,
                                            int64_t batch, float* out, void* stream) {
  return cowsdm_controller_finish_residual(c, normalized, reading, batch, out, nullptr, nullptr,
                                           stream);
}

extern "C" int32_t cowsdm_controller_finish_prepare_routes(
    const cowsdm_controller_t* c, const float* normalized, const float* reading, int64_t batch,
    float* out, const float* residual, float* out_sum, const cowsdm_controller_t* next,
    float* next_normalized, float* read_keys, float* write_keys, float* values,
    float* input_gate, float* forget_log_gate, int64_t reads, int64_t writes,
    float* read_weights, int64_t* read_indices, float* write_weights, int64_t* write_indices,
    void* stream) {
  if (!residual || !out_sum) {
    return fail(COWSDM_EARG, "controller finish and prepare: null residual or sum");
  }
  CtlParams F{};
  if (int32_t e = finish_params(c, normalized, reading, batch, out, residual, out_sum, F)) {
    return e;
  }
  CtlParams P{};
  if (int32_t e = prepare_params(next, out_sum, batch, next_normalized, read_keys, write_keys,
                                 values, input_gate, forget_log_gate, P)) {
    return e;
  }
  if (next->width != c->width) {
    return fail(COWSDM_EARG, "controller finish and prepare: the layers' widths differ");
  }
  CtlRoutes R{};
  if (int32_t e = route_params(next, batch, reads, writes, read_weights, read_indices,
                               write_weights, write_indices, R)) {
    return e;
  }
  if (batch == 0) return 0;
  if (!prepare_selects(P, R.root, batch * next->heads)) {
    if (int32_t e = cowsdm_controller_finish_residual(c, normalized, reading, batch, out,
                                                      residual, out_sum, stream)) {
      return e;
    }
    return cowsdm_controller_prepare_routes(next, out_sum, batch, next_normalized, read_keys,
                                            write_keys, values, input_gate, forget_log_gate,
                                            reads, writes, read_weights, read_indices,
                                            write_weights, write_indices, stream);
  }
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int mr = route_m(R, R.read_sub, R.read_k), mw = route_m(R, R.write_sub, R.write_k);
  if (mr == 0 && mw == 0) return launch_finish_prepare_routes<0, 0>(F, P, R, s);
  if (mr == 0) return mw == 1 ? launch_finish_prepare_routes<0, 1>(F, P, R, s) : launch_finish_prepare_routes<0, 2>(F, P, R, s);
  if (mw == 0) return mr == 1 ? launch_finish_prepare_routes<1, 0>(F, P, R, s) : launch_finish_prepare_routes<2, 0>(F, P, R, s);
  if (mr == 1) return mw == 1 ? launch_finish_prepare_routes<1, 1>(F, P, R, s) : launch_finish_prepare_routes<1, 2>(F, P, R, s);
  return mw == 1 ? launch_finish_prepare_routes<2, 1>(F, P, R, s) : launch_finish_prepare_routes<2, 2>(F, P, R, s);
}
