// cowsdm_product_key_routes: one lane or one wave per route row (routes.h
// holds the selections, which give the same bits).

#include "routes.h"

namespace cowsdm_impl {

template <int J, int M>
__global__ __launch_bounds__(kWave * kRouteWaves) void product_key_routes_kernel(
    const float* __restrict__ projected, int64_t rows, int root, int sub, int final_k,
    float* __restrict__ weights, int64_t* __restrict__ indices) {
  __shared__ float stage_val[kRouteWaves][kRouteMaxSelected];
  __shared__ int stage_pos[kRouteWaves][kRouteMaxSelected];
  __shared__ float pool_val[kRouteWaves][kWave];
  __shared__ int pool_pos[kRouteWaves][kWave];
  const int wave = static_cast<int>(threadIdx.x) / kWave;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kRouteWaves + wave;
  if (row >= rows) return;
  product_key_route_row<J, M>(projected, row, root, sub, final_k, weights, indices,
                              stage_val[wave], stage_pos[wave], pool_val[wave], pool_pos[wave]);
}

// One wave per workgroup, so that few rows still spread over the compute units.
template <int NR, int KP, bool FULL>
__global__ __launch_bounds__(kWave) void product_key_routes_lane_kernel(
    const float* __restrict__ projected, int64_t rows, int root, int sub, int final_k,
    float* __restrict__ weights, int64_t* __restrict__ indices) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kWave + threadIdx.x;
  const bool on = row < rows;
  product_key_route_lane<NR, KP, FULL>(on, projected + (on ? row : 0) * 2 * root, root, sub,
                                       final_k, weights + row * final_k,
                                       indices + row * final_k);
}

// One lane per row, or false where one wave per row is the better one.  Above
// sqrt(N) = 32 a row's scores do not fit in a lane's registers.  Below a few
// thousand rows neither fills the device and the shorter program wins: the
// sorted wave's where it applies (N = 256 K = 16: 3.4 us to 2,048 rows and
// 4.4 at 4,000, the lane's 5.7 to 6.3 at 8,192; K = 4: 3.4 to 4.5 against
// 3.6); for more routes the lane's if sqrt(N), the shortlist and K fill its
// networks (N = 1,024 K = 32, 64 rows: 11.9 us against 12.1) and the ranking
// wave's otherwise (N = 1,024 K = 24, 64 rows: 11.1 us against 15.2; 4,096
// rows: 20.2 against 15.9).
template <int NR, int KP>
bool launch_routes_lane_k(const float* projected, int64_t rows, int root, int sub, int final_k,
                          float* weights, int64_t* indices, hipStream_t stream) {
  const bool full = root == NR && sub == (KP < NR ? KP : NR) && final_k == KP &&
                    reinterpret_cast<uintptr_t>(projected) % 16 == 0;
  const bool sorted = route_row_sorted(root, final_k);
  if (sorted ? rows < kRouteLaneRows * (final_k > 8 ? 2 : 1) : !full && rows < kRouteLaneRows) {
    return false;
  }
  auto* const kernel = full ? &product_key_routes_lane_kernel<NR, KP, true>
                            : &product_key_routes_lane_kernel<NR, KP, false>;
  const int64_t blocks = (rows + kWave - 1) / kWave;
  hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kWave), 0, stream,
                     projected, rows, root, sub, final_k, weights, indices);
  return true;
}

template <int NR>
bool launch_routes_lane(const float* projected, int64_t rows, int root, int sub, int final_k,
                        float* weights, int64_t* indices, hipStream_t stream) {
  auto* const launch = final_k <= 4    ? &launch_routes_lane_k<NR, 4>
                       : final_k <= 8  ? &launch_routes_lane_k<NR, 8>
                       : final_k <= 16 ? &launch_routes_lane_k<NR, 16>
                                       : &launch_routes_lane_k<NR, 32>;
  return launch(projected, rows, root, sub, final_k, weights, indices, stream);
}

__global__ __launch_bounds__(kWave * kRouteWaves) void product_key_routes_sorted_kernel(
    const float* __restrict__ projected, int64_t rows, int root, int sub, int final_k,
    float* __restrict__ weights, int64_t* __restrict__ indices) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kRouteWaves +
                      static_cast<int>(threadIdx.x) / kWave;
  if (row >= rows) return;
  product_key_route_row_sorted(projected, row, root, sub, final_k, weights, indices);
}

template <int J, int M>
void launch_routes(const float* projected, int64_t rows, int root, int sub, int final_k,
                   float* weights, int64_t* indices, hipStream_t stream) {
  const int64_t blocks = (rows + kRouteWaves - 1) / kRouteWaves;
  hipLaunchKernelGGL((product_key_routes_kernel<J, M>), dim3(static_cast<uint32_t>(blocks)),
                     dim3(kWave * kRouteWaves), 0, stream, projected, rows, root, sub,
                     final_k, weights, indices);
}

template <int J>
void launch_routes_pairs(const float* projected, int64_t rows, int root, int sub,
                         int final_k, float* weights, int64_t* indices,
                         hipStream_t stream) {
  if (route_pair_m(sub, final_k) == 1)
    launch_routes<J, 1>(projected, rows, root, sub, final_k, weights, indices, stream);
  else
    launch_routes<J, 2>(projected, rows, root, sub, final_k, weights, indices, stream);
}

}  // namespace cowsdm_impl

using namespace cowsdm_impl;

extern "C" int32_t cowsdm_product_key_routes(const float* projected, int64_t rows,
                                             int64_t slots, int64_t selected,
                                             float* weights, int64_t* indices,
                                             void* stream) {
  if (rows < 0) return fail(-1, "product_key_routes: rows must be >= 0 (got %lld)",
                            static_cast<long long>(rows));
  int r = 0, k = 0, f = 0;
  if (int32_t e = route_geometry(slots, selected, r, k, f)) return e;
  if (rows > (int64_t{1} << 31) * kRouteWaves - kRouteWaves)
    return fail(-2, "product_key_routes: too many rows (%lld)", static_cast<long long>(rows));
  if (rows == 0) return 0;
  if (!projected || !weights || !indices)
    return fail(-1, "product_key_routes: null pointer argument");
  auto s = static_cast<hipStream_t>(stream);
  const bool lane =
      r <= 16 ? launch_routes_lane<16>(projected, rows, r, k, f, weights, indices, s)
      : r <= kRouteLaneRoot
          ? launch_routes_lane<kRouteLaneRoot>(projected, rows, r, k, f, weights, indices, s)
          : false;
  if (lane) return launch_status("product_key_routes");
  if (route_row_sorted(r, f)) {
    hipLaunchKernelGGL(product_key_routes_sorted_kernel,
                       dim3(static_cast<uint32_t>((rows + kRouteWaves - 1) / kRouteWaves)),
                       dim3(kWave * kRouteWaves), 0, s, projected, rows, r, k, f, weights,
                       indices);
  } else if (r <= kWave)
    launch_routes_pairs<1>(projected, rows, r, k, f, weights, indices, s);
  else if (r <= 4 * kWave)
    launch_routes_pairs<4>(projected, rows, r, k, f, weights, indices, s);
  else
    launch_routes_pairs<16>(projected, rows, r, k, f, weights, indices, s);
  return launch_status("product_key_routes");
}
