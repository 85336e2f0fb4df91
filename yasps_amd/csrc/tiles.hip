// Build and value gather of the tiled symmetric operator (tiles.hpp) from the mirrored full
// block-CSR of an operator without repeated (row, column) entries.
//
// Tiles are runs of kTileRows block rows in the order of a Hilbert curve through the given
// points (10 bits per axis of the points' cube; Skilling, "Programming the Hilbert curve",
// AIP Conf. Proc. 707, 2004): on the n = 48 tet cube 70% of the off-diagonal blocks stay
// inside a tile (Morton order 68%, the mesh's own layer order 38%), so 0.67 of the mirrored
// copy's entries are stored. Any order gives the same operator; a poor one only keeps more
// blocks in both tiles.
#include "tiles.hpp"
#include "values.hpp"

#include <hipcub/hipcub.hpp>

namespace ysp {
namespace {

constexpr unsigned kB = 256;

// Bounding box of the points, one workgroup: box[0..2] the low corner, box[3] the scale
// that maps the longest side to [0, 1024).
__global__ void __launch_bounds__(1024)
    tile_box_kernel(const double* __restrict__ p, uint32_t n, double* __restrict__ box) {
  double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
  for (uint32_t i = threadIdx.x; i < n; i += 1024)
    for (int c = 0; c < 3; ++c) {
      const double v = p[3 * static_cast<size_t>(i) + c];
      lo[c] = fmin(lo[c], v);
      hi[c] = fmax(hi[c], v);
    }
  __shared__ double s[6][16];
  for (int c = 0; c < 3; ++c)
    for (int o = 32; o > 0; o >>= 1) {
      lo[c] = fmin(lo[c], __shfl_xor(lo[c], o, 64));
      hi[c] = fmax(hi[c], __shfl_xor(hi[c], o, 64));
    }
  if (threadIdx.x % 64 == 0)
    for (int c = 0; c < 3; ++c) {
      s[c][threadIdx.x / 64] = lo[c];
      s[3 + c][threadIdx.x / 64] = hi[c];
    }
  __syncthreads();
  if (threadIdx.x == 0) {
    double side = 0.0;
    for (int c = 0; c < 3; ++c) {
      for (int w = 1; w < 16; ++w) {
        s[c][0] = fmin(s[c][0], s[c][w]);
        s[3 + c][0] = fmax(s[3 + c][0], s[3 + c][w]);
      }
      box[c] = s[c][0];
      side = fmax(side, s[3 + c][0] - s[c][0]);
    }
    box[3] = side > 0.0 ? 1023.0 / side : 0.0;
  }
}

__device__ __forceinline__ uint32_t spread3(uint32_t x) {
  x = (x | (x << 16)) & 0x030000ffu;
  x = (x | (x << 8)) & 0x0300f00fu;
  x = (x | (x << 4)) & 0x030c30c3u;
  return (x | (x << 2)) & 0x09249249u;
}

// Hilbert index of a point with 10 bits per axis (points outside the box or not finite
// are clamped: the order is only a matter of speed).
__global__ void __launch_bounds__(kB)
    tile_key_kernel(const double* __restrict__ p, uint32_t n, const double* __restrict__ box,
                    uint32_t* __restrict__ key, uint32_t* __restrict__ row) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  row[i] = i;
  uint32_t X[3];
  for (int c = 0; c < 3; ++c) {
    const double v = (p[3 * static_cast<size_t>(i) + c] - box[c]) * box[3];
    X[c] = v >= 0.0 ? (v <= 1023.0 ? static_cast<uint32_t>(v) : 1023u) : 0u;
  }
  constexpr uint32_t M = 512;
  for (uint32_t q = M; q > 1; q >>= 1) {
    const uint32_t m = q - 1;
    for (int c = 0; c < 3; ++c) {
      if (X[c] & q) X[0] ^= m;
      else {
        const uint32_t t = (X[0] ^ X[c]) & m;
        X[0] ^= t;
        X[c] ^= t;
      }
    }
  }
  X[1] ^= X[0];
  X[2] ^= X[1];
  uint32_t t = 0;
  for (uint32_t q = M; q > 1; q >>= 1)
    if (X[2] & q) t ^= q - 1;
  for (int c = 0; c < 3; ++c) X[c] ^= t;
  key[i] = (spread3(X[0]) << 2) | (spread3(X[1]) << 1) | spread3(X[2]);
}

__global__ void __launch_bounds__(kB) tile_iota_kernel(uint32_t n, uint32_t* __restrict__ row) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) row[i] = i;
}

__global__ void __launch_bounds__(kB)
    tile_of_kernel(const uint32_t* __restrict__ order, uint32_t n, uint32_t* __restrict__ tile) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) tile[order[i]] = i / kTileRows;
}

// Whether row r keeps its entry at column c: its own diagonal, the upper one of the two
// mirrored entries inside a tile, every entry into another tile.
__device__ __forceinline__ bool tile_keeps(const uint32_t* tile, uint32_t r, uint32_t c) {
  return c >= r || tile[c] != tile[r];
}

// One workgroup per tile: entry counts of its rows, positions by falling count (slices of
// rows of like lengths pad least), the slices' widths.
__global__ void __launch_bounds__(kTileRows)
    tile_sort_kernel(const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ col,
                     const uint32_t* __restrict__ tile, uint32_t n,
                     const uint32_t* __restrict__ order, uint32_t* __restrict__ rows,
                     uint32_t* __restrict__ lens, uint32_t* __restrict__ local,
                     uint32_t* __restrict__ widths, int* __restrict__ bad) {
  __shared__ uint32_t cnt[kTileRows];
  const uint32_t base = blockIdx.x * kTileRows, i = threadIdx.x;
  const bool live = base + i < n;
  uint32_t r = 0, len = 0;
  if (live) {
    r = order[base + i];
    for (uint32_t k = row_ptr[r]; k < row_ptr[r + 1]; ++k) {
      const uint32_t c = col[k];
      if (c >= n) {
        atomicOr(bad, 1);
        continue;
      }
      len += tile_keeps(tile, r, c);
    }
    if (len > kTileMaxRow) atomicOr(bad, 1);
  }
  cnt[i] = live ? len + 1 : 0;                 // positions past the last row sort last
  __syncthreads();
  uint32_t rank = 0;
  for (uint32_t j = 0; j < kTileRows; ++j)
    rank += cnt[j] > cnt[i] || (cnt[j] == cnt[i] && j < i);
  if (live) {
    rows[base + rank] = r;
    lens[base + rank] = len;
    local[r] = rank;
  }
  if (rank % 64 == 0) widths[base / 64 + rank / 64] = live ? 64 * len : 0;   // the slice's longest
}

__global__ void __launch_bounds__(kB)
    tile_fill_kernel(const uint32_t* __restrict__ row_ptr, const uint32_t* __restrict__ col,
                     const uint32_t* __restrict__ src, const uint32_t* __restrict__ tile,
                     const uint32_t* __restrict__ local, uint32_t n,
                     const uint32_t* __restrict__ rows, const uint32_t* __restrict__ slice_start,
                     uint32_t* __restrict__ entry, uint32_t* __restrict__ source) {
  const uint32_t pos = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t slice = pos / 64, lane = pos % 64;
  uint32_t at = slice_start[slice] + lane;
  const uint32_t end = slice_start[slice + 1];
  if (pos < n) {
    const uint32_t r = rows[pos];
    for (int cut = 0; cut < 2; ++cut)          // the tile's own entries first
      for (uint32_t k = row_ptr[r]; k < row_ptr[r + 1]; ++k) {
        const uint32_t c = col[k];
        if (!tile_keeps(tile, r, c) || (tile[c] != tile[r]) != (cut != 0)) continue;
        entry[at] = cut ? (kTileCut | (tile[c] * kTileRows + local[c])) : local[c];
        source[at] = src[k];
        at += 64;
      }
  }
  for (; at < end; at += 64) {                 // the slice's padding, never read by a product
    entry[at] = 0;
    source[at] = kTileNoSource;
  }
}

template <typename VT>
__global__ void __launch_bounds__(kB)
    tile_values_kernel(const double* __restrict__ sv, const uint32_t* __restrict__ source,
                       uint32_t entries, VT* __restrict__ out) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= entries) return;
  const uint32_t s = source[k];
  if (s == kTileNoSource) return;
  const double* B = sv + 9 * static_cast<size_t>(s & ~(kTrans | kDyn));
  double v[9];
#pragma unroll
  for (int j = 0; j < 9; ++j) v[j] = B[j];
  const bool tr = (s & kTrans) != 0;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j)
      out[tile_value(k) + 64 * (3 * i + j)] = static_cast<VT>(tr ? v[3 * j + i] : v[3 * i + j]);
}

}  // namespace
}  // namespace ysp

using namespace ysp;

extern "C" int ysp_bsr3_tiles_layout(const uint32_t* row_ptr, const uint32_t* col, uint32_t nnz,
                                     uint32_t n, const double* points, uint32_t* rows,
                                     uint32_t* lens, uint32_t* slice_start, uint32_t* work,
                                     uint32_t* entries, void* stream) {
  if (!entries || n % 3 || (n && (!row_ptr || !col || !rows || !lens || !slice_start || !work))) {
    ysp_set_error(__FILE__, __LINE__, "ysp_bsr3_tiles_layout: bad arguments");
    return YSP_ERR_ARG;
  }
  *entries = 0;
  const uint32_t nv = n / 3;
  if (nv == 0 || nnz == 0) return YSP_OK;
  hipStream_t s = as_stream(stream);
  const uint32_t tiles = (nv + kTileRows - 1) / kTileRows, slices = tiles * (kTileRows / 64);
  uint32_t* tile = work;
  uint32_t* local = work + nv;
  uint32_t* key = static_cast<uint32_t*>(scratch(131, sizeof(uint32_t) * nv));
  uint32_t* row = static_cast<uint32_t*>(scratch(121, sizeof(uint32_t) * nv));
  uint32_t* key2 = static_cast<uint32_t*>(scratch(122, sizeof(uint32_t) * nv));
  uint32_t* row2 = static_cast<uint32_t*>(scratch(123, sizeof(uint32_t) * nv));
  uint32_t* widths = static_cast<uint32_t*>(scratch(124, sizeof(uint32_t) * (slices + 1)));
  double* box = static_cast<double*>(scratch(125, 5 * sizeof(double)));
  if (!key || !row || !key2 || !row2 || !widths || !box) return YSP_ERR_HIP;
  int* bad = reinterpret_cast<int*>(box + 4);
  YSP_CHECK(hipMemsetAsync(bad, 0, sizeof(int), s));
  YSP_CHECK(hipMemsetAsync(widths, 0, sizeof(uint32_t) * (slices + 1), s));
  const dim3 g(grid_for(nv, kB)), b(kB);
  const uint32_t* order = row;
  if (points) {
    hipLaunchKernelGGL(tile_box_kernel, dim3(1), dim3(1024), 0, s, points, nv, box);
    hipLaunchKernelGGL(tile_key_kernel, g, b, 0, s, points, nv, box, key, row);
    hipcub::DoubleBuffer<uint32_t> kb(key, key2), rb(row, row2);
    size_t temp = 0;
    YSP_CHECK(hipcub::DeviceRadixSort::SortPairs(nullptr, temp, kb, rb, nv, 0, 30, s));
    void* tmp = scratch(126, temp);
    if (!tmp) return YSP_ERR_HIP;
    YSP_CHECK(hipcub::DeviceRadixSort::SortPairs(tmp, temp, kb, rb, nv, 0, 30, s));
    order = rb.Current();
  } else {
    hipLaunchKernelGGL(tile_iota_kernel, g, b, 0, s, nv, row);
  }
  hipLaunchKernelGGL(tile_of_kernel, g, b, 0, s, order, nv, tile);
  hipLaunchKernelGGL(tile_sort_kernel, dim3(tiles), dim3(kTileRows), 0, s, row_ptr, col, tile, nv,
                     order, rows, lens, local, widths, bad);
  size_t temp = 0;
  YSP_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, temp, widths, slice_start, slices + 1, s));
  void* tmp = scratch(127, temp);
  if (!tmp) return YSP_ERR_HIP;
  YSP_CHECK(hipcub::DeviceScan::ExclusiveSum(tmp, temp, widths, slice_start, slices + 1, s));
  YSP_CHECK_LAUNCH();
  uint32_t total = 0;
  int flag = 0;
  YSP_CHECK(hipMemcpyAsync(&total, slice_start + slices, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
  YSP_CHECK(hipMemcpyAsync(&flag, bad, sizeof(int), hipMemcpyDeviceToHost, s));
  YSP_CHECK(hipStreamSynchronize(s));
  *entries = flag ? 0 : total;                 // 0: rows too long for tiles
  return YSP_OK;
}

extern "C" int ysp_bsr3_tiles_entries(const uint32_t* row_ptr, const uint32_t* col,
                                      const uint32_t* src, uint32_t n, const uint32_t* rows,
                                      const uint32_t* slice_start, const uint32_t* work,
                                      uint32_t* entry, uint32_t* source, void* stream) {
  if (n % 3 || (n && (!row_ptr || !col || !src || !rows || !slice_start || !work || !entry || !source))) {
    ysp_set_error(__FILE__, __LINE__, "ysp_bsr3_tiles_entries: bad arguments");
    return YSP_ERR_ARG;
  }
  const uint32_t nv = n / 3;
  if (nv == 0) return YSP_OK;
  const uint32_t positions = (nv + kTileRows - 1) / kTileRows * kTileRows;
  hipLaunchKernelGGL(tile_fill_kernel, dim3(grid_for(positions, kB)), dim3(kB), 0, as_stream(stream),
                     row_ptr, col, src, work, work + nv, nv, rows, slice_start, entry, source);
  YSP_CHECK_LAUNCH();
  return YSP_OK;
}

extern "C" int ysp_bsr3_tiles_values(const double* static_values, const uint32_t* source,
                                     uint32_t entries, double* out64, float* out32, void* stream) {
  if (entries == 0) return YSP_OK;
  if (!static_values || !source) {
    ysp_set_error(__FILE__, __LINE__, "ysp_bsr3_tiles_values: bad arguments");
    return YSP_ERR_ARG;
  }
  const dim3 g(grid_for(entries, kB)), b(kB);
  if (out64)
    hipLaunchKernelGGL(tile_values_kernel<double>, g, b, 0, as_stream(stream), static_values, source,
                       entries, out64);
  if (out32)
    hipLaunchKernelGGL(tile_values_kernel<float>, g, b, 0, as_stream(stream), static_values, source,
                       entries, out32);
  YSP_CHECK_LAUNCH();
  return YSP_OK;
}
