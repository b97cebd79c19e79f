// Sector precompute on the device: sample -> sector assignment, stable radix
// sort by sector, per-sector offsets, sector centres, sorted trajectory and
// density, the gridding work list (sector chunks) and the adjoint's tile lists.
//
// Reference semantics: CUDA/inc/precomp_utils.hpp:34-153,
// CUDA/src/gpuNUFFT_operator_factory.cpp:128-270, CUDA/src/gpu/precomp_kernels.cu:8-177.

#include <algorithm>
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include "gnufft_internal.hpp"

namespace gnufft {

__global__ void __launch_bounds__(256) assign_sectors_kernel(Geom g, const float* __restrict__ traj,
                                                             uint32_t M, uint32_t* __restrict__ keys,
                                                             uint32_t* __restrict__ vals) {
  uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= M) return;
  int sx = sector_of(traj[t], g.G[0], g.sw);
  int sy = sector_of(traj[t + M], g.G[1], g.sw);
  int sz = 0;
  if (g.dim == 3) sz = sector_of(traj[t + 2 * (size_t)M], g.G[2], g.sw);
  keys[t] = (uint32_t)(sx + g.S[0] * (sy + g.S[1] * sz));
  vals[t] = t;
}

hipError_t launch_assign_sectors(const Geom& g, const float* traj, uint32_t M, uint32_t* keys,
                                 uint32_t* vals, hipStream_t s) {
  if (M == 0) return hipSuccess;
  unsigned blocks = (M + 255) / 256;
  hipLaunchKernelGGL(assign_sectors_kernel, dim3(blocks), dim3(256), 0, s, g, traj, M, keys, vals);
  return hipGetLastError();
}

// Radix passes at every size: below a million pairs the library's default is a merge
// sort of some 24 launches, twice a trajectory on the long path, where 16 bits of
// keys need two radix passes.
using SortConfig = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                              rocprim::default_config, 0>;

// Stable LSD radix sort of (sector, original index) pairs: within a sector
// samples keep their original order, the canonical order of the reference's
// std::sort (equal per-sector index sets, CUDA/src/gpuNUFFT_operator_factory.cpp:56-72).
hipError_t sort_pairs(void* temp, size_t* temp_bytes, const uint32_t* keys_in,
                      uint32_t* keys_out, const uint32_t* vals_in, uint32_t* vals_out,
                      uint32_t M, int key_bits, hipStream_t s) {
  return rocprim::radix_sort_pairs<SortConfig>(temp, *temp_bytes, keys_in, keys_out, vals_in, vals_out,
                                   (size_t)M, 0, key_bits, s);
}

// sdc[s] = first sorted position with key >= s (lower bound), s = 0..S.
// Equals the reference's [0, n0, n0+n1, ...] (gpuNUFFT_operator_factory.cpp:183-205).
__global__ void __launch_bounds__(256) sector_count_kernel(const uint32_t* __restrict__ keys,
                                                           uint32_t M, uint32_t S,
                                                           uint32_t* __restrict__ sdc) {
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s > S) return;
  uint32_t lo = 0, hi = M;
  while (lo < hi) {
    uint32_t mid = lo + (hi - lo) / 2;
    if (keys[mid] < s)
      lo = mid + 1;
    else
      hi = mid;
  }
  sdc[s] = lo;
}

hipError_t launch_sector_data_count(const uint32_t* sorted_keys, uint32_t M, uint32_t S,
                                    uint32_t* sdc, hipStream_t s) {
  unsigned blocks = (S + 1 + 255) / 256;
  hipLaunchKernelGGL(sector_count_kernel, dim3(blocks), dim3(256), 0, s, sorted_keys, M, S, sdc);
  return hipGetLastError();
}

// Centres c_a = s_a*sw + floor(sw/2), interleaved per sector
// (gpuNUFFT_operator_factory.cpp:207-270).
__global__ void __launch_bounds__(256) sector_centers_kernel(Geom g, uint32_t* __restrict__ out) {
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t S = (uint32_t)g.S[0] * g.S[1] * g.S[2];
  if (s >= S) return;
  uint32_t x = s % g.S[0];
  uint32_t y = (s / g.S[0]) % g.S[1];
  uint32_t z = s / ((uint32_t)g.S[0] * g.S[1]);
  uint32_t half = (uint32_t)(g.sw / 2);
  if (g.dim == 2) {
    out[2 * s] = x * g.sw + half;
    out[2 * s + 1] = y * g.sw + half;
  } else {
    out[3 * s] = x * g.sw + half;
    out[3 * s + 1] = y * g.sw + half;
    out[3 * s + 2] = z * g.sw + half;
  }
}

hipError_t launch_sector_centers(const Geom& g, uint32_t* centers, hipStream_t s) {
  uint32_t S = (uint32_t)g.S[0] * g.S[1] * g.S[2];
  hipLaunchKernelGGL(sector_centers_kernel, dim3((S + 255) / 256), dim3(256), 0, s, g, centers);
  return hipGetLastError();
}

// Sorted trajectory / density gather (precomp_kernels.cu:85-113).
__global__ void __launch_bounds__(256) gather_traj_kernel(const float* __restrict__ traj,
                                                          const float* __restrict__ dens,
                                                          const uint32_t* __restrict__ idx,
                                                          uint32_t M, int dim,
                                                          float* __restrict__ traj_sorted,
                                                          float* __restrict__ dens_sorted) {
  uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= M) return;
  uint32_t j = idx[t];
  for (int a = 0; a < dim; a++) traj_sorted[t + (size_t)a * M] = traj[j + (size_t)a * M];
  if (dens) dens_sorted[t] = dens[j];
}

hipError_t launch_gather_traj(const float* traj, const float* dens, const uint32_t* idx,
                              uint32_t M, int dim, float* traj_sorted, float* dens_sorted,
                              hipStream_t s) {
  if (M == 0) return hipSuccess;
  hipLaunchKernelGGL(gather_traj_kernel, dim3((M + 255) / 256), dim3(256), 0, s, traj, dens, idx,
                     M, dim, traj_sorted, dens_sorted);
  return hipGetLastError();
}

// Number of work chunks per sector, then an exclusive scan: chunk_off has
// S+1 entries, chunk_off[S] = total chunks.
__global__ void __launch_bounds__(256) chunk_count_kernel(const uint32_t* __restrict__ sdc,
                                                          uint32_t S, uint32_t chunk,
                                                          uint32_t* __restrict__ cnt) {
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s > S) return;
  if (s == S) {
    cnt[s] = 0;
    return;
  }
  uint32_t n = sdc[s + 1] - sdc[s];
  cnt[s] = (n + chunk - 1) / chunk;
}

hipError_t count_chunks(const uint32_t* sdc, uint32_t S, uint32_t chunk, uint32_t* cnt,
                        uint32_t* chunk_off, void* temp, size_t* temp_bytes, hipStream_t s) {
  if (temp == nullptr) {
    return rocprim::exclusive_scan(nullptr, *temp_bytes, cnt, chunk_off, 0u, (size_t)S + 1,
                                   rocprim::plus<uint32_t>(), s);
  }
  hipLaunchKernelGGL(chunk_count_kernel, dim3((S + 1 + 255) / 256), dim3(256), 0, s, sdc, S,
                     chunk, cnt);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return rocprim::exclusive_scan(temp, *temp_bytes, cnt, chunk_off, 0u, (size_t)S + 1,
                                 rocprim::plus<uint32_t>(), s);
}

__global__ void __launch_bounds__(256) fill_chunks_kernel(const uint32_t* __restrict__ sdc,
                                                          const uint32_t* __restrict__ chunk_off,
                                                          uint32_t S, uint32_t chunk,
                                                          Chunk* __restrict__ chunks) {
  uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= S) return;
  uint32_t b = sdc[s], e = sdc[s + 1];
  uint32_t o = chunk_off[s];
  for (uint32_t p = b; p < e; p += chunk) {
    Chunk c;
    c.sector = s;
    c.begin = p;
    c.end = (e - p > chunk) ? p + chunk : e;
    c.pad = 0;
    chunks[o++] = c;
  }
}

hipError_t launch_fill_chunks(const uint32_t* sdc, const uint32_t* chunk_off, uint32_t S,
                              uint32_t chunk, Chunk* chunks, hipStream_t s) {
  hipLaunchKernelGGL(fill_chunks_kernel, dim3((S + 255) / 256), dim3(256), 0, s, sdc, chunk_off,
                     S, chunk, chunks);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Tap table and the tile lists of the adjoint gridding. A sample goes into the
// list of every tile that one of its taps of nonzero weight falls in: its
// pairs (tile, sample) are written at the samples' exclusive counts and sorted
// by tile (stable: each list is in the caller's order, so that a round of the
// spread takes whole runs of a trajectory through its tile).
// ---------------------------------------------------------------------------
struct TileRange {  // tiles first, first + 1, .. (count of them, modulo n) along an axis
  int first, count, n;
};

// Tiles of the taps of nonzero weight among NX - 1 from grid index q.
template <int NX>
__device__ inline TileRange tile_range(int q, const float* w, int G, int width) {
  int a = NX - 1, b = -1;
#pragma unroll
  for (int t = 0; t < NX - 1; t++)
    if (w[t] != 0.0f) {
      a = min(a, t);
      b = t;
    }
  TileRange r;
  r.n = (G + width - 1) / width;
  if (b < 0) {
    r.first = r.count = 0;
    return r;
  }
  const int lo = wrap(q + a, G), len = b - a;
  r.first = lo / width;
  r.count = lo + len < G ? (lo + len) / width - r.first + 1
                         : r.n - r.first + wrap(lo + len, G) / width + 1;
  r.count = min(r.count, r.n);
  return r;
}

// First grid index and weights of the sample at p along axis d.
template <int NX>
__device__ inline int axis_taps(const Geom& g, const float* lut, int d, float p, float* w) {
  const int G = g.G[d];
  const int center = sector_of(p, G, g.sw) * g.sw + g.sw / 2;
  int lo, hi;
  tap_range(map_kspace_to_grid(p, G, center, g.off), g.Pmax, g.kradius, &lo, &hi);
#pragma unroll
  for (int t = 0; t < NX; t++) {
    float wt = 0.0f;
    if (lo + t <= hi && axis_weight(g, lut, d, lo + t, center, p, &wt)) w[t] = wt;
    else w[t] = 0.0f;
  }
  // taps that coincide on a grid shorter than the kernel
  if (g.kw > G)
    for (int t = NX - 1; t >= 0; t--)
      for (int u = 0; u < t && t >= G; u++)
        if (u == t % G) {
          w[u] += w[t];
          w[t] = 0.0f;
        }
  return wrap(center - g.off + lo, G);
}

template <int NX>
__device__ inline void store_taps(float4* out, int q, const float* w) {
  out[0] = make_float4(__int_as_float(q), w[0], w[1], w[2]);
  if constexpr (NX == 8) out[1] = make_float4(w[3], w[4], w[5], w[6]);
}

// Tiles reached by sample s of the tap table, per axis.
template <int DIM, int NX>
__device__ inline void sample_tiles(const Geom& g, const float4* taps, uint32_t s, TileRange* r) {
  r[2] = TileRange{0, 1, 1};
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    const float4* in = taps + ((size_t)d * g.M + s) * (NX / 4);
    const float4 a = in[0];
    float w[NX] = {a.y, a.z, a.w};
    if constexpr (NX == 8) {
      const float4 b = in[1];
      w[3] = b.x, w[4] = b.y, w[5] = b.z, w[6] = b.w;
    }
    r[d] = tile_range<NX>(__float_as_int(a.x), w, g.G[d], tile_width(DIM, d));
  }
}

// f(tile) for every tile of the ranges
template <int DIM, typename F>
__device__ inline void each_tile(const TileList& l, const TileRange* r, F f) {
  for (int z = 0; z < r[2].count; z++)
    for (int y = 0; y < r[1].count; y++)
      for (int x = 0; x < r[0].count; x++)
        f(tile_number<DIM>(l, (uint32_t)wrap(r[0].first + x, r[0].n), (uint32_t)wrap(r[1].first + y, r[1].n),
                           (uint32_t)wrap(r[2].first + z, r[2].n)));
}

template <int DIM, int NX>
__global__ void __launch_bounds__(256) taps_kernel(Geom g, const float* __restrict__ crds,
                                                   const float* __restrict__ dens,
                                                   const uint32_t* __restrict__ idx,
                                                   const float* __restrict__ lut, float4* __restrict__ taps,
                                                   uint32_t* __restrict__ pos, float* __restrict__ dens_sqrt,
                                                   uint32_t* __restrict__ counts) {
  const uint32_t s = blockIdx.x * 256 + threadIdx.x;
  if (s >= (uint32_t)g.M) return;
  const uint32_t j = idx[s];
  pos[j] = s;
  if (dens) dens_sqrt[j] = sqrtf(dens[s]);
  uint32_t n = 1;
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    float w[NX];
    const int q = axis_taps<NX>(g, lut, d, crds[(size_t)d * g.M + s], w);
    store_taps<NX>(taps + ((size_t)d * g.M + j) * (NX / 4), q, w);
    n *= (uint32_t)tile_range<NX>(q, w, g.G[d], tile_width(DIM, d)).count;
  }
  counts[j] = n;
}

hipError_t launch_taps(const Geom& g, const float* crds, const float* dens, const uint32_t* idx, const float* lut,
                       float4* taps, uint32_t* pos, float* dens_sqrt, uint32_t* counts, hipStream_t s) {
  if (g.M == 0) return hipSuccess;
  const bool wide = tap_vec(g.kw) == 2;
  auto kernel = g.dim == 3 ? (wide ? taps_kernel<3, 8> : taps_kernel<3, 4>)
                           : (wide ? taps_kernel<2, 8> : taps_kernel<2, 4>);
  hipLaunchKernelGGL(kernel, dim3((g.M + 255) / 256), dim3(256), 0, s, g, crds, dens, idx, lut, taps, pos,
                     dens_sqrt, counts);
  return hipGetLastError();
}

struct CountAt {  // counts[i], 0 past the last
  const uint32_t* counts;
  size_t n;
  __host__ __device__ uint64_t operator()(size_t i) const { return i < n ? counts[i] : 0; }
};

hipError_t scan_counts(void* temp, size_t* temp_bytes, const uint32_t* counts, uint64_t* offs, size_t n,
                       hipStream_t s) {
  auto in = rocprim::make_transform_iterator(rocprim::make_counting_iterator<size_t>(0), CountAt{counts, n});
  return rocprim::exclusive_scan(temp, *temp_bytes, in, offs, (uint64_t)0, n + 1, rocprim::plus<uint64_t>(), s);
}

template <int DIM, int NX>
__global__ void __launch_bounds__(256) emit_pairs_kernel(Geom g, TileList l, const float4* __restrict__ taps,
                                                         const uint64_t* __restrict__ offs,
                                                         uint32_t* __restrict__ keys,
                                                         uint32_t* __restrict__ vals) {
  const uint32_t s = blockIdx.x * 256 + threadIdx.x;
  if (s >= (uint32_t)g.M) return;
  TileRange r[3];
  sample_tiles<DIM, NX>(g, taps, s, r);
  uint64_t at = offs[s];
  each_tile<DIM>(l, r, [&](uint32_t tile) {
    keys[at] = tile;
    vals[at] = s;
    at++;
  });
}

hipError_t launch_emit_pairs(const Geom& g, const TileList& l, const float4* taps, const uint64_t* offs,
                             uint32_t* keys, uint32_t* vals, hipStream_t s) {
  if (g.M == 0) return hipSuccess;
  const dim3 grid((g.M + 255) / 256);
  const bool wide = tap_vec(g.kw) == 2;
  auto kernel = g.dim == 3 ? (wide ? emit_pairs_kernel<3, 8> : emit_pairs_kernel<3, 4>)
                           : (wide ? emit_pairs_kernel<2, 8> : emit_pairs_kernel<2, 4>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, g, l, taps, offs, keys, vals);
  return hipGetLastError();
}

hipError_t sort_tile_pairs(void* temp, size_t* temp_bytes, const uint32_t* keys_in, uint32_t* keys_out,
                           const uint32_t* vals_in, uint32_t* vals_out, size_t n, int key_bits, hipStream_t s) {
  return rocprim::radix_sort_pairs<SortConfig>(temp, *temp_bytes, keys_in, keys_out, vals_in, vals_out, n, 0, key_bits, s);
}

// Offset of tile t: lower bound of its key.
__global__ void __launch_bounds__(256) tile_offsets_kernel(const uint32_t* __restrict__ keys, size_t n,
                                                           uint32_t tiles, uint64_t* __restrict__ tile_off) {
  const uint32_t t = blockIdx.x * 256 + threadIdx.x;
  if (t > tiles) return;
  size_t lo = 0, hi = n;
  while (lo < hi) {
    const size_t mid = lo + (hi - lo) / 2;
    if (keys[mid] < t)
      lo = mid + 1;
    else
      hi = mid;
  }
  tile_off[t] = lo;
}

hipError_t launch_tile_offsets(const uint32_t* keys, size_t n, uint32_t tiles, uint64_t* tile_off, hipStream_t s) {
  hipLaunchKernelGGL(tile_offsets_kernel, dim3((tiles + 256) / 256), dim3(256), 0, s, keys, n, tiles, tile_off);
  return hipGetLastError();
}

struct TileCount {  // chunks, scratch slots and reduction tasks of tile t
  const uint64_t* tile_off;
  uint32_t tiles, chunk;
  __host__ __device__ TileTotals operator()(uint32_t t) const {
    if (t >= tiles) return TileTotals{0, 0, 0};
    const uint64_t n = tile_off[t + 1] - tile_off[t];
    const uint32_t m = n > chunk ? (uint32_t)((n + chunk - 1) / chunk) : 1u;
    return TileTotals{m, m > 1 ? m : 0u, m > 1 ? 1u : 0u};
  }
};

struct AddTotals {
  __host__ __device__ TileTotals operator()(const TileTotals& a, const TileTotals& b) const {
    return TileTotals{a.chunks + b.chunks, a.slots + b.slots, a.tasks + b.tasks};
  }
};

hipError_t scan_tile_chunks(void* temp, size_t* temp_bytes, const uint64_t* tile_off, uint32_t tiles,
                            uint32_t chunk, TileTotals* tot, hipStream_t s) {
  auto in = rocprim::make_transform_iterator(rocprim::make_counting_iterator<uint32_t>(0),
                                             TileCount{tile_off, tiles, chunk});
  return rocprim::exclusive_scan(temp, *temp_bytes, in, tot, TileTotals{0, 0, 0}, (size_t)tiles + 1,
                                 AddTotals(), s);
}

__global__ void __launch_bounds__(256) tile_chunks_kernel(TileCount count, const TileTotals* __restrict__ tot,
                                                          TileChunk* __restrict__ chunks,
                                                          TileTask* __restrict__ tasks) {
  const uint32_t t = blockIdx.x * 256 + threadIdx.x;
  if (t >= count.tiles) return;
  const TileTotals at = tot[t], mine = count(t);
  const uint64_t begin = count.tile_off[t], n = count.tile_off[t + 1] - begin;
  for (uint32_t i = 0; i < mine.chunks; i++) {
    const uint64_t b = (uint64_t)i * count.chunk;
    chunks[at.chunks + i] = TileChunk{begin + b, (uint32_t)(n - b < count.chunk ? n - b : count.chunk), t,
                                      mine.slots ? at.slots + i : kNoSlot, 0};
  }
  if (mine.tasks) tasks[at.tasks] = TileTask{t, at.slots, mine.slots, 0};
}

hipError_t fill_tile_chunks(const uint64_t* tile_off, uint32_t tiles, uint32_t chunk, const TileTotals* tot,
                            TileChunk* chunks, TileTask* tasks, hipStream_t s) {
  hipLaunchKernelGGL(tile_chunks_kernel, dim3((tiles + 255) / 256), dim3(256), 0, s,
                     TileCount{tile_off, tiles, chunk}, tot, chunks, tasks);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The same tables for short trajectories, where launches are what the build
// costs: a stable counting sort by sector and by tile at once, instead of two
// sorts and three scans of the library (a 2-D frame of 21 k samples: 31
// launches, 9 of them per sort). A workgroup takes kBlock samples of the
// caller's order and marks each in a bit mask per key (sectors, then tiles);
// counts and ranks are popcounts of the masks.
// ---------------------------------------------------------------------------
constexpr int kBlock = 128;

// Keys of sample j marked in mask[key][kBlock / 32].
template <int DIM, int NX>
__device__ inline void mark_keys(const Geom& g, const TileList& l, uint32_t sector, uint32_t S, const TileRange* r,
                                 uint32_t* mask) {
  const uint32_t word = threadIdx.x / 32, bit = 1u << (threadIdx.x % 32);
  atomicOr(&mask[sector * (kBlock / 32) + word], bit);
  each_tile<DIM>(l, r, [&](uint32_t tile) { atomicOr(&mask[(S + tile) * (kBlock / 32) + word], bit); });
}

__device__ inline uint32_t mask_count(const uint4& m) { return __popc(m.x) + __popc(m.y) + __popc(m.z) + __popc(m.w); }

// samples of the block before this thread's among those of mask m
__device__ inline uint32_t mask_rank(const uint32_t* m) {
  const uint32_t word = threadIdx.x / 32;
  uint32_t n = __popc(m[word] & ((1u << (threadIdx.x % 32)) - 1u));
  for (uint32_t w = 0; w < word; w++) n += __popc(m[w]);
  return n;
}

template <int DIM, int NX>
__global__ void __launch_bounds__(kBlock) short_count_kernel(Geom g, TileList l, ShortTables t) {
  extern __shared__ uint4 masks[];
  uint32_t* mask = reinterpret_cast<uint32_t*>(masks);
  const uint32_t keys = t.S + t.n_tiles, j = blockIdx.x * kBlock + threadIdx.x, M = (uint32_t)g.M;
  for (uint32_t k = threadIdx.x; k < keys; k += kBlock) masks[k] = make_uint4(0, 0, 0, 0);
  __syncthreads();
  if (j < M) {
    TileRange r[3];
    r[2] = TileRange{0, 1, 1};
    int sec[3] = {0, 0, 0};
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      const float p = t.traj[(size_t)d * M + j];
      float w[NX];
      const int q = axis_taps<NX>(g, t.lut, d, p, w);
      store_taps<NX>(t.taps + ((size_t)d * M + j) * (NX / 4), q, w);
      r[d] = tile_range<NX>(q, w, g.G[d], tile_width(DIM, d));
      sec[d] = sector_of(p, g.G[d], g.sw);
    }
    if (t.dens) t.dens_sqrt[j] = sqrtf(t.dens[j]);
    const uint32_t sector = (uint32_t)(sec[0] + g.S[0] * (sec[1] + g.S[1] * sec[2]));
    t.assigned[j] = sector;
    mark_keys<DIM, NX>(g, l, sector, t.S, r, mask);
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < keys; k += kBlock)
    t.counts[(size_t)k * gridDim.x + blockIdx.x] = mask_count(masks[k]);
}

template <int DIM, int NX>
__global__ void __launch_bounds__(kBlock) short_place_kernel(Geom g, TileList l, ShortTables t) {
  extern __shared__ uint4 masks[];
  uint32_t* mask = reinterpret_cast<uint32_t*>(masks);
  const uint32_t keys = t.S + t.n_tiles, j = blockIdx.x * kBlock + threadIdx.x, M = (uint32_t)g.M;
  for (uint32_t k = threadIdx.x; k < keys; k += kBlock) masks[k] = make_uint4(0, 0, 0, 0);
  uint32_t sector = 0;
  TileRange r[3];
  if (j < M) {
    sector = t.assigned[j];
    sample_tiles<DIM, NX>(g, t.taps, j, r);
  }
  __syncthreads();
  if (j < M) mark_keys<DIM, NX>(g, l, sector, t.S, r, mask);
  __syncthreads();
  if (j >= M) return;
  auto place = [&](uint32_t key) {
    return t.offs[(size_t)key * gridDim.x + blockIdx.x] + mask_rank(mask + key * (kBlock / 32));
  };
  const uint32_t at = place(sector);
  t.idx[at] = j;
  t.pos[j] = at;
  for (int d = 0; d < DIM; d++) t.traj_sorted[(size_t)d * M + at] = t.traj[(size_t)d * M + j];
  if (t.dens) t.dens_sorted[at] = t.dens[j];
  each_tile<DIM>(l, r, [&](uint32_t tile) { t.entries[place(t.S + tile) - M] = j; });
}

// Exclusive sums of three values over the 1024 threads of a workgroup; the
// totals in `all`.
__device__ inline uint3 block_sums(uint3 v, uint3* all) {
  __shared__ uint3 wsum[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint3 inc = v;
#pragma unroll
  for (int o = 1; o < 64; o *= 2) {
    const uint32_t x = __shfl_up(inc.x, o), y = __shfl_up(inc.y, o), z = __shfl_up(inc.z, o);
    if (lane >= o) inc.x += x, inc.y += y, inc.z += z;
  }
  __syncthreads();
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  uint3 before = make_uint3(0, 0, 0), sum = before;
  for (int w = 0; w < 16; w++) {
    if (w == wave) before = sum;
    sum.x += wsum[w].x, sum.y += wsum[w].y, sum.z += wsum[w].z;
  }
  *all = sum;
  return make_uint3(before.x + inc.x - v.x, before.y + inc.y - v.y, before.z + inc.z - v.z);
}

// Offsets, centres and work lists, by one workgroup.
template <int DIM>
__global__ void __launch_bounds__(1024) short_lists_kernel(Geom g, ShortTables t, uint32_t blocks) {
  const uint32_t tid = threadIdx.x, S = t.S, M = (uint32_t)g.M;
  auto off = [&](uint32_t key) { return t.offs[(size_t)key * blocks]; };
  uint3 all;
  // sectors: offsets, chunks and runs of chunks; a contiguous share per thread
  const uint32_t per_s = (S + 1023) / 1024, s0 = min(tid * per_s, S), s1 = min(s0 + per_s, S);
  uint3 n = make_uint3(0, 0, 0);
  for (uint32_t s = s0; s < s1; s++) {
    const uint32_t m = (off(s + 1) - off(s) + t.chunk - 1) / t.chunk;
    n.x += m;
    n.y += (m + kInterpRun - 1) / kInterpRun;
    t.sdc[s] = t.host[s] = off(s);
    const uint32_t half = (uint32_t)(g.sw / 2), x = s % g.S[0], yz = s / g.S[0];
    t.centers[DIM * s] = x * g.sw + half;
    t.centers[DIM * s + 1] = (DIM == 2 ? yz : yz % g.S[1]) * g.sw + half;
    if (DIM == 3) t.centers[DIM * s + 2] = (yz / g.S[1]) * g.sw + half;
  }
  uint3 at = block_sums(n, &all);
  if (tid == 0) t.sdc[S] = t.host[S] = M;
  for (uint32_t s = s0; s < s1; s++) {
    const uint32_t b = off(s), e = off(s + 1);
    for (uint32_t p = b; p < e; p += t.chunk) t.chunks[at.x++] = Chunk{s, p, min(p + t.chunk, e), 0};
    if (DIM == 3)
      for (uint32_t p = b; p < e; p += t.chunk * kInterpRun) t.runs[at.y++] = Chunk{s, p, min(p + t.chunk * kInterpRun, e), 0};
  }
  uint32_t* totals = t.host + S + 1;
  if (tid == 0) totals[0] = all.x, totals[1] = all.y;
  // tiles: entries per chunk (tile_chunk, then doubled until the partial tiles
  // fit), chunks, slots, tasks
  const uint32_t per_t = (t.n_tiles + 1023) / 1024, t0 = min(tid * per_t, t.n_tiles),
                 t1 = min(t0 + per_t, t.n_tiles);
  const uint32_t first = off(S), end = t.offs[(size_t)(S + t.n_tiles) * blocks];
  uint32_t chunk = tile_chunk(DIM, end - first);
  for (;; chunk *= 2) {
    n = make_uint3(0, 0, 0);
    for (uint32_t i = t0; i < t1; i++) {
      const uint32_t e = off(S + i + 1) - off(S + i), m = e > chunk ? (e + chunk - 1) / chunk : 1u;
      n.x += m;
      if (m > 1) n.y += m, n.z++;
    }
    at = block_sums(n, &all);
    if (all.y <= t.max_slots || chunk >= (1u << 30)) break;
  }
  for (uint32_t i = t0; i < t1; i++) {
    const uint32_t b = off(S + i) - first, e = off(S + i + 1) - first, m = e - b > chunk ? (e - b + chunk - 1) / chunk : 1u;
    for (uint32_t c = 0; c < m; c++)
      t.tile_chunks[at.x + c] =
          TileChunk{(uint64_t)b + (uint64_t)c * chunk, min(e - b - c * chunk, chunk), i, m > 1 ? at.y + c : kNoSlot, 0};
    if (m > 1) t.tile_tasks[at.z] = TileTask{i, at.y, m, 0};
    at.x += m;
    if (m > 1) at.y += m, at.z++;
  }
  if (tid == 0) totals[2] = all.x, totals[3] = all.y, totals[4] = all.z;
}

struct BlockCountAt {  // counts[i], 0 past the last
  const uint32_t* counts;
  size_t n;
  __host__ __device__ uint32_t operator()(size_t i) const { return i < n ? counts[i] : 0u; }
};

// Up to 6 M counts (48 MB of workspace), the keys' masks within the LDS: the counts are
// what it costs, 150 us at 3.8 M of them, 193 at 5.0 M, 214 at 6.0 M and 0.54 ms at 7.9 M,
// where the library's sorts take 0.34 ms (256^2 osf 2, 0.2 M samples).
bool short_tables_ok(uint32_t M, uint32_t S, uint32_t n_tiles) {
  const size_t keys = (size_t)S + n_tiles, blocks = ((size_t)M + kBlock - 1) / kBlock;
  return M > 0 && M <= (1u << 18) && keys <= 8192 && keys * blocks <= (6u << 20);
}

size_t short_tables_entries(const Geom& g, uint32_t M) {
  // tiles met by kw taps of an axis, with a partial last tile between the ends
  size_t most = M;
  for (int a = 0; a < g.dim; a++) {
    const int w = tile_width(g.dim, a);
    most *= (size_t)std::min((g.G[a] + w - 1) / w, 4 * tap_vec(g.kw) / w + 3);
  }
  return most;
}

size_t short_tables_words(uint32_t M, uint32_t S, uint32_t n_tiles) {
  return (size_t)(S + n_tiles) * ((M + kBlock - 1) / kBlock) + 1;
}

hipError_t launch_short_tables(const Geom& g, const TileList& l, const ShortTables& t, void* temp,
                               size_t* temp_bytes, hipStream_t s) {
  const uint32_t keys = t.S + t.n_tiles, blocks = ((uint32_t)g.M + kBlock - 1) / kBlock;
  const size_t n = (size_t)keys * blocks;
  auto in = rocprim::make_transform_iterator(rocprim::make_counting_iterator<size_t>(0), BlockCountAt{t.counts, n});
  if (!temp)
    return rocprim::exclusive_scan(nullptr, *temp_bytes, in, t.offs, 0u, n + 1, rocprim::plus<uint32_t>(), s);
  const bool wide = tap_vec(g.kw) == 2;
  const size_t lds = (size_t)keys * sizeof(uint4);
  auto count = g.dim == 3 ? (wide ? short_count_kernel<3, 8> : short_count_kernel<3, 4>)
                          : (wide ? short_count_kernel<2, 8> : short_count_kernel<2, 4>);
  auto place = g.dim == 3 ? (wide ? short_place_kernel<3, 8> : short_place_kernel<3, 4>)
                          : (wide ? short_place_kernel<2, 8> : short_place_kernel<2, 4>);
  hipError_t e = hipSuccess;
  if (lds > 64 * 1024) {
    e = hipFuncSetAttribute((const void*)count, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e == hipSuccess)
      e = hipFuncSetAttribute((const void*)place, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(count, dim3(blocks), dim3(kBlock), lds, s, g, l, t);
  e = hipGetLastError();
  if (e == hipSuccess)
    e = rocprim::exclusive_scan(temp, *temp_bytes, in, t.offs, 0u, n + 1, rocprim::plus<uint32_t>(), s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(place, dim3(blocks), dim3(kBlock), lds, s, g, l, t);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (g.dim == 3)
    hipLaunchKernelGGL(short_lists_kernel<3>, dim3(1), dim3(1024), 0, s, g, t, blocks);
  else
    hipLaunchKernelGGL(short_lists_kernel<2>, dim3(1), dim3(1024), 0, s, g, t, blocks);
  return hipGetLastError();
}

}  // namespace gnufft
