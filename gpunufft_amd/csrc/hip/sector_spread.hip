// Adjoint gridding with order-independent sums, for CG-SENSE on grids with an
// odd length. Reference: CUDA/src/gpu/atomic/atomic_gpuNUFFT_kernels.cu:302-617,
// texture_gpuNUFFT_kernels.cu:22-376.
//
// The two directions of the operator shift the grid by floor(G / 2) and
// ceil(G / 2); where a length is odd they are not adjoint to each other, CG works
// on a matrix that is not Hermitian, and rounding grows by orders of magnitude
// from iteration to iteration: two versions of the adjoint that differ in the
// order of their sums alone (2e-7 of the result) end up 1e-5 to 2e-2 apart after
// ten iterations (1e-6 on even grids). What such a solve returns is settled by how
// the adjoint rounds, so it keeps one definition of it, these sums.
//
// One workgroup per (run of at most 1024 samples of a sector, coil block) adds
// its samples to the padded sector in LDS in fixed point: 64-bit words, re and im
// as two packed 32-bit halves of a step of L1 / 2^30 (L1: the sum of the samples'
// magnitudes, so a half cannot overflow). Integer sums do not depend on their
// order. The sub-grids go to memory, and one thread per grid point and coil sums
// those that cover it, in a fixed order (periodic wrap and INVERSE fftshift folded
// in).
//
// Bound: the LDS atomics, and the sub-grids' way to memory and back (each grid point
// 1.6 times in 2-D and 2 times in 3-D at sector width 8 and kernel width 3). Per
// iteration at 525^2, kernel width 3, 12 coils, 122 k samples: sums 81 us, fold 24 us.
// A thread of the fold takes four coils (with one, ten iterations took 3042 instead
// of 2929 us).

#include <algorithm>

#include "gnufft_internal.hpp"

namespace gnufft {

namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr double kRoundMagic = 6755399441055744.0;  // 1.5 * 2^52: x + magic rounds x to an integer
constexpr double kFixedOne = 1073741824.0;          // 2^30

__host__ __device__ inline int padded_points(const Geom& g) { return g.dim == 3 ? g.P * g.P * g.P : g.P * g.P; }

// Kernel width 3: a step is L1 summed by `cb` coils to a quad of lanes (float sums:
// their order sets the last bits of the step), and values enter as doubles.
__host__ __device__ inline bool quad_sums(const Geom& g) { return g.kw == 3 && g.P >= 4; }

// Adds wt * v (in steps) to one word.
__device__ inline void fx_add(unsigned long long* w, double wt, double vx, double vy) {
  const uint32_t re = (uint32_t)__double_as_longlong(fma(wt, vx, kRoundMagic));
  const uint32_t im = (uint32_t)__double_as_longlong(fma(wt, vy, kRoundMagic));
  const uint32_t hi = im + (uint32_t)((int32_t)re >> 31);  // borrow of a negative re
  atomicAdd(w, ((unsigned long long)hi << 32) | re);
}

// NX - 1: weights per axis of the tap table.
template <int DIM, int NX>
__global__ void __launch_bounds__(kThreads) sector_sums_kernel(Geom g, SectorSpreadArgs a, int cb) {
  constexpr int NV = NX / 4;
  extern __shared__ unsigned long long sub[];  // [padded point][cb]
  __shared__ float l1_part[kWaves][4];
  __shared__ double scale_s[4], inv_s[4];
  const int P = g.P, PD = padded_points(g);
  const Chunk ch = a.chunks[blockIdx.x];
  const int n = (int)(ch.end - ch.begin);
  const int coil0 = (int)blockIdx.y * cb;
  const int wb = min(cb, a.n_coils - coil0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool quads = quad_sums(g);

  for (int i = tid; i < PD * cb; i += kThreads) sub[i] = 0ull;

  // the coils' steps
  if (quads) {
    const int c = (lane & 3) % cb;
    float l1 = 0.0f;
    for (int r = 0; r < 2; r++)
      for (int ps = 0; ps < cb; ps++) {
        const int j = r * kThreads + (tid & ~3) + ps * (4 / cb) + (tid & 3) / cb;
        if (j >= n || c >= wb) continue;
        const uint32_t src = a.idx[ch.begin + j];
        const float sq = a.dens ? a.dens[src] : 1.0f;
        float2 v = a.data[(size_t)(coil0 + c) * a.coil_stride + src];
        v.x *= sq;
        v.y *= sq;
        l1 += fmaxf(fabsf(v.x), fabsf(v.y));
      }
    for (int o = cb; o < 64; o <<= 1) l1 += __shfl_xor(l1, o);
    if (lane < cb) l1_part[wave][lane] = l1;
  } else {
    for (int c = 0; c < cb; c++) {
      float l1 = 0.0f;
      for (int i = tid; i < n; i += kThreads)
        if (c < wb) {
          const uint32_t src = a.idx[ch.begin + i];
          const float sq = a.dens ? a.dens[src] : 1.0f;
          const float2 v = a.data[(size_t)(coil0 + c) * a.coil_stride + src];
          l1 += fmaxf(fabsf(v.x), fabsf(v.y)) * sq;
        }
      for (int o = 32; o >= 1; o >>= 1) l1 += __shfl_xor(l1, o);
      if (lane == 0) l1_part[wave][c] = l1;
    }
  }
  __syncthreads();
  if (tid < cb) {
    double t = 0.0;
    for (int w = 0; w < kWaves; w++) t += (double)l1_part[w][tid];
    const double sc = t > 0.0 ? kFixedOne / t : 0.0;
    scale_s[tid] = sc;
    inv_s[tid] = sc > 0.0 ? 1.0 / sc : 0.0;
  }
  __syncthreads();

  // first grid index of the padded sector
  int o3[3];
  {
    const uint32_t x = ch.sector % (uint32_t)g.S[0], yz = ch.sector / (uint32_t)g.S[0];
    const int first = g.sw / 2 - g.off;
    o3[0] = wrap((int)x * g.sw + first, g.G[0]);
    o3[1] = wrap((int)(yz % (uint32_t)g.S[1]) * g.sw + first, g.G[1]);
    o3[2] = DIM == 3 ? wrap((int)(yz / (uint32_t)g.S[1]) * g.sw + first, g.G[2]) : 0;
  }

  // lanes = (sample slot, coil); slot k takes samples [k seg, (k + 1) seg), so
  // that the samples of one instruction are apart on their trajectory
  const int slots = 64 / cb, slot = lane / cb, c = lane % cb;
  const int seg = (n + slots - 1) / slots;
  const double scale = scale_s[c];
  for (int j = wave; j < seg; j += kWaves) {
    const int s = slot * seg + j;
    if (s >= n || c >= wb) continue;
    const uint32_t src = a.idx[ch.begin + s];
    const float sq = a.dens ? a.dens[src] : 1.0f;
    float2 v = a.data[(size_t)(coil0 + c) * a.coil_stride + src];
    double vx, vy;
    if (quads) {
      v.x *= sq;
      v.y *= sq;
      vx = (double)v.x * scale;
      vy = (double)v.y * scale;
    } else {
      const double k = (double)sq * scale;
      vx = (double)(float)(v.x * k);
      vy = (double)(float)(v.y * k);
    }
    int first[3];
    float w[3][NX - 1];
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      const float4* at = a.taps + ((size_t)d * g.M + src) * NV;
      const float4 t = at[0];
      const int q = __float_as_int(t.x) - o3[d];
      first[d] = min(q < 0 ? q + g.G[d] : q, P - 1);
      w[d][0] = t.y, w[d][1] = t.z, w[d][2] = t.w;
      if constexpr (NX == 8) {
        const float4 u = at[1];
        w[d][3] = u.x, w[d][4] = u.y, w[d][5] = u.z, w[d][6] = u.w;
      }
    }
    // (a tap past the sector's last point has weight zero)
#pragma unroll
    for (int tz = 0; tz < (DIM == 3 ? NX - 1 : 1); tz++) {
      const int iz = DIM == 3 ? min(first[DIM - 1] + tz, P - 1) : 0;
#pragma unroll
      for (int ty = 0; ty < NX - 1; ty++) {
        const int iy = min(first[1] + ty, P - 1);
        const float wzy = DIM == 3 ? w[DIM - 1][tz] * w[1][ty] : w[1][ty];
        if (wzy == 0.0f) continue;
        unsigned long long* row = sub + (iz * P + iy) * P * cb + c;
        const double rx = (double)wzy * vx, ry = (double)wzy * vy;
#pragma unroll
        for (int tx = 0; tx < NX - 1; tx++) {
          if (w[0][tx] == 0.0f) continue;
          unsigned long long* to = row + min(first[0] + tx, P - 1) * cb;
          if (quads)
            fx_add(to, (double)w[0][tx], rx, ry);
          else
            fx_add(to, (double)(wzy * w[0][tx]), vx, vy);
        }
      }
    }
  }
  __syncthreads();

  for (int cc = 0; cc < wb; cc++) {
    float2* dst = a.sub + ((size_t)blockIdx.x * a.n_coils + coil0 + cc) * PD;
    const double inv = inv_s[cc];
    for (int pt = tid; pt < PD; pt += kThreads) {
      const unsigned long long u = sub[pt * cb + cc];
      const int32_t re = (int32_t)(uint32_t)u;
      const int32_t im = (int32_t)(uint32_t)(u >> 32) - (re >> 31);
      dst[pt] = make_float2((float)(re * inv), (float)(im * inv));
    }
  }
}

// A grid point of kFoldCoils coils: the sum over the sectors covering it, z, y, x
// outermost to innermost, of the sum over the sector's chunks.
constexpr int kFoldCoils = 4;
template <int DIM>
__global__ void __launch_bounds__(256) sector_fold_kernel(Geom g, SectorSpreadArgs a) {
  const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
  if (e >= g.Ng) return;
  const int coil0 = (int)blockIdx.y * kFoldCoils;
  const int P = g.P, PD = padded_points(g);
  const int x = (int)(e % g.G[0]);
  const long long yz = e / g.G[0];
  const int y = (int)(yz % g.G[1]), z = (int)(yz / g.G[1]);
  const size_t stride = (size_t)a.n_coils * PD;
  float2 sum[kFoldCoils];
  size_t at[kFoldCoils];  // (coils past the last one repeat it)
#pragma unroll
  for (int q = 0; q < kFoldCoils; q++) {
    sum[q] = make_float2(0.0f, 0.0f);
    at[q] = (size_t)min(coil0 + q, a.n_coils - 1) * PD;
  }
  const uint32_t z0 = DIM == 3 ? a.cover_off[2][z] : 0, z1 = DIM == 3 ? a.cover_off[2][z + 1] : 1;
  for (uint32_t iz = z0; iz < z1; iz++) {
    const uint2 cz = DIM == 3 ? a.cover[2][iz] : make_uint2(0, 0);
    for (uint32_t iy = a.cover_off[1][y]; iy < a.cover_off[1][y + 1]; iy++) {
      const uint2 cy = a.cover[1][iy];
      for (uint32_t ix = a.cover_off[0][x]; ix < a.cover_off[0][x + 1]; ix++) {
        const uint2 cx = a.cover[0][ix];
        const uint32_t s = cx.x + (uint32_t)g.S[0] * (cy.x + (uint32_t)g.S[1] * cz.x);
        const uint32_t k0 = a.first[s], k1 = a.first[s + 1];
        if (k0 == k1) continue;
        const float2* src = a.sub + k0 * stride + cx.y + (size_t)P * (cy.y + (size_t)P * cz.y);
        float2 v[kFoldCoils];
#pragma unroll
        for (int q = 0; q < kFoldCoils; q++) v[q] = src[at[q]];
#pragma unroll 4
        for (uint32_t k = 1; k < k1 - k0; k++) {
#pragma unroll
          for (int q = 0; q < kFoldCoils; q++) {
            const float2 u = src[k * stride + at[q]];
            v[q].x += u.x;
            v[q].y += u.y;
          }
        }
#pragma unroll
        for (int q = 0; q < kFoldCoils; q++) {
          sum[q].x += v[q].x;
          sum[q].y += v[q].y;
        }
      }
    }
  }
  const size_t to = tile_store_index<DIM>(g, x, y, z, a.fold_shift);
#pragma unroll
  for (int q = 0; q < kFoldCoils; q++)
    if (coil0 + q < a.n_coils) a.grid[(size_t)(coil0 + q) * g.Ng + to] = sum[q];
}

// Coils per workgroup. Kernel width 3: at most a quad, for `per_cu` workgroups of
// the padded sector and its tables per CU, then fewer (this choice sets the
// order of the L1 sums, so it is part of what a solve returns).
int sums_coils(const Geom& g, int n_coils, int per_cu) {
  const bool quads = quad_sums(g);
  for (int per = !quads ? 3 : per_cu > 0 ? per_cu : default_per_cu(3); per >= 1; per--)
    for (int cb = 4; cb >= 1; cb /= 2) {
      if (cb > 1 && cb / 2 >= n_coils) continue;
      const size_t bytes = quads ? lane_bytes(g, cb) : (size_t)padded_points(g) * cb * 8;
      if (bytes <= lds_limit() / per - 1024) return cb;
    }
  return 0;
}

template <int DIM, int NX>
hipError_t sums_launch(const Geom& g, const SectorSpreadArgs& a, int cb, hipStream_t s) {
  const size_t lds = (size_t)padded_points(g) * cb * 8;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(sector_sums_kernel<DIM, NX>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((sector_sums_kernel<DIM, NX>), dim3(a.n_chunks, (a.n_coils + cb - 1) / cb), dim3(kThreads), lds,
                     s, g, a, cb);
  return hipGetLastError();
}

}  // namespace

size_t sector_sub_elems(const Geom& g) { return (size_t)padded_points(g); }

void sector_cover(const Geom& g, int axis, std::vector<uint32_t>* off, std::vector<uint2>* entries) {
  const int G = g.G[axis];
  std::vector<std::vector<uint2>> at((size_t)G);
  for (int n = 0; n < g.S[axis]; n++)
    for (int i = 0; i < g.P; i++)
      at[(size_t)wrap(n * g.sw + g.sw / 2 - g.off + i, G)].push_back(make_uint2((uint32_t)n, (uint32_t)i));
  off->assign(1, 0u);
  entries->clear();
  for (const auto& l : at) {
    entries->insert(entries->end(), l.begin(), l.end());
    off->push_back((uint32_t)entries->size());
  }
}

hipError_t launch_sector_spread(const Geom& g, const SectorSpreadArgs& a, int per_cu, hipStream_t s) {
  if (a.n_coils == 0) return hipSuccess;
  if (a.n_chunks > 0) {
    const int cb = sums_coils(g, a.n_coils, per_cu);
    if (cb == 0) return hipErrorInvalidValue;
    const bool wide = tap_vec(g.kw) == 2;
    hipError_t e;
    if (g.dim == 3)
      e = wide ? sums_launch<3, 8>(g, a, cb, s) : sums_launch<3, 4>(g, a, cb, s);
    else
      e = wide ? sums_launch<2, 8>(g, a, cb, s) : sums_launch<2, 4>(g, a, cb, s);
    if (e != hipSuccess) return e;
  }
  const dim3 grid((unsigned)((g.Ng + 255) / 256), (a.n_coils + kFoldCoils - 1) / kFoldCoils);
  if (g.dim == 3)
    hipLaunchKernelGGL(sector_fold_kernel<3>, grid, dim3(256), 0, s, g, a);
  else
    hipLaunchKernelGGL(sector_fold_kernel<2>, grid, dim3(256), 0, s, g, a);
  return hipGetLastError();
}

}  // namespace gnufft
