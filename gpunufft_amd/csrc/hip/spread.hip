// Adjoint gridding (Kaiser-Bessel spread) on the matrix cores, for CDNA4
// (gfx950). Reference: CUDA/src/gpu/atomic/atomic_gpuNUFFT_kernels.cu:302-617,
// texture_gpuNUFFT_kernels.cu:22-376.
//
// The grid is cut into tiles (16 x 8 x 4 points in 3-D, 16^2 in 2-D). A plan
// holds, per tile, the list of every sample with a tap inside it (a sample
// near a border is in the lists of all tiles it reaches) and, per sample, its
// taps' weights; a workgroup forms its tile's final values by itself and
// writes each grid point once: no atomics, no padded sub-grids, no fold over
// neighbours.
//
// A wave owns a sub-tile of 16 rows (3-D: 4 z x 4 y, 2-D: 16 y) by 4 points in
// x. Its sum over samples is a matrix product with the samples as the
// contraction index k,
//   D[row][(x, coil, re/im)] += (wz wy)[row][k] * (wx v)[k][(x, coil, re/im)],
// run as v_mfma_f32_16x16x4_f32, four samples per instruction: 8 / NC points
// in x times NC coils fill the 16 columns. Products and sums are 32-bit
// floats throughout. With one coil a sub-tile is 8 points wide: a matrix
// instruction covers all of it, where the columns of a second coil would idle.
// Against the two-coil kernel on one coil, over 48 volumes (64^3..152^3, osf
// 1.25..2, kernel width 3 and 5, an eighth of the fully sampled spokes to all):
// 152^3 osf 1.5 width 5 fully sampled 793 -> 545 us (sector sub-grids: 681),
// 128^3 osf 1.25 width 5 685 -> 495 (458), 128^3 osf 1.5 width 3 306 -> 248
// (216), 64^3 osf 1.5 width 3 84 -> 82 (54); the geometric mean goes from 0.78
// to 0.65 of the sector sub-grids' time, the volumes above it from 14 to 6.
//
// A tile's samples are taken in rounds of ER: weights (dense over the tile's
// points per axis) and density-weighted values are staged in LDS once for the
// whole workgroup; every wave then lists the round's samples that reach its
// sub-tile (ballots) and multiplies only those, while the next round's samples
// (addressed by list words loaded a round before) are on their way. The lists
// are in the caller's order: a round holds whole runs of the trajectory
// through the tile, which spread over its sub-tiles (in sector order a round
// fills one or two of them while the other waves wait: 0.80 ms against 0.77 ms
// at the 128^3 koosh workload, 0.30 against 0.27 ms at a 168 x 160 x 44 stack
// of spirals).
//
// Bound: 32 matrix-core cycles per four samples and 16 x 16 block. At 128^3
// osf 1.5, kernel width 3 and 8 coils a sample is in 3.4 sub-tiles of four
// blocks each, 108 cycles, 0.18 ms for 4.2 M samples on 1024 SIMDs; the grid
// itself (0.45 GB) takes 0.09 ms to write, and a tile reads 2.1 times its
// samples (taps and values, 116 bytes each). What is left is mostly waves of a
// workgroup waiting for the one with the most samples of a round (half of the
// wave cycles; matrix cores busy 30 %).
// Spread and fold, measured against sector sub-grids in LDS with a fold over
// neighbouring sectors: 0.91 -> 0.68 ms (128^3 koosh, 8 coils), 2.52 -> 0.81 ms
// (160^3 osf 2, 2.0 M samples, 8 coils), 0.59 -> 0.25 ms (168 x 160 x 44 stack,
// 6 coils), 126 -> 46 us (256^2 osf 2, 16 coils), 123 -> 32 us (224^2 kernel
// width 5, 12 coils), 13 -> 10 us (64^2, 1 coil).

#include <algorithm>

#include "gnufft_internal.hpp"

namespace gnufft {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(8)));  // two complex values

// Shape of a workgroup for NC coils (one wave per sub-tile).
template <int DIM, int NC>
struct TileShape {
  static constexpr int TX = tile_width(DIM, 0), TY = tile_width(DIM, 1), TZ = tile_width(DIM, 2);
  static constexpr int SUM = TX + TY + (DIM == 3 ? TZ : 0);
  static constexpr int SX = NC == 1 ? 8 : 4;        // x points of a sub-tile
  static constexpr int XB = 8 / NC;                 // x points in the 16 columns
  static constexpr int NM = SX / XB;                // 16 x 16 blocks of a sub-tile
  static constexpr int NSX = TX / SX;
  static constexpr int NW = tile_subs(DIM) * 4 / SX;
  static constexpr int NT = 64 * NW;
  static constexpr int H = DIM == 3 ? 4 : 2;        // staging threads per sample
  static constexpr int ER = NT / H;                 // samples per round
  // values: PP threads of two coils (16 bytes) per sample, VI samples each; one
  // coil: the last threads (in 3-D they have no axis)
  static constexpr int PP = NC == 1 ? 1 : NC / 2;
  static constexpr int V0 = NC == 1 ? NT - ER : 0;
  static constexpr int VI = ER * PP > NT ? ER * PP / NT : 1;
  // floats per staged sample: weights per axis, values; a multiple of four
  // with an odd quotient, so rows of different samples start in 16 distinct
  // bank groups
  static constexpr int RAW = (SUM + 2 * NC + 3) & ~3;
  static constexpr int ST = (RAW / 4) % 2 ? RAW : RAW + 4;
  // the finished tile [coil][z][y][x] complex, rows padded so that the
  // accumulators' columns and row groups fall into distinct banks
  static constexpr int YS = DIM == 3 ? 2 * TX : 2 * TX + 4;
  static constexpr int ZS = TY * YS + (DIM == 3 ? 16 : 0);
  static constexpr int CS = TZ * ZS + 4;
  // bytes: (ER + 1) staged samples (the last stays zero), a word of hit bits
  // per sample and a byte list per wave, or in the same place the finished
  // tile
  static constexpr size_t hit_off = (size_t)(ER + 1) * ST * 4;
  static constexpr size_t list_off = hit_off + (size_t)ER * 4;
  static constexpr size_t staged = list_off + (size_t)NW * ER + 16;
  static constexpr size_t out = (size_t)NC * CS * 4;
  static constexpr size_t lds = staged > out ? staged : out;
  static_assert(ER % 64 == 0 && ER < 255, "the threads of a wave share a staging role, a list holds bytes");
};

// Workgroup bid -> work item: runs of kRun consecutive items per XCD
// (workgroups are dispatched round-robin over the 8 XCDs), so neighbouring
// tiles, which share samples, meet in one L2 while heavy regions still
// spread over all XCDs (128^3 koosh: 702 us in runs of 16, 678 in runs of 4;
// a 168 x 160 x 44 stack: 289 in runs of 64, 262 and 257).
constexpr uint32_t kRun = 4;
__device__ inline uint32_t run_item(uint32_t bid) {
  const uint32_t x = bid & 7u, j = bid >> 3;
  return (j / kRun) * (8u * kRun) + x * kRun + (j % kRun);
}
static inline uint32_t run_blocks(uint32_t n) {
  return (n + 8u * kRun - 1) / (8u * kRun) * (8u * kRun);
}

// A sample's taps along one axis: first grid index and up to NX - 1 weights.
template <int NX>
struct Taps {
  int q;
  float w[NX - 1];
};

template <int NX>
__device__ inline Taps<NX> load_taps(const float4* at) {
  Taps<NX> t;
  const float4 a = at[0];
  t.q = __float_as_int(a.x);
  t.w[0] = a.y, t.w[1] = a.z, t.w[2] = a.w;
  if constexpr (NX == 8) {
    const float4 b = at[1];
    t.w[3] = b.x, t.w[4] = b.y, t.w[5] = b.z, t.w[6] = b.w;
  }
  return t;
}

// Weights of the T points of a tile's axis from t0 on, written to dst (zero
// where the sample has no tap); returns a bit per four points reached.
template <int NX>
__device__ inline uint32_t tile_weights(const Taps<NX>& t, int t0, int T, int G, float* dst) {
  float4* d4 = reinterpret_cast<float4*>(dst);
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (4 * i < T) d4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  // the image of the sample nearest to the tile
  int s = t.q - t0;
  s = s >= T ? s - G : s <= -(NX - 1) ? s + G : s;
  uint32_t bits = 0;
#pragma unroll
  for (int u = 0; u < NX - 1; u++)
    if (s + u >= 0 && s + u < T && t.w[u] != 0.0f) {
      dst[s + u] = t.w[u];
      bits |= 1u << ((s + u) >> 2);
    }
  // on grids shorter than a tile and the taps together its other images can
  // reach the tile too (their taps fall on other points, G away)
  if (G < T + NX)
    for (int f = -1; f <= 1; f += 2)
#pragma unroll
      for (int u = 0; u < NX - 1; u++) {
        const int i = s + f * G + u;
        if (i >= 0 && i < T && t.w[u] != 0.0f) {
          dst[i] = t.w[u];
          bits |= 1u << (i >> 2);
        }
      }
  return bits;
}

// One workgroup: chunk `ci` of the tile lists, coils [group * NC, ...).
// NX - 1: weights per axis of the tap table.
// SORTED: the data are in sector order.
template <int DIM, int NC, int NX, bool SORTED = false>
__device__ __forceinline__ void tile_spread_body(const Geom& g, const SpreadArgs& a, uint32_t ci, int group) {
  using S = TileShape<DIM, NC>;
  constexpr int ER = S::ER, ST = S::ST;
  extern __shared__ float4 smem4[];
  char* smem = reinterpret_cast<char*>(smem4);
  float* ent = reinterpret_cast<float*>(smem);
  uint8_t* hit = reinterpret_cast<uint8_t*>(smem + S::hit_off);  // 4 bytes per sample
  uint8_t* list = reinterpret_cast<uint8_t*>(smem + S::list_off);

  const TileChunk ch = a.tiles.chunks[ci];
  const uint32_t n = ch.n;
  const uint32_t* entries = a.tiles.entries + ch.begin;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int t0[3];
  tile_start<DIM>(a.tiles, ch.tile, t0);
  const int coil0 = group * NC;

  // Staging. Weights: thread (e, h) takes axis h of sample e (3-D: h = 3 has
  // none). Values: thread (ve, part) takes two coils of samples ve, ve + NT /
  // PP, ..
  const int e = tid % ER;
  const int h = __builtin_amdgcn_readfirstlane(tid / ER);
  const bool has_axis = h < DIM;
  const int axis = has_axis ? h : 0;
  const int ve = (tid - S::V0) / S::PP, part = tid % S::PP;
  const bool has_value = tid >= S::V0 && ve < ER;
  const bool dens = a.dens != nullptr;
  const float4* taps = a.taps + (size_t)axis * g.M * (NX / 4);
  const float2* data = a.data + (size_t)(coil0 + 2 * part) * a.coil_stride;
  const int coils = a.n_coils - coil0 - 2 * part;  // of this thread
  Taps<NX> ta;
  float sq[S::VI];
  float4 v[S::VI];
  uint32_t je = 0, jv[S::VI];  // list words of the round after the loaded one
  const uint32_t rounds = (n + ER - 1) / ER;
  auto at = [&](uint32_t r, int k) { return r * ER + (uint32_t)k; };  // list position of sample k of round r
  auto load_words = [&](uint32_t r) {
    if (has_axis && at(r, e) < n) je = entries[at(r, e)];
#pragma unroll
    for (int q = 0; q < S::VI; q++) {
      const int k = ve + q * (S::NT / S::PP);
      if (has_value && at(r, k) < n) jv[q] = entries[at(r, k)];
    }
  };
  auto load_round = [&](uint32_t r) {
    if (has_axis && at(r, e) < n) ta = load_taps<NX>(taps + (size_t)je * (NX / 4));
#pragma unroll
    for (int q = 0; q < S::VI; q++) {
      v[q] = make_float4(0.f, 0.f, 0.f, 0.f);
      sq[q] = 1.0f;
      if (!has_value || at(r, ve + q * (S::NT / S::PP)) >= n) continue;
      if (dens) sq[q] = a.dens[jv[q]];
      const uint32_t from = SORTED ? a.pos[jv[q]] : jv[q];
      if (coils > 0) {
        const float2 t = data[from];
        v[q].x = t.x, v[q].y = t.y;
      }
      if (coils > 1) {
        const float2 t = data[(size_t)a.coil_stride + from];
        v[q].z = t.x, v[q].w = t.y;
      }
    }
  };
  load_words(0);
  load_round(0);
  load_words(1);
  if (tid < ST) ent[ER * ST + tid] = 0.0f;  // the padding sample

  // sub-tile of this wave
  const int sx = wave % S::NSX;
  const int sy = DIM == 3 ? wave / S::NSX : 0;
  const int k = lane >> 4, r = lane & 15;
  const int xi = r / (2 * NC), vi = r % (2 * NC);
  f32x4 acc[S::NM];
#pragma unroll
  for (int m = 0; m < S::NM; m++) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint8_t* mylist = list + wave * ER;
  // per-lane float offsets inside a staged sample
  const int off_a = DIM == 3 ? S::TX + 4 * sy + (r & 3) : S::TX + r;
  const int off_z = S::TX + S::TY + (r >> 2);
  const int off_x = S::SX * sx + xi;
  const int off_v = S::SUM + vi;

  for (uint32_t round = 0; round < rounds; round++) {
    // stage this round's samples (no hits where the list has ended)
    if (has_axis && at(round, e) >= n) {
      hit[4 * e + axis] = 0;
    } else if (has_axis) {
      const int T = axis == 0 ? S::TX : axis == 1 ? S::TY : S::TZ;
      const int before = axis == 0 ? 0 : axis == 1 ? S::TX : S::TX + S::TY;
      hit[4 * e + axis] = (uint8_t)tile_weights<NX>(ta, t0[axis], T, g.G[axis], ent + e * ST + before);
    }
#pragma unroll
    for (int q = 0; q < S::VI; q++) {
      const int s = ve + q * (S::NT / S::PP);
      if (!has_value || at(round, s) >= n) continue;
      float2* to = reinterpret_cast<float2*>(ent + s * ST + S::SUM + 4 * part);
      to[0] = make_float2(v[q].x * sq[q], v[q].y * sq[q]);
      to[1] = make_float2(v[q].z * sq[q], v[q].w * sq[q]);
    }
    __syncthreads();
    load_round(round + 1);
    load_words(round + 2);

    // this wave's samples of the round: rank q sits at [q % 4][q / 4], the
    // order in which lane group q % 4 consumes them, padded to whole pairs
    // of groups
    int cnt = 0;
#pragma unroll
    for (int q = 0; q < ER / 64; q++) {
      const int s = q * 64 + lane;
      const uint32_t hb = *reinterpret_cast<const uint32_t*>(hit + 4 * s);
      bool in = (hb >> (sx * (S::SX / 4))) & ((1u << (S::SX / 4)) - 1u);
      if (DIM == 3) in = in && ((hb >> (8 + sy)) & 1u);
      const uint64_t b = __ballot(in);
      if (in) {
        const int rank = cnt + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32),
                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
        mylist[(rank & 3) * (ER / 4) + (rank >> 2)] = (uint8_t)s;
      }
      cnt += __popcll(b);
    }
    const int pairs = (cnt + 7) >> 3;
    if (lane < 8 * pairs - cnt) {
      const int rank = cnt + lane;
      mylist[(rank & 3) * (ER / 4) + (rank >> 2)] = (uint8_t)ER;
    }

    // (one past a list's last pair is read, and not used)
    const uint16_t* ids = reinterpret_cast<const uint16_t*>(mylist + k * (ER / 4));
    uint32_t two = ids[0];
    for (int i = 0; i < pairs; i++) {
      // the operands of two groups of four samples in flight together
      const float* row[2] = {ent + (two & 255u) * ST, ent + (two >> 8) * ST};
      two = ids[i + 1];
      float wa[2], val[2], wx[2][S::NM];
#pragma unroll
      for (int q = 0; q < 2; q++) {
        wa[q] = row[q][off_a];
        if (DIM == 3) wa[q] *= row[q][off_z];
        val[q] = row[q][off_v];
        if constexpr (NC == 8) {  // (SX == 4)
          const float4 w4 = *reinterpret_cast<const float4*>(row[q] + S::SX * sx);
          wx[q][0] = w4.x, wx[q][1] = w4.y, wx[q][2] = w4.z, wx[q][3] = w4.w;
        } else {
#pragma unroll
          for (int m = 0; m < S::NM; m++) wx[q][m] = row[q][off_x + S::XB * m];
        }
      }
#pragma unroll
      for (int q = 0; q < 2; q++)
#pragma unroll
        for (int m = 0; m < S::NM; m++)
          acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(wa[q], wx[q][m] * val[q], acc[m], 0, 0, 0);
    }
    __syncthreads();  // the round is consumed
  }

  // The finished tile goes through LDS: lane (k, column) holds rows 4k .. 4k+3
  // of its column (y = 4 sy + j at z = k in 3-D, y = 4 k + j in 2-D); the grid
  // takes whole rows of 128 bytes (8-byte stores of single points would each
  // be a transaction of their own at the L2).
  float* out = reinterpret_cast<float*>(smem);
  if (n) {
    float* o = out + (vi >> 1) * S::CS + (DIM == 3 ? k * S::ZS + 4 * sy * S::YS : 4 * k * S::YS) +
               2 * (S::SX * sx + xi) + (vi & 1);
#pragma unroll
    for (int m = 0; m < S::NM; m++)
#pragma unroll
      for (int j = 0; j < 4; j++) o[2 * S::XB * m + j * S::YS] = acc[m][j];
    __syncthreads();
  }
  constexpr int HALF = tile_points(DIM) / 2;  // pairs of points in x
  for (int q = tid; q < NC * HALF; q += S::NT) {
    const int cc = q / HALF, pt = 2 * (q % HALF);
    const int c = coil0 + cc;
    if (c >= a.n_coils) break;
    const int x = pt % S::TX, y = (pt / S::TX) % S::TY, z = pt / (S::TX * S::TY);
    f32x4u two = {0.f, 0.f, 0.f, 0.f};
    if (n) two = *reinterpret_cast<const f32x4u*>(out + cc * S::CS + z * S::ZS + y * S::YS + 2 * x);
    if (ch.slot != kNoSlot) {
      *reinterpret_cast<f32x4u*>(a.scratch + ((size_t)ch.slot * a.n_coils + c) * tile_points(DIM) + pt) = two;
      continue;
    }
    const int gx = t0[0] + x, gy = t0[1] + y, gz = t0[2] + z;
    if (gx >= g.G[0] || gy >= g.G[1] || (DIM == 3 && gz >= g.G[2])) continue;
    float2* dst = a.grid + (size_t)c * g.Ng;
    // the two points are neighbours unless the row ends or the shift's wrap
    // falls between them
    if (gx + 1 < g.G[0] && !(a.fold_shift && gx + 1 == g.shift_inv[0])) {
      *reinterpret_cast<f32x4u*>(dst + tile_store_index<DIM>(g, gx, gy, gz, a.fold_shift)) = two;
    } else {
      dst[tile_store_index<DIM>(g, gx, gy, gz, a.fold_shift)] = make_float2(two[0], two[1]);
      if (gx + 1 < g.G[0])
        dst[tile_store_index<DIM>(g, gx + 1, gy, gz, a.fold_shift)] = make_float2(two[2], two[3]);
    }
  }
}

// Four workgroups of 8 waves fill a CU up to 64 registers (two more cost 15 us
// of 683 at 128^3).
template <int DIM, int NC, int NX, bool SORTED>
__global__ void __launch_bounds__((TileShape<DIM, NC>::NT))
    __attribute__((amdgpu_waves_per_eu(DIM == 3 && NX == 4 ? 8 : 4))) tile_spread_kernel(Geom g, SpreadArgs a) {
  const uint32_t ci = run_item(blockIdx.x);
  if (ci >= a.tiles.n_chunks) return;
  tile_spread_body<DIM, NC, NX, SORTED>(g, a, ci, blockIdx.y);
}

// Sum of a tile's chunks, in chunk order, into the grid. One workgroup per
// (task, coil, 256 points).
template <int DIM>
__device__ inline void tile_reduce_body(const Geom& g, const SpreadArgs& a, uint32_t task, int c, int block) {
  constexpr int TX = tile_width(DIM, 0), TY = tile_width(DIM, 1);
  const TileTask t = a.tiles.tasks[task];
  const int pt = block * 256 + (int)threadIdx.x;
  const size_t stride = (size_t)a.n_coils * tile_points(DIM);
  const float2* base = a.scratch + (size_t)t.slot * stride + (size_t)c * tile_points(DIM) + pt;
  float2 acc = base[0];
#pragma unroll 8
  for (uint32_t k = 1; k < t.count; k++) {
    const float2 v = base[k * stride];
    acc.x += v.x;
    acc.y += v.y;
  }
  int t0[3];
  tile_start<DIM>(a.tiles, t.tile, t0);
  const int gx = t0[0] + pt % TX, gy = t0[1] + (pt / TX) % TY, gz = t0[2] + pt / (TX * TY);
  if (gx < g.G[0] && gy < g.G[1] && (DIM == 2 || gz < g.G[2]))
    a.grid[(size_t)c * g.Ng + tile_store_index<DIM>(g, gx, gy, gz, a.fold_shift)] = acc;
}

template <int DIM>
__global__ void __launch_bounds__(256) tile_reduce_kernel(Geom g, SpreadArgs a) {
  tile_reduce_body<DIM>(g, a, blockIdx.x, blockIdx.y, blockIdx.z);
}

template <typename K>
hipError_t allow_lds(K kernel, size_t lds) {
  if (lds <= 64 * 1024) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

template <int DIM, int NC, int NX>
hipError_t tile_launch(const Geom& g, const SpreadArgs& a, hipStream_t s) {
  const size_t lds = TileShape<DIM, NC>::lds;
  auto kernel = a.pos ? tile_spread_kernel<DIM, NC, NX, true> : tile_spread_kernel<DIM, NC, NX, false>;
  hipError_t e = allow_lds(kernel, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(run_blocks(a.tiles.n_chunks), (a.n_coils + NC - 1) / NC),
                     dim3(TileShape<DIM, NC>::NT), lds, s, g, a);
  return hipGetLastError();
}

template <int DIM, int NX>
hipError_t tile_launch_nc(const Geom& g, const SpreadArgs& a, hipStream_t s) {
  switch (tile_coils(a.n_coils)) {
    case 8: return tile_launch<DIM, 8, NX>(g, a, s);
    case 4: return tile_launch<DIM, 4, NX>(g, a, s);
    case 2: return tile_launch<DIM, 2, NX>(g, a, s);
    default: return tile_launch<DIM, 1, NX>(g, a, s);
  }
}

}  // namespace

hipError_t launch_spread(const Geom& g, const SpreadArgs& a, hipStream_t s) {
  if (a.n_coils == 0) return hipSuccess;
  hipError_t e;
  const bool wide = tap_vec(g.kw) == 2;
  if (g.dim == 3)
    e = wide ? tile_launch_nc<3, 8>(g, a, s) : tile_launch_nc<3, 4>(g, a, s);
  else
    e = wide ? tile_launch_nc<2, 8>(g, a, s) : tile_launch_nc<2, 4>(g, a, s);
  if (e != hipSuccess || a.tiles.n_tasks == 0) return e;
  const dim3 rg(a.tiles.n_tasks, a.n_coils, tile_points(g.dim) / 256);
  if (g.dim == 3)
    hipLaunchKernelGGL(tile_reduce_kernel<3>, rg, dim3(256), 0, s, g, a);
  else
    hipLaunchKernelGGL(tile_reduce_kernel<2>, rg, dim3(256), 0, s, g, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Batches of operators: one launch per coil-group size NC over (operator,
// chunk, coil group) items.
// ---------------------------------------------------------------------------
namespace {

template <int DIM, int NC, int NX>
__global__ void __launch_bounds__((TileShape<DIM, NC>::NT))
    tile_spread_batch_kernel(const BatchOp* __restrict__ ops, BatchList l) {
  uint4 it;
  if (!batch_item(l, blockIdx.x, &it)) return;
  const BatchOp& op = ops[it.x];
  tile_spread_body<DIM, NC, NX>(op.g, op.s, it.y, (int)it.z);
}

// task (operator, task, coil, block of 256 points) per workgroup
template <int DIM>
__global__ void __launch_bounds__(256) tile_reduce_batch_kernel(const BatchOp* __restrict__ ops,
                                                                const uint4* __restrict__ items) {
  const uint4 it = items[blockIdx.x];
  const BatchOp& op = ops[it.x];
  tile_reduce_body<DIM>(op.g, op.s, it.y, (int)it.z, (int)it.w);
}

template <int DIM, int NC, int NX>
hipError_t tile_batch(const BatchOp* ops, const BatchList& l, size_t lds, hipStream_t s) {
  hipError_t e = allow_lds(tile_spread_batch_kernel<DIM, NC, NX>, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((tile_spread_batch_kernel<DIM, NC, NX>), dim3(8u * (l.max_range ? l.max_range : 1u)),
                     dim3(TileShape<DIM, NC>::NT), lds, s, ops, l);
  return hipGetLastError();
}

template <int DIM, int NX>
hipError_t tile_batch_nc(int nc, const BatchOp* ops, const BatchList& l, size_t lds, hipStream_t s) {
  switch (nc) {
    case 8: return tile_batch<DIM, 8, NX>(ops, l, lds, s);
    case 4: return tile_batch<DIM, 4, NX>(ops, l, lds, s);
    case 2: return tile_batch<DIM, 2, NX>(ops, l, lds, s);
    default: return tile_batch<DIM, 1, NX>(ops, l, lds, s);
  }
}

}  // namespace

hipError_t launch_spread_batch(int dim, int nx, int nc, const BatchOp* ops, const BatchList& l,
                               size_t lds, hipStream_t s) {
  if (l.n == 0) return hipSuccess;
  if (dim == 3)
    return nx == 8 ? tile_batch_nc<3, 8>(nc, ops, l, lds, s) : tile_batch_nc<3, 4>(nc, ops, l, lds, s);
  return nx == 8 ? tile_batch_nc<2, 8>(nc, ops, l, lds, s) : tile_batch_nc<2, 4>(nc, ops, l, lds, s);
}

hipError_t launch_tile_reduce_batch(int dim, const BatchOp* ops, const BatchList& tasks, hipStream_t s) {
  if (tasks.n == 0) return hipSuccess;
  if (dim == 3)
    hipLaunchKernelGGL(tile_reduce_batch_kernel<3>, dim3(tasks.n), dim3(256), 0, s, ops, tasks.items);
  else
    hipLaunchKernelGGL(tile_reduce_batch_kernel<2>, dim3(tasks.n), dim3(256), 0, s, ops, tasks.items);
  return hipGetLastError();
}

size_t spread_lds_bytes(int dim, int nc) {
  switch (nc) {
    case 8: return dim == 3 ? TileShape<3, 8>::lds : TileShape<2, 8>::lds;
    case 4: return dim == 3 ? TileShape<3, 4>::lds : TileShape<2, 4>::lds;
    case 2: return dim == 3 ? TileShape<3, 2>::lds : TileShape<2, 2>::lds;
    default: return dim == 3 ? TileShape<3, 1>::lds : TileShape<2, 1>::lds;
  }
}

bool sector_cover_ok(const Geom& g) {
  // padded sectors (with periodic images) meeting one sector, all axes; with
  // P <= 2 sw and no image of a sector meeting itself at most five per axis
  bool few = true;
  for (int a = 0; a < g.dim; a++) few = few && g.P <= 2 * g.sw && g.P <= g.G[a];
  if (few) return true;
  long long cands = 1;
  for (int a = 0; a < g.dim; a++) {
    const int G = g.G[a], S = g.S[a];
    int most = 0;
    for (int s = 0; s < S; s++) {
      const int lo = s * g.sw, hi = std::min(lo + g.sw, G);
      int m = 0;
      for (int n = 0; n < S; n++) {
        const int first = n * g.sw + g.sw / 2 - g.off;
        bool meets = false;
        for (int i = 0; i < g.P && !meets; i++) {
          const int q = ((first + i) % G + G) % G;
          meets = q >= lo && q < hi;
        }
        m += meets ? 1 : 0;
      }
      most = std::max(most, m);
    }
    cands *= (long long)most * ((g.P + G - 1) / G);
  }
  return cands <= 256;
}

}  // namespace gnufft
